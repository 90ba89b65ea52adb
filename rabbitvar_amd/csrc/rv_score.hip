// Scoring kernels (gfx950).  Positions whose alleles all live in the dense table (the vast majority):
//   k_score_prepick  simple mode: every dense position's status, and the list of those that can print,
//                    from the rows alone, while the realigner works on the host
//   k_score_list, k_score_dense  those listed positions, one wavefront each or, many, one per lane
//   k_score_pick, k_score_dense  -p and somatic mode: the positions that need scoring, one per lane
// Positions with descriptors, insertions or realignment changes (CSR records):
//   k_score_cx       one wavefront each
//   k_fisher         the p-value of every record they emitted (--fisher), one wavefront each
// The scoring itself is score_position_in(); the template parameters size its work area.
#include <hip/hip_runtime.h>

#include "rv_fisher_wave.h"
#include "rv_kernels.h"
#include "rv_score_body.h"

#include <mutex>

namespace rv {

// Picks the dense positions that need scoring (score_needed) into S.pick_list.  Most positions
// end at those checks, and a wavefront of the scoring kernel takes as long as its slowest lane, so
// the scoring kernel then runs full wavefronts of positions that all do the work.  One ballot and
// one counter update per wavefront; the list's order does not matter (every record carries its
// position and rank).
__global__ void __launch_bounds__(256) k_score_pick(ScoreIn S) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    bool need = false;
    const int p = S.dense_lo + i;
    // (the emitting somatic pass reads the rows of the wanted positions only)
    if (i < S.dense_n && !(S.want && !S.want[i])) need = dense_needed(S, p);
    const unsigned long long m = __ballot(need);
    const int lane = (int)(threadIdx.x & 63u);
    unsigned base = 0;
    if (lane == 0 && m) base = atomicAdd(S.pick_count, (unsigned)__popcll(m));
    base = __shfl(base, 0);
    if (need) S.pick_list[base + (unsigned)__popcll(m & ((1ull << lane) - 1ull))] = p;
}

// Most dense positions cannot print: their variants are a read or two.  This pass over the rows needs
// nothing the realigner makes (a position that ends up on the record list is scored from there, and
// its status and listing here are passed over), so it costs the call nothing (0.37 ms beside host work on
// a 5 Mb contig at 60x, bound by the rows' 1.4 GB); the steps after the realigner then read the few
// listed positions instead of scoring every position with a mismatch: 0.16 ms (28,000 of them, a lane
// each) where 1.48 + 0.15 went.
__global__ void __launch_bounds__(256) k_score_prepick(ScoreIn S) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    bool need = false;
    const int p = S.dense_lo + i;
    if (i < S.dense_n) {
        uint8_t st = 0;
        if (dense_row_needed(S, p)) need = dense_can_print(S, p, st);
        S.status[i] = st;
    }
    const unsigned long long m = __ballot(need);
    const int lane = (int)(threadIdx.x & 63u);
    unsigned base = 0;
    if (lane == 0 && m) base = atomicAdd(S.pick_count, (unsigned)__popcll(m));
    base = __shfl(base, 0);
    if (need) S.pick_list[base + (unsigned)__popcll(m & ((1ull << lane) - 1ull))] = p;
}

// How many listed positions are scored one per lane.  A wavefront per position costs the chip 25 ns a
// position once all its wavefronts (16 a CU) are busy; one per lane 3 ns, but with 64 differing positions
// in a wavefront the first takes 0.1 ms.  Scoring of calls at 60x that print m dense positions, ms, a wavefront each /
// a lane each: 1,000 0.11 / 0.15, 2,000 0.14 / 0.15, 4,100 0.22 / 0.19, 16,000 0.53 / 0.21, 66,000 1.74 / 0.30.
constexpr int SCORE_LANES_MIN = 3072;

// min_count: a shorter list is k_score_list's
__global__ void __launch_bounds__(128) k_score_dense(ScoreIn S, int min_count) {
    const int m = (int)*S.pick_count;
    if (m < min_count) return;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < m; i += (int)(gridDim.x * blockDim.x)) {
        const int p = S.pick_list[i];
        // single bases only: the longest string is a genotype ("A/C")
        score_position<16, 4>(S, p, true, p - S.dense_lo);
    }
}

namespace {
// bases of the reference window around a position, copied to LDS by its wavefront (the steps look
// bases up one by one, a global read each otherwise)
constexpr int NEAR_BEFORE = 128, NEAR = 384;
__device__ __forceinline__ RefWindow stage_near(const ScoreIn& S, int p, char* near) {
    for (int j = (int)(threadIdx.x & 63u); j < NEAR; j += 64) {
        const int k = p - NEAR_BEFORE + j;
        near[j] = k >= S.ref_lo && k <= S.ref_hi ? S.ref[k - S.ref_lo] : '\0';
    }
    return RefWindow{S.ref, S.ref_lo, S.ref_hi, near, p - NEAR_BEFORE, NEAR};
}
}  // namespace

// One wavefront per position, its work area and the reference around it in LDS, the steps on its
// first lane (bound by that lane's dependent steps).  The positions differ in every branch (descriptor
// forms, allele counts, string lengths), so 64 of them in one wavefront ran one after another, each
// through its own scratch memory; and the record list's work area of 14 KB per lane in scratch (1 MB
// per wavefront) is more than the runtime can give every hardware queue when several engines score at
// once.
__global__ void __launch_bounds__(64) k_score_list(ScoreIn S) {
    __shared__ ScoreWork<16, 4> work;
    __shared__ char near[NEAR];
    const int m = (int)*S.pre_count;
    if (m >= SCORE_LANES_MIN) return;
    for (int i = (int)blockIdx.x; i < m; i += (int)gridDim.x) {
        const int p = S.pre_list[i];
        const RefWindow rf = stage_near(S, p, near);
        __syncthreads();
        if (threadIdx.x == 0) score_position_in<16, 4>(S, p, true, p - S.dense_lo, work, rf);
        __syncthreads();
    }
}

// The record list's positions.  Their entries and descriptor text are copied to LDS too, all lanes at
// once (the steps follow them one dependent load after another otherwise), where they fit: 64 entries
// and 1 KB of text, so that seven positions share a CU.  Dense indels, 872 positions: 0.60 ms of scoring
// (0.90 before the copies and k_fisher).
__global__ void __launch_bounds__(64) k_score_cx(ScoreIn S) {
    constexpr int ENTRIES = 64, TEXT = 1024, WORDS = (int)(sizeof(CxEntry) / 4);
    static_assert(sizeof(CxEntry) % 8 == 0, "copied in words");
    __shared__ ScoreWork<1536, MAXV> work;
    __shared__ char near[NEAR];
    __shared__ CxEntry ent[ENTRIES];
    __shared__ char text[TEXT];
    const int i = (int)blockIdx.x, lane = (int)threadIdx.x;
    if (S.want && !S.want[S.dense_n + i]) return;
    const int off = S.cx_off[i], n = S.cx_off[i + 1] - off;
    CxView view{i, n, S.cx + off, S.cx_arena, 0};
    const RefWindow rf = stage_near(S, S.cx_pos[i], near);
    if (n <= ENTRIES) {
        const uint32_t* src = reinterpret_cast<const uint32_t*>(S.cx + off);
        uint32_t* dst = reinterpret_cast<uint32_t*>(ent);
        for (int w = lane; w < n * WORDS; w += 64) dst[w] = src[w];
        view.entries = ent;
        __syncthreads();
        uint32_t lo = ~0u, hi = 0u;
        if (lane < n) {
            lo = ent[lane].desc_off;
            hi = lo + (uint32_t)ent[lane].desc_len;
        }
        for (int o = 32; o > 0; o >>= 1) {
            const uint32_t a = (uint32_t)__shfl_xor((int)lo, o), b = (uint32_t)__shfl_xor((int)hi, o);
            lo = a < lo ? a : lo;
            hi = b > hi ? b : hi;
        }
        if (lo < hi && hi - lo <= TEXT) {
            for (uint32_t j = lane; j < hi - lo; j += 64) text[j] = S.cx_arena[lo + j];
            view.arena = text;
            view.arena_lo = lo;
        }
    }
    __syncthreads();
    if (lane == 0) score_position_in<1536, MAXV>(S, S.cx_pos[i], false, S.dense_n + i, work, rf, &view);
}

// The Fisher column of the records the kernels above appended: bound by the divisions of a stretch and
// the serial sum.  Scoring with it 0.25 ms where a lane alone took 0.52 (2.2 kb amplicon at 2500x).
// At 60x a tail has some thirty terms and most lanes idle: 0.31 ms for the 28,600 records of a 5 Mb contig;
// the million records of a -p call on 1 Mb take 0.9 ms where a lane each, in the scoring kernel, took
// 0.2 (of 2.3 ms of scoring either way).  The grid of 2,048 wavefronts is 8 a CU of the 20 that fit.
__global__ void __launch_bounds__(64) k_fisher(ScoreIn S) {
    __shared__ double terms[FISHER_TERMS];
    const unsigned n = readable_records(S);
    for (unsigned i = blockIdx.x; i < n; i += gridDim.x) {
        OutRec& o = S.out[i];
        const double p = fisher_two_sided_wave(o.rfc, o.rrc, o.fwd, o.rev, LGTable{S.lgamma_tab, S.lgamma_n}, terms,
                                               (int)threadIdx.x);
        if (threadIdx.x == 0) o.fisher_p = p;
    }
}

__global__ void __launch_bounds__(256) k_fisher_table(const int* tab, int n, double* out, const double* lgt, int lgt_n) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        double l, r;
        double two = fisher_two_sided(tab[4 * i], tab[4 * i + 1], tab[4 * i + 2], tab[4 * i + 3], &l, &r,
                                      LGTable{lgt, lgt_n});
        out[3 * i] = two;
        out[3 * i + 1] = l;
        out[3 * i + 2] = r;
    }
}

__global__ void __launch_bounds__(64) k_zero_u32(unsigned* p, int n) {
    const int i = (int)threadIdx.x;
    if (i < n) p[i] = 0u;
}

hipError_t launch_score(const ScoreIn& S, hipStream_t s) {
    if (S.dense_n > 0 && S.pre_list) {
        if (!S.pre_count) return hipErrorInvalidValue;
        // how many are listed is known on the device: the kernel whose turn it is not returns at once
        hipLaunchKernelGGL(k_score_list, dim3((unsigned)(S.dense_n < SCORE_LANES_MIN ? S.dense_n : SCORE_LANES_MIN)),
                           dim3(64), 0, s, S);
        if (S.dense_n >= SCORE_LANES_MIN) {
            ScoreIn L = S;
            L.pick_list = const_cast<int32_t*>(S.pre_list);
            L.pick_count = const_cast<unsigned*>(S.pre_count);
            const int blocks = (S.dense_n + 127) / 128;
            hipLaunchKernelGGL(k_score_dense, dim3((unsigned)(blocks < 2048 ? blocks : 2048)), dim3(128), 0, s, L,
                               SCORE_LANES_MIN);
        }
    } else if (S.dense_n > 0) {
        if (!S.pick_list || !S.pick_count) return hipErrorInvalidValue;
        // the count starts at zero with a fill kernel (no memset node if a caller captures this)
        hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(64), 0, s, S.pick_count, 1);
        hipLaunchKernelGGL(k_score_pick, dim3((S.dense_n + 255) / 256), dim3(256), 0, s, S);
        const int blocks = (S.dense_n + 127) / 128;
        hipLaunchKernelGGL(k_score_dense, dim3((unsigned)(blocks < 8192 ? blocks : 8192)), dim3(128), 0, s, S, 0);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (S.n_cx > 0) hipLaunchKernelGGL(k_score_cx, dim3((unsigned)S.n_cx), dim3(64), 0, s, S);
    // only the simple printer has the column; how many records there are is known on the device
    if (S.cfg.fisher && S.somatic == SCORE_SIMPLE && S.max_out > 0)
        hipLaunchKernelGGL(k_fisher, dim3(S.max_out < 2048u ? S.max_out : 2048u), dim3(64), 0, s, S);
    return hipGetLastError();
}

hipError_t launch_score_prepick(const ScoreIn& S, hipStream_t s) {
    if (S.dense_n <= 0) return hipSuccess;
    if (!S.pick_list || !S.pick_count || !S.status) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(64), 0, s, S.pick_count, 1);
    hipLaunchKernelGGL(k_score_prepick, dim3((S.dense_n + 255) / 256), dim3(256), 0, s, S);
    return hipGetLastError();
}

hipError_t launch_fisher_table(const int* tab, int n, double* out, const double* lgt, int lgt_n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fisher_table, dim3((n + 255) / 256), dim3(256), 0, s, tab, n, out, lgt, lgt_n);
    return hipGetLastError();
}

// ---------------------------------------------------------------- the allocation-free Fisher entry
// rv_fisher_tables_noalloc works in this file-scope device array instead of engine buffers: the
// log-gamma table, then the tables in, then the p-values out, for at most FISHER_NOALLOC_MAX_TABLES tables
// per call.  Each GPU holds its own copy until the process ends; every call on one GPU uses it, so
// calls that overlap on one GPU race.  Nothing in it has to start at zero: a call writes the inputs
// it reads and every output it returns.
constexpr size_t FNA_LGT = 0;
constexpr size_t FNA_IN = FNA_LGT + sizeof(double) * FISHER_LGT_N;
constexpr size_t FNA_OUT = FNA_IN + sizeof(int) * 4 * FISHER_NOALLOC_MAX_TABLES;
constexpr size_t FNA_BYTES = FNA_OUT + sizeof(double) * 3 * FISHER_NOALLOC_MAX_TABLES;
static __device__ __align__(256) unsigned char scratch[FNA_BYTES];

namespace {
constexpr int FNA_MAX_DEVICES = 64;
std::mutex fna_mu;
unsigned char* fna_ptr[FNA_MAX_DEVICES];  // the device address of `scratch`, per device (nullptr: not set up)
double fna_host_lgt[FISHER_LGT_N];        // the host-built table, computed once (static storage)
bool fna_host_ready = false;
}  // namespace

// Set-up on the current device (once): the scratch array's device address, and the log-gamma table
// copied into it.
static hipError_t fisher_noalloc_setup(unsigned char*& base, const char** err) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) {
        *err = "no current HIP device";
        return e;
    }
    if (dev < 0 || dev >= FNA_MAX_DEVICES) {
        *err = "device index beyond the scratch table";
        return hipErrorInvalidDevice;
    }
    std::lock_guard<std::mutex> lk(fna_mu);
    if (!fna_ptr[dev]) {
        if (!fna_host_ready) {
            fisher_lgamma_table(fna_host_lgt, FISHER_LGT_N);
            fna_host_ready = true;
        }
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            *err = "hipGetSymbolAddress(scratch) failed";
            return e != hipSuccess ? e : hipErrorInvalidSymbol;
        }
        e = hipMemcpy((unsigned char*)p + FNA_LGT, fna_host_lgt, sizeof fna_host_lgt, hipMemcpyHostToDevice);
        if (e != hipSuccess) {
            *err = "log-gamma table upload failed";
            return e;
        }
        fna_ptr[dev] = (unsigned char*)p;
    }
    base = fna_ptr[dev];
    return hipSuccess;
}

hipError_t fisher_tables_noalloc(const int* tab, int n, double* out, const char** err) {
    unsigned char* base = nullptr;
    hipError_t e = fisher_noalloc_setup(base, err);
    if (e != hipSuccess) return e;
    int* din = (int*)(base + FNA_IN);
    double* dout = (double*)(base + FNA_OUT);
    const double* lgt = (const double*)(base + FNA_LGT);
    if ((e = hipMemcpy(din, tab, sizeof(int) * 4 * (size_t)n, hipMemcpyHostToDevice)) != hipSuccess) {
        *err = "table upload failed";
        return e;
    }
    if ((e = launch_fisher_table(din, n, dout, lgt, FISHER_LGT_N, nullptr)) != hipSuccess) {
        *err = "Fisher kernel launch failed";
        return e;
    }
    if ((e = hipMemcpy(out, dout, sizeof(double) * 3 * (size_t)n, hipMemcpyDeviceToHost)) != hipSuccess) {
        *err = "result download failed";
        return e;
    }
    return hipSuccess;
}

}  // namespace rv
