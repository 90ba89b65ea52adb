// Pileup kernels for gfx950: one lane per read (or, for the CIGAR rewrite rules, one wavefront) for
// the prep pass, one wavefront per read for the walk, one lane per dense row for initialisation, one
// lane per anchor record for the deferred subtraction.
#include <hip/hip_runtime.h>

#include "rv_kernels.h"
#include "rv_pileup_body.h"

namespace rv {

// Reads of one M run, one per lane (their rewrite looks at a few bases at either end), and without local
// realignment the others too (300 kb at 60x with an indel in nearly every read: 0.06 ms, 0.44 a wavefront
// each); with it those are listed for k_prep_rules.  One update of each counter per wavefront.
__global__ void __launch_bounds__(256) k_prep(const WalkArgs* A, PrepRec* prep, uint32_t* cig, WalkCounters* ctr,
                                              PrepCounts* counts, int32_t* rules) {
    // arguments as values, so that the stores below cannot force reloads (see k_walk)
    const ReadsDev R = A->R;
    const Window W = A->W;
    const Config cfg = A->cfg;
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = (int)(threadIdx.x & 63u);
    int span = 0, tot = 0;
    bool by_rules = false;
    if (r < R.n) {
        PrepRec p;
        by_rules = prep_lane(r, R, W, cfg, A->dup, ctr, cig, p, span, tot);
        prep[r] = p;
    }
    for (int o = 32; o > 0; o >>= 1) {
        const int a = __shfl_xor(span, o), b = __shfl_xor(tot, o);
        span = a > span ? a : span;
        tot = b > tot ? b : tot;
    }
    const unsigned long long m = __ballot(by_rules);
    unsigned base = 0;
    if (lane == 0) {
        // (a stale value only costs an update)
        if (span > *(volatile int*)&counts->max_span) atomicMax(&counts->max_span, span);
        if (tot > *(volatile int*)&ctr->max_read_length) atomicMax(&ctr->max_read_length, tot);
        if (m) base = atomicAdd(&counts->n_rules, (unsigned)__popcll(m));
    }
    base = (unsigned)__shfl((int)base, 0);
    if (by_rules) rules[base + (unsigned)__popcll(m & ((1ull << lane) - 1ull))] = (int32_t)r;
}

// The listed reads, one wavefront each: its lanes copy the read to LDS and run the rules over the
// CIGAR text there, all of them the same steps, so that a rule's start offsets are tried at once
// (a single lane took 115 us a read, most of it in those searches).  (One read per lane among
// the others, the rules' branches serialised whole wavefronts over texts in scratch memory.)
__global__ void __launch_bounds__(64) k_prep_rules(const WalkArgs* A, PrepRec* prep, uint32_t* cig, WalkCounters* ctr,
                                                   const PrepCounts* counts, const int32_t* rules) {
    __shared__ char seq[STAGE_LEN];
    __shared__ uint8_t qual[STAGE_LEN];
    __shared__ uint32_t rec[MAXC];
    __shared__ CigarWork work;
    const ReadsDev R = A->R;
    const Window W = A->W;
    const Config cfg = A->cfg;
    const int lane = (int)threadIdx.x;
    const unsigned n = counts->n_rules;
    for (unsigned k = blockIdx.x; k < n; k += gridDim.x) {
        const int64_t r = rules[k];
        const int64_t so = R.seq_off[r];
        const int lseq = (int)(R.seq_off[r + 1] - so);
        const bool staged = lseq <= STAGE_LEN;
        if (staged)
            for (int i = lane; i < lseq; i += 64) {
                seq[i] = (char)R.bases[so + i];
                qual[i] = R.quals[so + i];
            }
        __syncthreads();
        PrepRec p = prep[r];
        int tot = 0;
        const ReadView rd{staged ? seq : (const char*)(R.bases + so), staged ? qual : R.quals + so, lseq};
        const bool ok = prep_other<true>(r, R, W, cfg, rd, p, rec, &work, tot);
        __syncthreads();
        if (lane == 0) {
            if (!ok) atomicAdd(&ctr->capacity, 1ull);
            if (tot > *(volatile int*)&ctr->max_read_length) atomicMax(&ctr->max_read_length, tot);
            prep[r] = p;
        }
        const int nw = p.ncig + 1 < MAXC ? p.ncig + 1 : MAXC;
        for (int i = lane; i < nw; i += 64) cig[(size_t)r * MAXC + i] = rec[i];
        __syncthreads();
    }
}

// -t: marks the reads the record filter drops as duplicates (before prep, which then skips them)
__global__ void __launch_bounds__(256) k_dedup(const WalkArgs* A) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r < A->R.n) A->dup[r] = is_duplicate(A->R, A->cfg, r) ? 1 : 0;
}

__global__ void __launch_bounds__(256) k_fill_rows(DenseRow* rows, int n) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) fill_row_one(rows, i);
}

namespace {
// The launch arguments through scalar loads: nothing writes them during the launch, which the
// compiler cannot see past the walk's own stores
__device__ __forceinline__ WalkArgs load_args(const WalkArgs* A) {
    static_assert(sizeof(WalkArgs) % 4 == 0, "copied in words");
    typedef const __attribute__((address_space(4))) uint32_t* ConstWords;
    const ConstWords w = (ConstWords)(uintptr_t)A;
    WalkArgs a;
    uint32_t* const o = reinterpret_cast<uint32_t*>(&a);
#pragma unroll
    for (int i = 0; i < (int)(sizeof(WalkArgs) / 4); i++) o[i] = w[i];
    return a;
}
}  // namespace

// One workgroup walks nreads consecutive reads (sorted by position), one wavefront per read at a
// time, into an LDS tile that starts TILE_MARGIN bases before the first read; the tile is added to
// the dense rows once at the end.

__global__ void __launch_bounds__(WALK_THREADS) k_walk(const WalkArgs* A, const PrepRec* prep, const uint32_t* cig,
                                                       int nreads) {
    const int waves = (int)(blockDim.x / warpSize);
    // the wavefront index is uniform across its lanes; saying so lets the per-read state live in
    // scalar registers
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / warpSize));
    const int lane = (int)(threadIdx.x % warpSize);
    // what every read needs, as values: read through a pointer, the compiler would reload it from
    // global memory after every store and atomic of the walk (they could alias)
    const int64_t n = A->R.n;
    const uint8_t* const bases = A->R.bases;
    const uint8_t* const quals = A->R.quals;
    // neighbouring tiles overlap by a read's length, so consecutive ones go to one XCD (workgroups are
    // dealt to the eight in turn): their rows are then added to in one L2
    const unsigned per = gridDim.x / 8, more = gridDim.x % 8, xcd = blockIdx.x % 8;
    const unsigned tile = xcd * per + (xcd < more ? xcd : more) + blockIdx.x / 8;
    const int64_t r0 = (int64_t)tile * nreads;
    const int tile_lo = __builtin_amdgcn_readfirstlane((r0 < n ? prep[r0].position : 0) - TILE_MARGIN);
    const PlainArgs plain = plain_args(A->W, A->cfg, tile_lo);
    // reads after each wavefront's first are handed out as wavefronts finish (reads differ in cost;
    // every contribution merges the same way whichever wavefront walks it)
    __shared__ int walk_next;
    if (threadIdx.x == 0) walk_next = waves;
    tile_init((int)threadIdx.x, (int)blockDim.x, A->W, tile_lo);
    const int here = (int)(n - r0 < nreads ? n - r0 : nreads);
    constexpr int WORDS = (int)(sizeof(PrepRec) / 16);
    for (int i = (int)threadIdx.x; i < here * WORDS; i += (int)blockDim.x)
        reinterpret_cast<uint4*>(walk_prep)[i] = reinterpret_cast<const uint4*>(prep + r0)[i];
    __syncthreads();
    WaveStage* const st = &walk_stage[wave];
    int k = wave;
    WalkFetch f{0, 0, 0};
    if (k < here) f = walk_fetch(walk_prep[k], r0 + k, bases, quals, cig, lane);
    while (k < here) {
        // the previous read's steps are done with the copy before it is overwritten, and the copy is
        // complete before any lane reads it (LDS operations of one wavefront complete in order)
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        walk_put(walk_prep[k], f, st, lane);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        int nk = 0;
        if (lane == 0) nk = atomicAdd(&walk_next, 1);
        nk = __builtin_amdgcn_readfirstlane(nk);
        if (nk < here) f = walk_fetch(walk_prep[nk], r0 + nk, bases, quals, cig, lane);
        if (uniform(walk_prep[k].status) == RD_PARSE) {
            unsigned tseq = 0;
            const int done = walk_plain(walk_prep[k], (int)(r0 + k), plain, lane, wave, tseq);
            if (done == 0 || done < uniform(walk_prep[k].rlen1)) {
                // any other read: the whole walker, with the launch arguments loaded here, so that they
                // hold no registers in the steps above
                const WalkArgs args = load_args(A);
                walk_staged(walk_prep[k], r0 + k, args.R, args.W, args.cfg, args.S, lane, wave, tile_lo, done, tseq);
            }
        }
        k = nk;
    }
    __syncthreads();
    tile_flush(tile_lo, A->S.dense, A->S.dense_lo, A->S.dense_n, (int)threadIdx.x, (int)blockDim.x);
}

__global__ void __launch_bounds__(256) k_anchor(const Anchor* A, const unsigned* n_anchors, unsigned cap, DenseRow* rows,
                                                  int dense_lo, int dense_n, Config cfg) {
    unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    unsigned n = *n_anchors;
    if (n > cap) n = cap;
    if (i < n) anchor_one(i, A, rows, dense_lo, dense_n, cfg);
}

// Copies the listed dense rows into a packed buffer (indices outside the window yield zero rows).
// One lane per 16-byte word.
__global__ void __launch_bounds__(256) k_gather_rows(const DenseRow* rows, int dense_n, const int32_t* idx, int n,
                                                       DenseRow* out) {
    constexpr int WORDS = (int)(sizeof(DenseRow) / 16);
    const int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= (int64_t)n * WORDS) return;
    const int64_t k = w / WORDS;
    const int j = (int)(w - k * WORDS);
    const int r = idx[k];
    uint4 v = make_uint4(0, 0, 0, 0);
    if (r >= 0 && r < dense_n) v = reinterpret_cast<const uint4*>(rows)[(int64_t)r * WORDS + j];
    reinterpret_cast<uint4*>(out)[w] = v;
}

// noPassingReads over the region's records: counts the records passes_one accepts.  One lane per
// record; one counter update per wavefront.
__global__ void __launch_bounds__(256) k_no_passing(const WalkArgs* A, int start, int end, unsigned* count) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool passes = i < A->R.n && passes_one(A->R, i, start, end);
    const unsigned long long m = __ballot(passes);
    if ((threadIdx.x & 63) == 0 && m) atomicAdd(count, (unsigned)__popcll(m));
}

// ---------------------------------------------------------------- launch wrappers
static inline unsigned grid_for(int64_t n, int block) { return (unsigned)((n + block - 1) / block); }

hipError_t launch_prep(const WalkArgs* A, int64_t n, PrepRec* prep, uint32_t* cig, WalkCounters* ctr,
                       PrepCounts* counts, int32_t* rules, bool dedup, bool realign, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    if (n > (int64_t)0x7fffffff) return hipErrorInvalidValue;  // the list holds 32-bit read indices
    if (dedup) {
        hipLaunchKernelGGL(k_dedup, dim3(grid_for(n, 256)), dim3(256), 0, s, A);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(k_prep, dim3(grid_for(n, 256)), dim3(256), 0, s, A, prep, cig, ctr, counts, rules);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || !realign) return e;
    // more wavefronts than the chip holds at once (5 a SIMD, 5,120), each then taking every 8,192nd read;
    // how many are listed is known on the device
    const unsigned blocks = (unsigned)(n < 8192 ? n : 8192);
    hipLaunchKernelGGL(k_prep_rules, dim3(blocks), dim3(64), 0, s, A, prep, cig, ctr, (const PrepCounts*)counts,
                       (const int32_t*)rules);
    return hipGetLastError();
}
hipError_t launch_fill_rows(DenseRow* rows, int n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill_rows, dim3(grid_for(n, 256)), dim3(256), 0, s, rows, n);
    return hipGetLastError();
}
hipError_t launch_walk(const WalkArgs* A, int64_t n, const PrepRec* prep, const uint32_t* cig, int nreads,
                       hipStream_t s) {
    if (n <= 0) return hipSuccess;
    if (nreads < 1 || nreads > WALK_READS_MAX) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_walk, dim3(grid_for(n, nreads)), dim3(WALK_THREADS), 0, s, A, prep, cig, nreads);
    return hipGetLastError();
}
hipError_t launch_no_passing(const WalkArgs* A, int64_t n, int start, int end, unsigned* count, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_no_passing, dim3(grid_for(n, 256)), dim3(256), 0, s, A, start, end, count);
    return hipGetLastError();
}
hipError_t launch_anchor(const Anchor* a, const unsigned* n_anchors, unsigned cap, DenseRow* rows, int dense_lo,
                         int dense_n, const Config& cfg, hipStream_t s) {
    if (cap == 0) return hipSuccess;
    hipLaunchKernelGGL(k_anchor, dim3(grid_for(cap, 256)), dim3(256), 0, s, a, n_anchors, cap, rows, dense_lo, dense_n,
                       cfg);
    return hipGetLastError();
}

hipError_t launch_gather_rows(const DenseRow* rows, int dense_n, const int32_t* idx, int n, DenseRow* out,
                              hipStream_t s) {
    if (n <= 0) return hipSuccess;
    constexpr int WORDS = (int)(sizeof(DenseRow) / 16);
    hipLaunchKernelGGL(k_gather_rows, dim3(grid_for((int64_t)n * WORDS, 256)), dim3(256), 0, s, rows, dense_n, idx, n,
                       out);
    return hipGetLastError();
}

}  // namespace rv
