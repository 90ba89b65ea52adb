// alignedVariants' robin_hood slot order on the device, one table growth (epoch) at a time.
//
// robin_hood keeps its keys sorted by home slot (an overflow area instead of wrap-around) and,
// within a home, by the info byte's hash bits descending, equal bytes in placement order.  An
// epoch re-inserts the previous table's keys in that table's slot order, then takes its own
// insertions (some erased right after: transient keys).  Per epoch:
//   1. the kept and the transient keys are counted per home; one scan over the homes gives where
//      each home's keys start and the first slot free of earlier homes' keys (a packed home takes
//      x -> max(x, home) + count of that slot, and such maps compose), so displacements and runs
//      (separated by a free slot) can be read off per home;
//   2. the steps are scattered to their homes (their order inside a home is not needed);
//   3. for each run that can reach a displacement of 6, one wavefront finds the first step at which
//      each info-byte overflow displacement (6, 14, 30, 62, 126) is reached.  Every set present in
//      the epoch is a subset of its kept keys plus one transient key, so runs evolve independently,
//      and the packing of the keys placed before a step says what has been reached by then: 64
//      trial steps are packed at once and narrowed, in place of replaying the run's insertions
//      (which took 0.2-0.5 us each, one after another: the longest run's length was the epoch's);
//   4. with the halving steps known, each key's place within its home follows from the hash bits
//      at its placement level, then placement order.
//
// Tables up to SO_SMALL_CAP slots (the first eleven epochs) run in one launch of one workgroup with
// the per-home counters in LDS: such an epoch holds too little work for the chip, and its cost as
// separate launches was their latency.  Larger tables take eight launches per epoch.
#include <hip/hip_runtime.h>

#include "rv_kernels.h"
#include "rv_slotorder_body.h"

namespace rv {

__global__ void __launch_bounds__(SO_SMALL_THREADS) k_so_small(const SoSched* D, const int32_t* ops, const uint8_t* tr,
                                                                int32_t* ord0, int32_t* ord1, int32_t* fin,
                                                                uint32_t* tsteps, unsigned* flags, SoEpochState* large) {
    so_small(D, ops, tr, ord0, ord1, fin, tsteps, flags, large);
}

__global__ void __launch_bounds__(256) k_so_home_count(SoEpoch E) { so_home_count(E); }
__global__ void __launch_bounds__(256) k_so_home_reduce(SoEpoch E) { so_home_reduce(E); }
__global__ void __launch_bounds__(1024) k_so_home_carry(SoEpoch E) { so_home_carry(E); }
__global__ void __launch_bounds__(256) k_so_home_scan(SoEpoch E) { so_home_scan(E); }
__global__ void __launch_bounds__(256) k_so_scatter(SoEpoch E) { so_scatter(E); }
__global__ void __launch_bounds__(64) k_so_simulate(SoEpoch E) { so_simulate(E); }
__global__ void __launch_bounds__(256) k_so_final(SoEpoch E) { so_final(E); }

// ---- alignedVariants' operations: the processing order's positions whose status is nonzero, in
// order (status 2: erased right after its insertion)

// record-list positions override their dense rows' status (one status per window position)
__global__ void __launch_bounds__(256) k_so_status_merge(uint8_t* status, int dense_lo, int dense_n,
                                                          const int32_t* cx_pos, int ncx) {
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= ncx) return;
    const int i = cx_pos[k] - dense_lo;
    if (i >= 0 && i < dense_n) status[i] = status[dense_n + k];
}
__global__ void __launch_bounds__(256) k_so_count(const int32_t* proc, int n, const uint8_t* st, int dense_lo,
                                                   int dense_n, SoBlockCount* bcount, SoSched* D) {
    so_ops_count(proc, n, st, dense_lo, dense_n, bcount, D);
}
__global__ void __launch_bounds__(256) k_so_compact(const int32_t* proc, int n, const uint8_t* st, int dense_lo,
                                                     int dense_n, const SoBlockCount* bcount, int32_t* ops, uint8_t* tr,
                                                     SoSched* D) {
    so_ops_compact(proc, n, st, dense_lo, dense_n, bcount, ops, tr, D);
}

hipError_t launch_so_ops(const int32_t* proc, int n, uint8_t* status, int dense_lo, int dense_n, const int32_t* cx_pos,
                         int ncx, SoBlockCount* bcount, int32_t* ops, uint8_t* tr, SoSched* D, hipStream_t s) {
    hipError_t e;
    if (ncx > 0) {
        hipLaunchKernelGGL(k_so_status_merge, dim3((unsigned)((ncx + 255) / 256)), dim3(256), 0, s, status, dense_lo,
                           dense_n, cx_pos, ncx);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    const unsigned nb = (unsigned)so_blocks(n);
    hipLaunchKernelGGL(k_so_count, dim3(nb), dim3(256), 0, s, proc, n, status, dense_lo, dense_n, bcount, D);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_so_compact, dim3(nb), dim3(256), 0, s, proc, n, status, dense_lo, dense_n, bcount, ops, tr, D);
    return hipGetLastError();
}

hipError_t launch_so_small(const SoSched* D, const int32_t* ops, const uint8_t* tr, int32_t* ord0, int32_t* ord1,
                           int32_t* fin, uint32_t* tsteps, unsigned* flags, SoEpochState* large, hipStream_t s) {
    hipLaunchKernelGGL(k_so_small, dim3(1), dim3(SO_SMALL_THREADS), 0, s, D, ops, tr, ord0, ord1, fin, tsteps, flags,
                       large);
    return hipGetLastError();
}

hipError_t launch_so_epoch(const SoEpoch& E, hipStream_t s) {
    // whole blocks of SO_HB homes; the scans assume it
    if (E.cap < SO_HB || (E.cap & (E.cap - 1)) || E.S <= 0) return hipErrorInvalidValue;
    hipError_t e = hipMemsetAsync(E.st, 0, 2 * sizeof(uint32_t) * (size_t)E.cap, s);  // st and te
    if (e != hipSuccess) return e;
    const dim3 gs((unsigned)((E.S + 255) / 256)), gh((unsigned)(E.cap / SO_HB)), b(256);
    hipLaunchKernelGGL(k_so_home_count, gs, b, 0, s, E);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_so_home_reduce, gh, b, 0, s, E);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_so_home_carry, dim3(1), dim3(1024), 0, s, E);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_so_home_scan, gh, b, 0, s, E);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_so_scatter, gs, b, 0, s, E);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    // 16 wavefronts a CU, of the 26 whose buffers fit: most runs are short, and cost a few dependent reads
    // each
    hipLaunchKernelGGL(k_so_simulate, dim3((unsigned)(E.cap / 64 < 4096 ? E.cap / 64 : 4096)), dim3(64), 0, s, E);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (E.n_keep <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_so_final, dim3((unsigned)((E.n_keep + 255) / 256)), b, 0, s, E);
    return hipGetLastError();
}

// ---- the printer's record order: records by (their position's index in the slot order, position,
// allele order); positions without an alignedVariants key sort after all others

// kept: the number of keys, on the device (the small tables' order is not waited for)
__global__ void __launch_bounds__(256) k_so_rank_scatter(const int32_t* order, const int32_t* kept, int dense_lo,
                                                          int dense_n, int32_t* rank_of) {
    const int r = blockIdx.x * 256 + threadIdx.x;
    if (r >= *kept) return;
    const long long i = (long long)order[r] - dense_lo;
    if (i >= 0 && i < dense_n) rank_of[i] = r;
}

__global__ void __launch_bounds__(256) k_so_rank_keys(const OutRec* recs, int n, const int32_t* rank_of, int dense_lo,
                                                       int dense_n, long long pos_base, unsigned long long* key,
                                                       int32_t* idx, unsigned* bad) {
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j >= n) return;
    const int32_t p = recs[j].position, ord = recs[j].order;
    const long long i = (long long)p - dense_lo;
    const int32_t r = (i >= 0 && i < dense_n) ? rank_of[i] : -1;
    const unsigned long long rk = r < 0 ? 0xffffffull : (unsigned long long)r;
    const long long off = (long long)p - pos_base;
    if (r >= 0xffffff || off < 0 || off >= (1ll << 30) || ord < 0 || ord >= 1024) atomicOr(bad, 1u);
    key[j] = (rk << 40) | ((unsigned long long)(off & ((1ll << 30) - 1)) << 10) | (unsigned long long)(ord & 1023);
    idx[j] = j;
}

hipError_t launch_so_rank(const int32_t* order, const int32_t* kept, int max_keep, const OutRec* recs, int n, int dense_lo, int dense_n,
                          long long pos_base, int32_t* rank_of, unsigned long long* key, int32_t* idx, unsigned* bad,
                          hipStream_t s) {
    hipError_t e;
    if (dense_n > 0 && (e = hipMemsetAsync(rank_of, 0xff, sizeof(int32_t) * (size_t)dense_n, s)) != hipSuccess) return e;
    if (max_keep > 0) {
        hipLaunchKernelGGL(k_so_rank_scatter, dim3((unsigned)((max_keep + 255) / 256)), dim3(256), 0, s, order, kept,
                           dense_lo, dense_n, rank_of);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    if (n > 0) {
        hipLaunchKernelGGL(k_so_rank_keys, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, recs, n, rank_of, dense_lo,
                           dense_n, pos_base, key, idx, bad);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace rv
