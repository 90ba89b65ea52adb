// Two-sided Fisher p-value of one 2x2 table by a whole wavefront, the same bits as fisher_two_sided.
//
// The tails are sums of hypergeometric terms, each the one before it times two quotients, and every
// 11th term is computed afresh (hg_acc).  So the stretches between multiples of 11 do not depend on
// each other: each lane computes one, 64 stretches at a time, with the serial code's own steps, and
// the sum then runs over the terms in the serial order with the serial code's checks.  A lane alone
// spends two dependent divisions per term; at a few thousand reads that is most of a position's
// scoring (0.28 of 0.52 ms on a 2.2 kb amplicon at 2500x).
#pragma once
#include "rv_fisher.h"

namespace rv {

constexpr int FISHER_STRETCH = 11;
constexpr int FISHER_TERMS = 64 * FISHER_STRETCH;  // a batch; the caller's LDS array

// One tail: `sum` takes the terms from `idx` on (towards `last`, dir = +1 or -1; p is the term before
// idx and a the state that made it) while they lie below q.  All lanes hold the same values.
__device__ inline void fisher_tail(HG& a, double& p, double& sum, int& idx, int dir, int last, int min, int max, double q,
                                   double* terms, int lane) {
    sum = 0.;
    const auto more = [&] { return p < 0.99999999 * q && (dir > 0 ? idx <= last : idx >= last); };
    while (more()) {
        const int i0 = idx;
        const int stop = dir > 0 ? max : min;  // terms outside [min, max] are not computed ahead
        // the first multiple of 11 from i0 on: lane 0 goes on from the state up to it, lane k takes the
        // stretch that starts at the (k - 1)-th
        const int b0 = dir > 0 ? (i0 + FISHER_STRETCH - 1) / FISHER_STRETCH * FISHER_STRETCH
                               : i0 / FISHER_STRETCH * FISHER_STRETCH;
        const int head = (b0 - i0) * dir;
        HG h = a;
        const int from = lane == 0 ? i0 : b0 + dir * FISHER_STRETCH * (lane - 1);
        const int n = lane == 0 ? head : FISHER_STRETCH;
        for (int t = 0; t < n; t++) {
            const int i = from + dir * t;
            if (dir > 0 ? i > stop : i < stop) break;
            terms[(i - i0) * dir] = hg_acc(i, 0, 0, 0, h);
        }
        __syncthreads();
        const int ahead = (stop - i0) * dir + 1, full = head + 63 * FISHER_STRETCH;
        const int have = ahead < full ? ahead : full;
        int k = 0;
        double next = have > 0 ? terms[0] : 0.;
        while (k < have && more()) {
            sum += p;
            p = next;
            k++;
            idx += dir;
            if (k < have) next = terms[k];
        }
        __syncthreads();
        a.n11 = idx - dir;
        a.p = p;
        if (have <= 0) {  // below min: the serial step
            if (!more()) break;
            sum += p;
            p = hg_acc(idx, 0, 0, 0, a);
            idx += dir;
        }
    }
}

// Every lane of a 64-thread workgroup calls this with the same table and gets the same value.
__device__ inline double fisher_two_sided_wave(int n11, int n12, int n21, int n22, LGTable lg, double* terms, int lane) {
    HG aux{0, 0, 0, 0, 0, lg};
    const int n1_ = n11 + n12, n_1 = n11 + n21, n = n11 + n12 + n21 + n22;
    const int max = n_1 < n1_ ? n_1 : n1_;
    int min = n1_ + n_1 - n;
    if (min < 0) min = 0;
    if (min == max) return 1.;
    const double q = hg_acc(n11, n1_, n_1, n, aux);
    double left, right;
    double p = hg_acc(min, 0, 0, 0, aux);
    int i = min + 1;
    fisher_tail(aux, p, left, i, 1, max, min, max, q, terms, lane);
    if (p < 1.00000001 * q) left += p;
    p = hg_acc(max, 0, 0, 0, aux);
    int j = max - 1;
    fisher_tail(aux, p, right, j, -1, 0, min, max, q, terms, lane);
    if (p < 1.00000001 * q) right += p;
    const double two = left + right;
    return two > 1. ? 1. : two;
}

}  // namespace rv
