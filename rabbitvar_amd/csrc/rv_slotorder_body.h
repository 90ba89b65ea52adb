// Device bodies of the slot-order kernels (rv_slotorder.hip, which describes the method).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "rv_slotorder.h"

namespace rv {

__device__ inline unsigned long long so_mix(int32_t k) {
    const unsigned long long x = (unsigned long long)(long long)k;
    return __umul64hi(x, 0xde5fb9d2630458e9ull) + x * 0xde5fb9d2630458e9ull;
}

// displacement at which an info byte overflows at increments 32, 16, 8, 4, 2: 6, 14, 30, 62, 126
__device__ inline int so_disp(int level) { return (8 << level) - 2; }

// The map x -> max(x + a, b) of "first slot free of the keys so far" over a range of homes (a =
// its keys), with its transient keys beside it.  A home h with c > 0 keys is (c, h + c).
struct SoMap {
    int a, b, t;
};
constexpr int SO_NONE = -(1 << 29);  // b of a range without keys
__device__ inline SoMap so_then(const SoMap& f, const SoMap& g) {  // f first
    const int fb = f.b + g.a;
    return {f.a + g.a, fb > g.b ? fb : g.b, f.t + g.t};
}
// the first free slot after the keys of `f`, from an empty table (-1: none, so that home 0 starts
// a run like any other)
__device__ inline int so_free(const SoMap& f) { return f.a == 0 ? -1 : f.b; }

// inclusive scan over the wavefront
__device__ inline SoMap so_wave_scan(SoMap m, int lane) {
    for (int o = 1; o < 64; o <<= 1) {
        const SoMap p{__shfl_up(m.a, o), __shfl_up(m.b, o), __shfl_up(m.t, o)};
        if (lane >= o) m = so_then(p, m);
    }
    return m;
}
// exclusive scan over a workgroup of WAVES wavefronts; *total = all of it.  `tot`: WAVES entries of
// LDS, free again after the next barrier.
template <int WAVES>
__device__ inline SoMap so_block_scan(const SoMap& mine, SoMap* tot, int tid, SoMap* total) {
    const int lane = tid & 63, wave = tid >> 6;
    const SoMap inc = so_wave_scan(mine, lane);
    if (lane == 63) tot[wave] = inc;
    SoMap ex{__shfl_up(inc.a, 1), __shfl_up(inc.b, 1), __shfl_up(inc.t, 1)};
    if (lane == 0) ex = SoMap{0, SO_NONE, 0};
    __syncthreads();
    SoMap before{0, SO_NONE, 0}, all{0, SO_NONE, 0};
    for (int w = 0; w < WAVES; w++) {
        if (w < wave) before = so_then(before, tot[w]);
        all = so_then(all, tot[w]);
    }
    if (total) *total = all;
    return so_then(before, ex);
}

// An epoch's per-home state once its steps are scattered: st[h] / te[h] = the end of home h's kept /
// transient steps in step / tstep (home h - 1's end is its start), nf[h] = 1 + the first slot free
// of earlier homes' keys.
template <class NF>
struct SoHomes {
    const uint32_t *st, *te;
    const NF* nf;
    const uint32_t *step, *tstep;
    const uint16_t* hm;  // each kept step's home, or null (it then follows from the key)
    const int32_t *prev, *ops;
    int np, steps, cap, n_keep, n_tr, x_end;
    uint32_t mask;
    __device__ int start(int h) const { return h > 0 ? (int)st[h - 1] : 0; }
    __device__ int count(int h) const { return (int)st[h] - start(h); }
    __device__ int tstart(int h) const { return h > 0 ? (int)te[h - 1] : 0; }
    __device__ int x(int h) const { return (int)nf[h] - 1; }
    __device__ int32_t key(uint32_t s) const { return s < (uint32_t)np ? prev[s] : ops[s - (uint32_t)np]; }
    __device__ int home(uint32_t s) const { return (int)(so_mix(key(s)) & mask); }
};

#define SO_WAVE_SYNC() __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront")

// The largest displacement of those of a run's n kept keys that are placed before step T (es, eh:
// their steps and homes, grouped by home; off: the run's first home), with one more key of home u
// when EXTRA.  Every lane has its own T and u; the keys are the same for all.
template <bool EXTRA>
__device__ inline int so_packed(const uint32_t* es, const uint16_t* eh, int off, int n, unsigned T, int u) {
    int x = 0, md = -1;  // x: the first slot free of the keys so far
    bool left = EXTRA;
#pragma unroll 4
    for (int i = 0; i < n; i++) {
        const int h = (int)eh[i] - off;
        if (EXTRA && left && h > u) {
            x = (x > u ? x : u) + 1;
            md = x - 1 - u > md ? x - 1 - u : md;
            left = false;
        }
        if (es[i] < T) {
            x = (x > h ? x : h) + 1;
            md = x - 1 - h > md ? x - 1 - h : md;
        }
    }
    if (EXTRA && left) {
        x = (x > u ? x : u) + 1;
        md = x - 1 - u > md ? x - 1 - u : md;
    }
    return md;
}

__device__ inline unsigned so_wave_min(unsigned v) {
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned w = __shfl_xor(v, o);
        v = w < v ? w : v;
    }
    return v;
}

// LDS copy of one run's kept keys (the larger tables' are in global memory)
struct SoRunLds {
    uint32_t es[SO_RUN_MAX];
    uint16_t eh[SO_RUN_MAX];
};

// One wavefront: the run whose first home with a displacement of 5 or more is h (others return at
// once).  Lowers first[l] to the first step at which the run reaches displacement so_disp(l).  Its
// kept keys' displacements only grow, so that step is found by packing the keys placed before 64
// trial steps at once, one per lane, and narrowing; a transient key is tried against the keys
// placed before it.  COPY: the run's keys go to `copy` first (else H, in LDS, holds their homes);
// returns false, with nothing done, when they do not fit it.
template <bool COPY, class NF>
__device__ inline bool so_run(const SoHomes<NF>& H, int h, int lane, SoRunLds* copy, unsigned* first) {
    // the run's first home, and whether an earlier home of it reaches a displacement of 5
    int a = -1;
    for (int base = h; base >= 0; base -= 64) {
        const int hh = base - lane;
        const bool in = hh >= 0;
        const int c = in ? H.count(hh) : 0, xx = in ? H.x(hh) : 0;
        const bool head = c > 0 && xx < hh;
        const bool deep = hh < h && c > 0 && (xx > hh ? xx : hh) + c - 1 - hh >= 5;
        const unsigned long long mh = __ballot(head), md = __ballot(deep);
        const int f = mh ? __ffsll((long long)mh) - 1 : 64;
        if (md & (f < 63 ? (2ull << f) - 1ull : ~0ull)) return true;
        if (mh) {
            a = base - f;
            break;
        }
    }
    if (a < 0) return true;
    // its end (the first later home past a free slot) and largest displacement
    int maxd = 0, hi = H.n_keep, xe = H.x_end;
    for (int base = h; base < H.cap; base += 64) {
        const int hh = base + lane;
        const bool in = hh < H.cap;
        const int c = in ? H.count(hh) : 0, xx = in ? H.x(hh) : 0;
        const unsigned long long me = __ballot(in && hh > h && xx < hh);
        const int f = me ? __ffsll((long long)me) - 1 : 64;
        const int d = lane < f && c > 0 ? (xx > hh ? xx : hh) + c - 1 - hh : 0;
        for (int l = 0; l < 5; l++)
            if (__ballot(d >= so_disp(l) - 1)) maxd = maxd > so_disp(l) - 1 ? maxd : so_disp(l) - 1;
        for (int l = 0; l < 5; l++)
            if (__ballot(d >= so_disp(l))) maxd = maxd > so_disp(l) ? maxd : so_disp(l);
        if (me) {
            hi = H.start(base + f);
            xe = H.x(base + f);
            break;
        }
    }
    if (maxd >= so_disp(4)) {  // reached, at whichever step: the table grows early
        // (stored by every lane: the end of a branch on the lane would be joined to the one that takes
        // the caller's next run, and lanes that skip both would go around its loop without lane 0)
        *(volatile unsigned*)&first[4] = 0u;
        return true;
    }
    const int lo = H.start(a), last = xe - 1;
    const int t0 = H.tstart(a);
    const int t1 = last >= H.cap ? H.n_tr : (int)H.te[last];
    const int nk = hi - lo, nt = t1 - t0;
    int top = -1;
    for (int l = 0; l < 5 && maxd + (nt > 0 ? 1 : 0) >= so_disp(l); l++) top = l;
    if (top < 0) return true;
    if (COPY) {
        if (nk > SO_RUN_MAX) return false;
        for (int i = lane; i < nk; i += 64) {
            const uint32_t s = H.step[lo + i];
            copy->es[i] = s;
            copy->eh[i] = (uint16_t)(H.home(s) - a);
        }
        SO_WAVE_SYNC();
    }
    const uint32_t* es = COPY ? copy->es : H.step + lo;
    const uint16_t* eh = COPY ? copy->eh : H.hm + lo;
    const int off = COPY ? 0 : a;
    if (nk <= 64) {
        // every kept step is a trial
        const uint32_t s = lane < nk ? es[lane] : ~0u;
        const int md = so_packed<false>(es, eh, off, nk, lane < nk ? s + 1u : 0u, 0);
        for (int l = 0; l <= top; l++) {
            const unsigned m = so_wave_min(md >= so_disp(l) ? s : ~0u);
            if (lane == 0 && m < *(volatile unsigned*)&first[l]) atomicMin(&first[l], m);
        }
    } else {
        unsigned from = 0;  // not reached by the keys placed before it
        for (int l = 0; l <= top; l++) {
            const unsigned fl = *(volatile unsigned*)&first[l];
            unsigned to = fl < (unsigned)H.steps ? fl : (unsigned)H.steps;
            bool any = false;
            while (to > from) {
                const unsigned by = (to - from + 63) / 64;
                const unsigned T = to - from > by * (unsigned)(lane + 1) ? from + by * (unsigned)(lane + 1) : to;
                const unsigned long long m = __ballot(so_packed<false>(es, eh, off, nk, T, 0) >= so_disp(l));
                if (!m) break;  // not before `to`
                any = true;
                const int f = __ffsll((long long)m) - 1;
                to = (unsigned)__shfl((int)T, f);
                if (f > 0) from = (unsigned)__shfl((int)T, f - 1);
                if (by == 1) break;
            }
            if (any && lane == 0) atomicMin(&first[l], to - 1u);
        }
    }
    for (int j0 = 0; j0 < nt; j0 += 256) {
        unsigned t[4];
        const unsigned fl = *(volatile unsigned*)&first[top];  // they do not decrease with the level
#pragma unroll
        for (int k = 0; k < 4; k++) t[k] = j0 + 64 * k + lane < nt ? H.tstep[t0 + j0 + 64 * k + lane] : ~0u;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if (!__ballot(t[k] < fl)) continue;
            const int md = so_packed<true>(es, eh, off, nk, t[k], t[k] < fl ? H.home(t[k]) - a : 0);
            for (int l = 0; l <= top; l++) {
                const unsigned m = so_wave_min(t[k] < fl && md >= so_disp(l) ? t[k] : ~0u);
                if (lane == 0 && m < *(volatile unsigned*)&first[l]) atomicMin(&first[l], m);
            }
        }
    }
    SO_WAVE_SYNC();
    return true;
}

// The halving steps of an epoch from the first steps reaching each displacement: a flag raised at
// step t halves the increment before step t + 1 (when there is one).
struct SoHalve {
    int nh;
    uint32_t at[4];
};
__device__ inline SoHalve so_halvings(const unsigned* first, int S) {
    SoHalve H;
    H.nh = 0;
    for (int l = 0; l < 4; l++) {
        const unsigned f = first[l];
        H.at[l] = f + 1u;
        if (f != 0xffffffffu && f + 1u < (unsigned)S) H.nh = l + 1;
    }
    return H;
}
// a key's rank among the keys of its home: smaller first (then the placement step)
__device__ inline uint32_t so_level_key(const SoHalve& H, uint32_t step, int32_t k) {
    const uint32_t hb = (uint32_t)(so_mix(k) >> 59);
    int ph = 0;
    while (ph < H.nh && H.at[ph] <= step) ph++;
    uint32_t c = (~(hb >> H.nh)) & ((1u << (5 - H.nh)) - 1u);
    for (int l = H.nh - 1; l >= 0; l--) {
        const uint32_t late = ph > l ? 1u : 0u;
        const uint32_t bit = late ? 0u : ((~hb >> l) & 1u);
        c = (c << 2) | (late << 1) | bit;
    }
    return c;
}
// kept key i of the home-grouped steps to its place in slot order
template <class NF>
__device__ inline void so_place(const SoHomes<NF>& H, const SoHalve& L, int i, int32_t* out, unsigned* flags) {
    const uint32_t s = H.step[i];
    const int32_t key = H.key(s);
    const int home = (int)(so_mix(key) & H.mask);
    const int g0 = H.start(home), g1 = (int)H.st[home];
    if (g1 - g0 >= SO_GROUP_MAX) {
        atomicOr(&flags[SO_F_GROUP], 1u);
        return;
    }
    int rank = 0;
    if (g1 - g0 > 1) {
        const uint32_t mine = so_level_key(L, s, key);
        for (int j = g0; j < g1; j++) {
            const uint32_t sj = H.step[j];
            if (sj == s) continue;
            const uint32_t cj = so_level_key(L, sj, H.key(sj));
            if (cj < mine || (cj == mine && sj < s)) rank++;
        }
    }
    out[g0 + rank] = key;
}

// ---------------------------------------------------------------- small tables, one workgroup
constexpr int SO_W = SO_SMALL_THREADS / 64;
__device__ inline void so_small(const SoSched* D, const int32_t* ops, const uint8_t* tr, int32_t* ord0, int32_t* ord1,
                                int32_t* fin, uint32_t* tsteps, unsigned* flags, SoEpochState* large) {
    __shared__ uint32_t st[SO_SMALL_CAP], te[SO_SMALL_CAP], step[SO_SMALL_KEEP];
    // a home in list holds two keys or more
    __shared__ uint16_t nf[SO_SMALL_CAP], hm[SO_SMALL_KEEP], list[SO_SMALL_KEEP / 2];
    __shared__ SoMap tot[SO_W];
    __shared__ unsigned first[5];
    __shared__ int n_list, n_next;
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // every sequence starts here: the flags and the larger tables' state
    if (tid < SO_FLAGS) flags[tid] = 0u;
    if (tid < SO_EPOCHS_MAX) {
        for (int l = 0; l < 5; l++) large[tid].first[l] = 0xffffffffu;
        large[tid].n_list = 0u;
    }
    __syncthreads();
    for (int e = 0;; e++) {
        SoEpochRange r;
        if (!so_epoch_range(*D, e, r) || r.cap > SO_SMALL_CAP) return;
        const int cap = r.cap, np = r.np, S = r.np + (r.b - r.a), n_keep = r.keep;
        const int32_t* prev = (e & 1) ? ord1 : ord0;
        int32_t* out = r.last ? fin : ((e & 1) ? ord0 : ord1);
        const int32_t* eops = ops + r.a;
        const uint8_t* etr = tr + r.a;
        const uint32_t mask = (uint32_t)cap - 1u;
        for (int h = tid; h < cap; h += SO_SMALL_THREADS) st[h] = te[h] = 0u;
        if (tid < 5) first[tid] = 0xffffffffu;
        if (tid == 0) n_list = n_next = 0;
        __syncthreads();
        for (int s = tid; s < S; s += SO_SMALL_THREADS) {
            const int32_t k = s < np ? prev[s] : eops[s - np];
            const bool t = tr && s >= np && etr[s - np];
            atomicAdd(&(t ? te : st)[so_mix(k) & mask], 1u);
        }
        __syncthreads();
        {
            const int per = cap > SO_SMALL_THREADS ? cap / SO_SMALL_THREADS : 1;
            const int h0 = tid * per < cap ? tid * per : cap, h1 = h0 + per < cap ? h0 + per : cap;
            SoMap m{0, SO_NONE, 0};
            for (int h = h0; h < h1; h++) {
                const int c = (int)st[h];
                m = so_then(m, SoMap{c, c > 0 ? h + c : SO_NONE, (int)te[h]});
            }
            const SoMap before = so_block_scan<SO_W>(m, tot, tid, nullptr);
            int at = before.a, tat = before.t, x = so_free(before);
            for (int h = h0; h < h1; h++) {
                const int c = (int)st[h], ct = (int)te[h];
                st[h] = (uint32_t)at;
                te[h] = (uint32_t)tat;
                nf[h] = (uint16_t)(x + 1);
                at += c;
                tat += ct;
                if (c > 0) {
                    const int xn = (x > h ? x : h) + c;
                    // the first home of a stretch with displacements of 5 or more
                    if (xn - 1 - h >= 5 && x - h < 5) list[atomicAdd(&n_list, 1)] = (uint16_t)h;
                    x = xn;
                }
            }
        }
        __syncthreads();
        for (int s = tid; s < S; s += SO_SMALL_THREADS) {
            const int32_t k = s < np ? prev[s] : eops[s - np];
            const int h = (int)(so_mix(k) & mask);
            if (tr && s >= np && etr[s - np])
                tsteps[atomicAdd(&te[h], 1u)] = (uint32_t)s;
            else {
                const uint32_t at = atomicAdd(&st[h], 1u);
                step[at] = (uint32_t)s;
                hm[at] = (uint16_t)h;
            }
        }
        __syncthreads();
        SoMap all{0, SO_NONE, 0};
        for (int w = 0; w < SO_W; w++) all = so_then(all, tot[w]);
        const SoHomes<uint16_t> H{st,  te,  nf,  step,   tsteps, hm, prev,         eops,
                                  np,  S,   cap, n_keep, S - n_keep, so_free(all), mask};
        for (;;) {
            int i = 0;
            if (lane == 0) i = atomicAdd(&n_next, 1);
            i = __builtin_amdgcn_readfirstlane(__shfl(i, 0));
            if (i >= n_list) break;
            (void)so_run<false>(H, (int)list[i], lane, nullptr, first);
        }
        __syncthreads();
        if (first[4] != 0xffffffffu) {  // an early growth: no later table's order would hold
            if (tid == 0) atomicOr(&flags[SO_F_GROW], 1u);
            return;
        }
        const SoHalve L = so_halvings(first, S);
        for (int i = tid; i < n_keep; i += SO_SMALL_THREADS) so_place(H, L, i, out, flags);
        __syncthreads();
    }
}

// ---------------------------------------------------------------- larger tables, one launch per step
// Whether an earlier step found that the order does not hold: the steps after it are left out (their
// input may never have been written).  Positions inserted in another table's slot order (-p, where
// nearly all of them stay) crowd the low homes of each smaller table into one run of half its keys, which
// the trial packings go through one key after another: 20 kb at 30x, whose table of 2,048 slots grows
// early, 6.9 ms with every table worked out and 0.57 up to that one.
__device__ inline bool so_declined(const SoEpoch& E) {
    return (E.flags[SO_F_RUN] | E.flags[SO_F_GROUP] | E.flags[SO_F_GROW]) != 0u;
}
__device__ inline void so_home_count(const SoEpoch& E) {
    const int s = (int)(blockIdx.x * 256 + threadIdx.x);
    if (s >= E.S || so_declined(E)) return;
    const int32_t k = s < E.np ? E.prev[s] : E.ops[s - E.np];
    const bool t = E.tr && s >= E.np && E.tr[s - E.np];
    atomicAdd(&(t ? E.te : E.st)[so_mix(k) & E.mask], 1u);
}

// the map of this thread's SO_HB / 256 homes
__device__ inline SoMap so_homes_of(const SoEpoch& E, int h0) {
    SoMap m{0, SO_NONE, 0};
    for (int h = h0; h < h0 + SO_HB / 256; h++) {
        const int c = (int)E.st[h];
        m = so_then(m, SoMap{c, c > 0 ? h + c : SO_NONE, (int)E.te[h]});
    }
    return m;
}

__device__ inline void so_home_reduce(const SoEpoch& E) {
    if (so_declined(E)) return;
    __shared__ SoMap tot[4];
    const int tid = (int)threadIdx.x;
    SoMap all;
    (void)so_block_scan<4>(so_homes_of(E, (int)blockIdx.x * SO_HB + tid * (SO_HB / 256)), tot, tid, &all);
    if (tid == 0) {
        E.carry[3 * blockIdx.x] = all.a;
        E.carry[3 * blockIdx.x + 1] = all.b;
        E.carry[3 * blockIdx.x + 2] = all.t;
    }
}

// exclusive scan of the blocks' maps, in place; the table's end
__device__ inline void so_home_carry(const SoEpoch& E) {
    if (so_declined(E)) return;
    __shared__ SoMap tot[16];
    const int tid = (int)threadIdx.x, nb = E.cap / SO_HB;
    const int per = (nb + 1023) / 1024;
    const int b0 = tid * per < nb ? tid * per : nb, b1 = b0 + per < nb ? b0 + per : nb;
    SoMap m{0, SO_NONE, 0};
    for (int b = b0; b < b1; b++) m = so_then(m, SoMap{E.carry[3 * b], E.carry[3 * b + 1], E.carry[3 * b + 2]});
    SoMap all;
    SoMap at = so_block_scan<16>(m, tot, tid, &all);
    for (int b = b0; b < b1; b++) {
        const SoMap v{E.carry[3 * b], E.carry[3 * b + 1], E.carry[3 * b + 2]};
        E.carry[3 * b] = at.a;
        E.carry[3 * b + 1] = at.b;
        E.carry[3 * b + 2] = at.t;
        at = so_then(at, v);
    }
    if (tid == 0) E.state->x_end = so_free(all);
}

__device__ inline void so_home_scan(const SoEpoch& E) {
    if (so_declined(E)) return;
    __shared__ SoMap tot[4];
    constexpr int PER = SO_HB / 256;
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int h0 = (int)blockIdx.x * SO_HB + tid * PER;
    const SoMap carry{E.carry[3 * blockIdx.x], E.carry[3 * blockIdx.x + 1], E.carry[3 * blockIdx.x + 2]};
    const SoMap before = so_then(carry, so_block_scan<4>(so_homes_of(E, h0), tot, tid, nullptr));
    int at = before.a, tat = before.t, x = so_free(before);
    unsigned deep = 0;  // this thread's homes that start a stretch with displacements of 5 or more
    for (int j = 0; j < PER; j++) {
        const int h = h0 + j, c = (int)E.st[h], ct = (int)E.te[h];
        E.st[h] = (uint32_t)at;
        E.te[h] = (uint32_t)tat;
        E.nf[h] = (uint32_t)(x + 1);
        at += c;
        tat += ct;
        if (c > 0) {
            const int xn = (x > h ? x : h) + c;
            if (xn - 1 - h >= 5 && x - h < 5) deep |= 1u << j;
            x = xn;
        }
    }
    // one counter update per wavefront
    const int mine = __popcll((unsigned long long)deep);
    int inc = mine;
    for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(inc, o);
        if (lane >= o) inc += v;
    }
    int base = 0;
    if (lane == 63 && inc > 0) base = (int)atomicAdd(&E.state->n_list, (unsigned)inc);
    base = __shfl(base, 63) + inc - mine;
    for (int j = 0; j < PER; j++)
        if (deep >> j & 1u) E.list[base++] = h0 + j;
}

__device__ inline void so_scatter(const SoEpoch& E) {
    const int s = (int)(blockIdx.x * 256 + threadIdx.x);
    if (s >= E.S || so_declined(E)) return;
    const int32_t k = s < E.np ? E.prev[s] : E.ops[s - E.np];
    const int h = (int)(so_mix(k) & E.mask);
    if (E.tr && s >= E.np && E.tr[s - E.np])
        E.tstep[atomicAdd(&E.te[h], 1u)] = (uint32_t)s;
    else
        E.step[atomicAdd(&E.st[h], 1u)] = (uint32_t)s;
}

__device__ inline SoHomes<uint32_t> so_homes(const SoEpoch& E) {
    return SoHomes<uint32_t>{E.st, E.te,  E.nf,     E.step,           E.tstep, nullptr, E.prev, E.ops,
                             E.np, E.S,   E.cap, E.n_keep, E.S - E.n_keep, E.state->x_end, E.mask};
}

__device__ inline void so_simulate(const SoEpoch& E) {
    __shared__ SoRunLds copy;
    if (so_declined(E)) return;
    const int lane = (int)threadIdx.x;
    const SoHomes<uint32_t> H = so_homes(E);
    const int n = (int)E.state->n_list;
    for (int i = (int)blockIdx.x; i < n; i += (int)gridDim.x)
        if (!so_run<true>(H, E.list[i], lane, &copy, E.state->first) && lane == 0)
            atomicOr(&E.flags[SO_F_RUN], 1u);
}

__device__ inline void so_final(const SoEpoch& E) {
    const int i = (int)(blockIdx.x * 256 + threadIdx.x);
    if (i >= E.n_keep || so_declined(E)) return;
    if (i == 0 && E.state->first[4] != 0xffffffffu) atomicOr(&E.flags[SO_F_GROW], 1u);
    so_place(so_homes(E), so_halvings(E.state->first, E.S), i, E.out, E.flags);
}

// ---------------------------------------------------------------- the operations
__device__ inline int so_status(const uint8_t* st, int dense_lo, int dense_n, int32_t p) {
    const long long i = (long long)p - dense_lo;
    return (i >= 0 && i < dense_n) ? st[i] : 0;
}

// operations and kept keys per block of SO_CB processing entries
__device__ inline void so_ops_count(const int32_t* proc, int n, const uint8_t* st, int dense_lo, int dense_n,
                                    SoBlockCount* bcount, SoSched* D) {
    __shared__ int wsum[4], wkept[4];
    const int tid = (int)threadIdx.x, base = (int)blockIdx.x * SO_CB;
    if (blockIdx.x == 0 && tid < SO_EPOCHS_MAX) D->grow[tid] = 0x7fffffff;
    int c = 0, k = 0;
    for (int j = 0; j < SO_CB / 256; j++) {
        const int i = base + j * 256 + tid;
        const int v = i < n ? so_status(st, dense_lo, dense_n, proc[i]) : 0;
        c += __popcll(__ballot(v != 0));
        k += __popcll(__ballot(v != 0 && v != 2));
    }
    if ((tid & 63) == 0) {
        wsum[tid >> 6] = c;
        wkept[tid >> 6] = k;
    }
    __syncthreads();
    if (tid == 0) bcount[blockIdx.x] = SoBlockCount{wsum[0] + wsum[1] + wsum[2] + wsum[3], wkept[0] + wkept[1] + wkept[2] + wkept[3]};
}

// the operations written in processing order, and the growth schedule: the operation after the one
// that fills a table to its load limit grows it
__device__ inline void so_ops_compact(const int32_t* proc, int n, const uint8_t* st, int dense_lo, int dense_n,
                                      const SoBlockCount* bcount, int32_t* ops, uint8_t* tr, SoSched* D) {
    __shared__ int wcnt[4], wkept[4];
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int base = (int)blockIdx.x * SO_CB;
    int run = 0, kept = 0;  // operations and kept keys before this block
    for (int b = tid; b < (int)blockIdx.x; b += 256) {
        run += bcount[b].ops;
        kept += bcount[b].kept;
    }
    for (int o = 32; o > 0; o >>= 1) {
        run += __shfl_xor(run, o);
        kept += __shfl_xor(kept, o);
    }
    if (lane == 0) {
        wcnt[wave] = run;
        wkept[wave] = kept;
    }
    __syncthreads();
    run = wcnt[0] + wcnt[1] + wcnt[2] + wcnt[3];
    kept = wkept[0] + wkept[1] + wkept[2] + wkept[3];
    __syncthreads();
    for (int j = 0; j < SO_CB / 256; j++) {
        const int i = base + j * 256 + tid;
        const int32_t p = i < n ? proc[i] : 0;
        const int v = i < n ? so_status(st, dense_lo, dense_n, p) : 0;
        const bool keep = v != 0 && v != 2;
        const unsigned long long m = __ballot(v != 0), mk = __ballot(keep);
        if (lane == 0) {
            wcnt[wave] = __popcll(m);
            wkept[wave] = __popcll(mk);
        }
        __syncthreads();
        int woff = 0, koff = 0;
        for (int w = 0; w < wave; w++) {
            woff += wcnt[w];
            koff += wkept[w];
        }
        if (v) {
            const unsigned long long below = (1ull << lane) - 1ull;
            const int at = run + woff + __popcll(m & below);
            ops[at] = p;
            tr[at] = v == 2 ? 1 : 0;
            if (keep) {
                const int count = kept + koff + __popcll(mk & below) + 1;  // keys present after it
                if (count >= 6) {
                    const int e = 63 - __clzll((unsigned long long)(count / 6));  // the one table this can fill
                    if (e < SO_EPOCHS_MAX && so_limit(8ll << e) == count) D->grow[e] = at + 1;
                }
            }
        }
        run += wcnt[0] + wcnt[1] + wcnt[2] + wcnt[3];
        kept += wkept[0] + wkept[1] + wkept[2] + wkept[3];
        __syncthreads();
    }
    if (blockIdx.x == gridDim.x - 1 && tid == 0) {
        D->m = run;
        D->kept = kept;
    }
}

}  // namespace rv
