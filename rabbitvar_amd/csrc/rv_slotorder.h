// Layouts of the device slot order (rv_slotorder.hip) shared by the kernels and the engine.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace rv {

constexpr int SO_RUN_MAX = 1024;  // kept keys of one run of a larger table (more: SO_F_RUN)
constexpr int SO_GROUP_MAX = 64;  // keys of one home
constexpr int SO_EPOCHS_MAX = 28; // tables of 8 << 0 .. 8 << 27 slots
constexpr int SO_HB = 2048;       // homes per workgroup of a large table's scans
constexpr int SO_CB = 2048;       // processing entries per workgroup
// The one-workgroup kernel's largest table: its counters (4 B of kept and of transient steps, 2 B of
// free slot per home, 6 B per kept step) fill most of one CU's 160 KB of LDS.
constexpr int SO_SMALL_CAP = 8192;
constexpr int SO_SMALL_KEEP = SO_SMALL_CAP * 80 / 100;
constexpr int SO_SMALL_THREADS = 1024;

// an insertion that finds this many of `cap` slots used doubles the table first
__host__ __device__ inline long long so_limit(long long cap) { return cap * 80 / 100; }

// The operations' growth schedule: grow[e] = the operation after the one that fills table e (8 << e
// slots) to its limit, or INT_MAX; the table grows when there is such an operation.
struct SoSched {
    int32_t m, kept;  // operations, keys present at the end
    int32_t grow[SO_EPOCHS_MAX];
};
struct SoEpochRange {
    int cap, a, b;  // operations [a, b)
    int np, keep;   // keys re-inserted first, keys present at the end
    bool last;
};
__host__ __device__ inline bool so_epoch_range(const SoSched& D, int e, SoEpochRange& r) {
    if (e >= SO_EPOCHS_MAX || (e > 0 && D.grow[e - 1] >= D.m)) return false;
    r.cap = 8 << e;
    r.a = e > 0 ? D.grow[e - 1] : 0;
    r.last = e + 1 >= SO_EPOCHS_MAX || D.grow[e] >= D.m;
    r.b = r.last ? D.m : D.grow[e];
    r.np = e > 0 ? (int)so_limit(4ll << e) : 0;
    r.keep = r.last ? D.kept : (int)so_limit(8ll << e);
    return true;
}

// flags raised by the kernels; any of them: the order does not hold and the host works it out
enum : int { SO_F_RUN = 0, SO_F_GROUP = 1, SO_F_GROW = 2, SO_FLAGS = 4 };

struct SoBlockCount {
    int32_t ops, kept;
};

inline int so_blocks(int n) { return n > SO_CB ? (n + SO_CB - 1) / SO_CB : 1; }

struct SoEpochState {
    unsigned first[5];  // the first step reaching each overflow displacement (~0: none)
    unsigned n_list;
    int32_t x_end;  // the first slot after the last key
    int32_t pad;
};

struct SoEpoch {  // one table of more than SO_SMALL_CAP slots
    const int32_t* prev;  // the previous table's keys in slot order (re-inserted first)
    int np;
    const int32_t* ops;  // the epoch's operations (keys) and transient flags (nullptr: none)
    const uint8_t* tr;
    int S;       // np + operations
    int n_keep;  // keys present at the epoch's end
    int cap;
    uint32_t mask;
    uint32_t *st, *te, *nf;  // per home (te follows st in memory)
    uint32_t *step, *tstep;  // kept steps by home (n_keep), transient ones (S - n_keep)
    int32_t* carry;          // three per SO_HB homes
    int32_t* list;           // homes whose runs may need simulating (at most cap / 2)
    SoEpochState* state;     // set up by the small tables' kernel
    int32_t* out;
    unsigned* flags;
};

}  // namespace rv
