// Kernel launch interface of the pileup / scoring device stages.
#pragma once
#include <hip/hip_runtime.h>

#include "rv_pileup_body.h"
#include "rv_score.h"
#include "rv_slotorder.h"

namespace rv {

// what the prep pass counts beside WalkCounters; starts at zero
struct PrepCounts {
    int max_span;
    unsigned n_rules;  // reads listed for the CIGAR rewrite rules
};
// rules: room for n read indices
hipError_t launch_prep(const WalkArgs* A, int64_t n, PrepRec* prep, uint32_t* cig, WalkCounters* ctr,
                       PrepCounts* counts, int32_t* rules, bool dedup, bool realign, hipStream_t s);
hipError_t launch_fill_rows(DenseRow* rows, int n, hipStream_t s);
hipError_t launch_walk(const WalkArgs* A, int64_t n, const PrepRec* prep, const uint32_t* cig, int nreads,
                       hipStream_t s);
hipError_t launch_no_passing(const WalkArgs* A, int64_t n, int start, int end, unsigned* count, hipStream_t s);
hipError_t launch_anchor(const Anchor* a, const unsigned* n_anchors, unsigned cap, DenseRow* rows, int dense_lo,
                         int dense_n, const Config& cfg, hipStream_t s);

static_assert(sizeof(DenseRow) % 16 == 0, "dense rows are copied in 16-byte words");
hipError_t launch_gather_rows(const DenseRow* rows, int dense_n, const int32_t* idx, int n, DenseRow* out,
                              hipStream_t s);

hipError_t launch_key_list(const DenseRow* rows, int dense_n, int dense_lo, unsigned long long* keys, int32_t* pos,
                           unsigned* count, hipStream_t s);
hipError_t launch_slot_keys(const int32_t* keys, int n, int cap_log2, int idx_bits, unsigned long long* comp,
                            int32_t* val, hipStream_t s);
// temp == nullptr: sets temp_bytes only
hipError_t sort_key_pairs(void* temp, size_t& temp_bytes, const unsigned long long* kin, unsigned long long* kout,
                          const int32_t* vin, int32_t* vout, int n, int end_bit, hipStream_t s);

// ---- robin_hood slot order by growth epochs (rv_slotorder.hip)
// alignedVariants' operations: the entries of `proc` (n positions, the processing order) whose
// status is nonzero, in order, after the record-list positions' status overrides their dense rows'
// (status holds dense_n rows then ncx record-list positions), and their growth schedule.  bcount:
// so_blocks(n) entries.
hipError_t launch_so_ops(const int32_t* proc, int n, uint8_t* status, int dense_lo, int dense_n, const int32_t* cx_pos,
                         int ncx, SoBlockCount* bcount, int32_t* ops, uint8_t* tr, SoSched* D, hipStream_t s);
// clears flags and the larger tables' state, then the epochs of tables up to SO_SMALL_CAP slots: each
// epoch's slot order into ord1, ord0, ord1, ..., the last one of the schedule into fin; tr may be
// null (no transient keys); tsteps: as many entries as transient keys
hipError_t launch_so_small(const SoSched* D, const int32_t* ops, const uint8_t* tr, int32_t* ord0, int32_t* ord1,
                           int32_t* fin, uint32_t* tsteps, unsigned* flags, SoEpochState* large, hipStream_t s);
// one epoch of a larger table
hipError_t launch_so_epoch(const SoEpoch& E, hipStream_t s);
// record sort keys for the printer's order: (index of the record's position in `order`, or last;
// position - pos_base; allele order), with idx = record index; *bad set when a field does not fit
// (rank_of: dense_n entries, overwritten; *kept <= max_keep: the order's length)
hipError_t launch_so_rank(const int32_t* order, const int32_t* kept, int max_keep, const OutRec* recs, int n,
                          int dense_lo, int dense_n, long long pos_base, int32_t* rank_of, unsigned long long* key,
                          int32_t* idx, unsigned* bad, hipStream_t s);

// the largest displacement of n keys laid out in slot order in a table of 2^cap_log2 slots, into
// *out (which must hold 0 beforehand); v, pm: n entries; temp == nullptr sets temp_bytes only
hipError_t launch_max_displacement(const int32_t* keys, int n, int cap_log2, int32_t* v, int32_t* pm, int* out,
                                   void* temp, size_t& temp_bytes, hipStream_t s);

hipError_t launch_score(const ScoreIn& S, hipStream_t s);
// k_score_prepick into S.pick_list / S.pick_count (dense_n entries, then the count) and S.status
// (dense_n entries); S needs the rows, the reference window, the region and the configuration only
hipError_t launch_score_prepick(const ScoreIn& S, hipStream_t s);
hipError_t launch_fisher_table(const int* tab, int n, double* out, const double* lgt, int lgt_n, hipStream_t s);
// the allocation-free variant's whole call (host tables in, host p-values out; rv_score.hip)
constexpr int FISHER_NOALLOC_MAX_TABLES = 1 << 16;
hipError_t fisher_tables_noalloc(const int* tab, int n, double* out, const char** err);

}  // namespace rv
