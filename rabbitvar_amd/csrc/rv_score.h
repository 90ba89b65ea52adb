// Per-position scoring (device): restates ToVarsBuilder::process for one position
// (reference src/ToVarsBuilder.cpp:97-205 and the helpers it calls, :213-1116), the simple-mode
// output filter (src/modes/simpleMode.cpp:144-208 with include/Variant.h:99-248) and the two-sided
// Fisher exact test the printer adds with --fisher (src/modes/simpleMode.cpp:96-108; htslib's
// kt_fisher_exact, whose published algorithm is restated in fisher_two_sided below).
//
// A lane works out one position's records, one position per lane or per wavefront (see rv_score.hip).
// Positions whose alleles are all single-base A/C/G/T rows read the dense pileup table; positions the host touched (non-dense descriptors, insertions,
// realignment results) read a CSR record list.  Printed variants are appended to an output
// buffer with their strings in an arena; the host only formats numbers.
//
// This header holds the layouts shared with the host; the device code is in rv_score_body.h.
#pragma once
#include <hip/hip_runtime.h>

#include "rv_common.h"

namespace rv {

struct HVarD {
    int32_t cnt, fwd, rev, hicnt, locnt, extracnt;
    double pmean, qmean, mqmean, nm;
    int32_t pstd, qstd;
};

struct CxEntry {
    int32_t kind;  // 0 nonInsertionVariants, 1 insertionVariants
    uint32_t desc_off;
    int32_t desc_len;
    int32_t pad;
    HVarD v;
};

struct OutRec {
    int32_t position, order, start, end;
    int32_t tpc, poscov, rfc, rrc, fwd, rev, shift3, msint, hicnt, hicov, pstd, qstd, vartype;
    int32_t nfields;  // 5 for a pileup line without a reference variant
    double freq, pmean, qmean, mq, hlr, hifreq, extrafreq, msi, nm, fisher_p, fisher_ratio;
    uint64_t str_off;  // byte offset into the string arena (the arena can exceed 4 GiB)
    uint16_t len[7];  // refallele, varallele, genotype, bias, leftseq, rightseq, descriptor
    int32_t kind;     // OUT_VARIANT, or (somatic passes) OUT_REF / OUT_REF_ONLY / OUT_VARIANT_RAW
    int32_t start_rank;  // host: the position's rank in the printer's order
};
static_assert(sizeof(OutRec) == 192, "OutRec layout (records are copied to the host as they are)");

// OutRec kinds.  Simple mode emits printed variants only.  The somatic pass emits a position's
// Vars: every non-reference variant in CMP_VARI order plus its reference variant (OUT_REF, as
// createVariant left it), or the reference-only form of a position without variants (OUT_REF_ONLY,
// ToVarsBuilder.cpp:1074-1097), and the variants a failed reference lookup left as createVariant made
// them (OUT_VARIANT_RAW).
enum : int { OUT_VARIANT = 0, OUT_REF = 1, OUT_REF_ONLY = 2, OUT_VARIANT_RAW = 3 };
// ScoreIn::somatic.  A tumor/normal pair is scanned first (each position's state, nothing emitted),
// then the positions that can print a line are emitted.
enum : int { SCORE_SIMPLE = 0, SCORE_SOMATIC_SCAN = 1, SCORE_SOMATIC_EMIT = 2 };
// status of a scanned position: kept with variants (some of which pass the counts of isGoodVar), or
// kept without (reference only)
enum : int { SOM_VARS = 1, SOM_VARS_CAND = 5, SOM_REF = 3 };
// ScoreIn::want: emit a position's variants, or its reference-only record
enum : int { WANT_VARS = 1, WANT_REF = 2 };

enum : int { VT_SNV = 0, VT_INS = 1, VT_DEL = 2, VT_COMPLEX = 3, VT_EMPTY = 4, VT_SV = 5 };

struct ScoreIn {
    const DenseRow* rows;
    int dense_lo, dense_n;
    const int32_t* cx_pos;
    int n_cx;
    const int32_t* cx_off;
    const CxEntry* cx;
    const char* cx_arena;
    const int32_t* cx_cov;
    const uint8_t* cx_key;
    const char* ref;
    int ref_lo, ref_hi, chr_len;
    int region_start, region_end;
    Config cfg;
    OutRec* out;
    unsigned* n_out;
    unsigned max_out;
    char* arena;
    unsigned long long* arena_used;
    unsigned long long arena_cap;
    uint8_t* status;  // per dense row, then per record-list position: 1 = alignedVariants entry kept,
                      // 2 = added and erased again (nothing above -f), 0 = not added; somatic: SOM_*
    int somatic;                // SCORE_*
    const uint8_t* want;        // SCORE_SOMATIC_EMIT: per status slot, WANT_* or 0
    unsigned long long* counters;  // [0] capacity overflows, [1] insertion side effects on p+1,
                                   // [2] sorts above 16 elements, [3] qstd ambiguous rows
    const double* lgamma_tab;      // host-built kf_lgamma of the integers (fisher_lgamma_table)
    int lgamma_n;
    // dense positions to score, picked by k_score_pick (dense_n entries, then the count)
    int32_t* pick_list;
    unsigned* pick_count;
    // simple mode without -p: the dense positions that can print and every dense position's status,
    // worked out by k_score_prepick while the realigner runs (from the pileup's rows and the
    // reference alone); nullptr: k_score_pick and k_score_dense
    const int32_t* pre_list;
    const unsigned* pre_count;
    const uint8_t* pre_status;
};

}  // namespace rv
