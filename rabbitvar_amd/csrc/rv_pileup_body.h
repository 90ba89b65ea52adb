// Per-item bodies of the pileup kernels (one read, one dense row, one anchor).  rv_pileup.hip says which
// take a lane and which a wavefront.
//
// Reference stages: src/recordPreprocessor.cpp:101-180 (filters), src/parseCigar.cpp:497-628
// (per-read setup, NM filter, modifyCigar, cleanupCigar, drop rules), :629-972 (walk),
// :1471-1490 (insertion-anchor subtraction).
#pragma once
#include "rv_walk.h"

namespace rv {

// Read batch in device memory, structure of arrays (the region iterator's records in order)
struct ReadsDev {
    const int32_t* pos0;
    const uint16_t* flag;
    const uint8_t* mapq;
    const uint8_t* has_nm;
    const int32_t* nm;
    const int32_t* mpos0;
    const int32_t* tid;
    const int32_t* mtid;
    const int64_t* seq_off;
    const int64_t* cig_off;
    const uint8_t* bases;
    const uint8_t* quals;
    const uint32_t* cigar;
    int64_t n;
    const uint8_t* drop;  // -Z: per read, 1 = dropped by the downsampling draw (nullptr without -Z)
};

// Everything the prep and walk kernels read besides the per-read records, kept in device memory
// so that uniform fields are read with scalar loads rather than copied to private memory.
struct WalkArgs {
    ReadsDev R;
    Window W;
    Config cfg;
    WalkSink S;
    uint8_t* dup;  // -t: per read, 1 = dropped as a duplicate (nullptr without -t)
};

// ---------------------------------------------------------------- duplicate removal (-t)
// recordPreprocessor.cpp:153-176.  The reference keeps a set of keys, clears it whenever a record's
// alignment start differs from the start of the key it inserted last, and drops a read whose key
// is already in the set.  Keys exist only for reads whose mate starts before base 10 (start, mate
// contig name, mate start) and for paired reads flagged unmapped (start, CIGAR text).  Over the
// records in iterator order, with the ones the flag/MAPQ/length filters dropped invisible to it,
// that is: a read is a duplicate when an earlier read with the same key lies in the same run of
// consecutive records that share its alignment start.
RV_HD bool rec_filtered(const ReadsDev& R, const Config& c, int64_t i) {
    const int lseq = (int)(R.seq_off[i + 1] - R.seq_off[i]);
    return (R.flag[i] & c.samfilter) != 0 || (R.drop && R.drop[i]) || (int)R.mapq[i] < c.mappingQuality ||
           lseq == 1;
}
// 0: no key; 1: keyed by the mate; 2: keyed by the CIGAR
RV_HD int dup_kind(const ReadsDev& R, int64_t i) {
    if (R.mpos0[i] + 1 < 10) return 1;
    const uint16_t f = R.flag[i];
    return ((f & 1) && (f & 4)) ? 2 : 0;
}
// getMateReferenceName (recordPreprocessor.cpp:80-90): "*" unpaired, "=" same contig, else the
// mate contig's name (one name per contig id)
RV_HD int mate_name(const ReadsDev& R, int64_t i) {
    if (!(R.flag[i] & 1)) return -3;
    if (R.tid[i] == R.mtid[i]) return -2;
    return R.mtid[i];
}
RV_HD bool same_dup_key(const ReadsDev& R, int64_t i, int64_t j, int kind) {
    if (kind == 1) return R.mpos0[i] == R.mpos0[j] && mate_name(R, i) == mate_name(R, j);
    const int64_t a = R.cig_off[i], b = R.cig_off[j];
    const int64_t na = R.cig_off[i + 1] - a;
    if (na != R.cig_off[j + 1] - b) return false;
    for (int64_t k = 0; k < na; k++) {
        const uint32_t x = R.cigar[a + k], y = R.cigar[b + k];
        if ((x >> 4) != (y >> 4)) return false;
        // bam_cigar_opchr prints every op code past 'B' (9) as '?'
        const uint32_t ox = (x & 15u) > 9u ? 10u : (x & 15u), oy = (y & 15u) > 9u ? 10u : (y & 15u);
        if (ox != oy) return false;
    }
    return true;
}
RV_HD bool is_duplicate(const ReadsDev& R, const Config& c, int64_t i) {
    if (rec_filtered(R, c, i)) return false;
    const int kind = dup_kind(R, i);
    if (kind == 0) return false;
    const int32_t s = R.pos0[i];
    for (int64_t j = i - 1; j >= 0; j--) {
        if (rec_filtered(R, c, j)) continue;
        if (R.pos0[j] != s) return false;
        if (dup_kind(R, j) == kind && same_dup_key(R, i, j, kind)) return true;
    }
    return false;
}

__device__ __forceinline__ uint32_t packed_seq_word(const uint8_t* seq, int lseq, int w) {
    uint32_t v = 0;
    for (int b = 0; b < 4; b++) {
        int byte = 4 * w + b;
        int i0 = 2 * byte, i1 = 2 * byte + 1;
        uint32_t hi = i0 < lseq ? (uint32_t)nt16_code((char)seq[i0]) : 0u;
        uint32_t lo = i1 < lseq ? (uint32_t)nt16_code((char)seq[i1]) : 0u;
        if (i0 < lseq) v |= ((hi << 4) | lo) << (8 * b);
    }
    return v;
}

// One read's filters and fields up to the CIGAR rewrite.  False when the read goes no further (p
// holds why).  span: the reach of the read around its alignment (the dense window's size).
__device__ inline bool prep_head(int64_t r, const ReadsDev& R, const Config& cfg, const uint8_t* dup, WalkCounters* ctr,
                                 PrepRec& p, int& span) {
    p.status = RD_PARSE;
    p.flags = 0;
    p.nm_eff = 0;
    p.rlen1 = 0;
    p.total_len = 0;
    p.reflen = 0;
    p.qual_before0 = 0;
    p.pad = 0;
    const uint16_t flag = R.flag[r];
    const int64_t so = R.seq_off[r];
    const int lseq = (int)(R.seq_off[r + 1] - so);
    p.flag = flag;
    p.mapq = R.mapq[r];
    p.same_contig = R.tid[r] == R.mtid[r] ? 1 : 0;
    p.mpos0 = R.mpos0[r];
    p.pos0 = R.pos0[r];
    p.seq_off = so;
    const int64_t co = R.cig_off[r];
    const int ncig = (int)(R.cig_off[r + 1] - co);
    p.lseq = lseq;
    p.position = p.pos0 + 1;
    p.ncig = 0;
    int reflen = 0, idlen = 0;
    for (int i = 0; i < ncig; i++) {
        const uint32_t w = R.cigar[co + i];
        const int o = cop(w);
        if (o == OP_M || o == OP_D || o == OP_N || o == OP_EQ || o == OP_X) reflen += clen(w);
        if (o == OP_I || o == OP_D) idlen += clen(w);
    }
    span = lseq + reflen + 8;
    p.reflen = reflen;
    if ((flag & cfg.samfilter) != 0 || (R.drop && R.drop[r]) || (int)p.mapq < cfg.mappingQuality || lseq == 1 ||
        (dup && dup[r])) {
        p.status = RD_FILTERED;
        return false;
    }
    if (ncig <= 0) {
        p.status = RD_NOWALK;
        return false;
    }
    int tnm = 0;
    if (R.has_nm[r]) {
        tnm = R.nm[r] - idlen;
        if (tnm > cfg.mismatch) {
            p.status = RD_NM;
            return false;
        }
    } else if (flag & 4) {
        p.status = RD_NM;
        return false;
    }
    p.nm_eff = tnm;
    // a CIGAR longer than the record slot is refused before anything is written: the region then
    // fails with a capacity error (the host checks the counter) instead of walking a cut record
    if (ncig > MAXC_IN) {
        p.status = RD_NOWALK;
        p.flags |= 2;
        atomicAdd(&ctr->capacity, 1ull);
        return false;
    }
    if (lseq > 0) {
        const int i0 = (lseq - 1) & ~1;
        const char* s = (const char*)(R.bases + so);
        p.qual_before0 = (nt16_code(s[i0]) << 4) | (i0 + 1 < lseq ? nt16_code(s[i0 + 1]) : 0);
    }
    return true;
}

// The drop rules after the rewrite (n_cigar words in rec).  tot: the read's length for
// maxReadLength, or 0.
__device__ inline void prep_tail(const uint32_t* rec, int n_cigar, uint16_t flag, const Config& cfg, PrepRec& p, int& tot) {
    p.ncig = n_cigar;
    tot = 0;
    if (n_cigar <= 0) {
        p.status = RD_NOWALK;
        return;
    }
    if (cop(rec[0]) == OP_S && clen(rec[0]) >= 10 && cop(rec[n_cigar - 1]) == OP_S && clen(rec[n_cigar - 1]) >= 10) {
        p.status = RD_NOWALK;
        return;
    }
    int rlen1 = 0, len = 0;
    for (int i = 0; i < n_cigar; i++) {
        int o = cop(rec[i]), l = clen(rec[i]);
        if (o == OP_M || o == OP_I) rlen1 += l;
        if (o == OP_M || o == OP_I || o == OP_S) len += l;
    }
    p.rlen1 = rlen1;
    p.total_len = len;
    if (cfg.minmatch != 0 && rlen1 < cfg.minmatch) {
        p.status = RD_NOWALK;
        return;
    }
    tot = len;
    if (flag & 2048) p.status = RD_NOWALK;
}

// A read of one M run (see single_m_run): its words to out[0, 3)
__device__ inline void prep_single_m(int64_t r, const ReadsDev& R, const Window& W, const Config& cfg, PrepRec& p,
                                     uint32_t* out, WalkCounters* ctr, int& tot) {
    tot = 0;
    int m = clen(R.cigar[R.cig_off[r]]), s5 = 0, s3 = 0;
    if (cfg.performLocalRealignment) {
        const int64_t so = R.seq_off[r];
        single_m_clips(RefView{W.ref, W.ref_lo, W.ref_hi}, ReadView{(const char*)(R.bases + so), R.quals + so, p.lseq},
                       p.position, m, s5, s3);
        if (s5 || s3) p.flags |= 1;
    }
    if ((s5 > 0) + (s3 > 0) > ((p.lseq + 1) / 2 + 3) / 4) {  // the words exceed the record: refused as in prep_head
        p.status = RD_NOWALK;
        p.flags = 2;
        atomicAdd(&ctr->capacity, 1ull);
        return;
    }
    p.position += s5;
    const uint32_t wm = ((uint32_t)m << 4) | OP_M, w5 = ((uint32_t)s5 << 4) | OP_S, w3 = ((uint32_t)s3 << 4) | OP_S;
    const uint32_t rec[3] = {s5 ? w5 : wm, s5 ? wm : w3, w3};
    out[0] = rec[0];
    out[1] = rec[1];
    out[2] = rec[2];
    // what prep_tail works out, for these lengths: neither clip reaches 10 bases
    p.ncig = 1 + (s5 > 0) + (s3 > 0);
    p.rlen1 = m;
    p.total_len = m + s5 + s3;
    if (cfg.minmatch != 0 && m < cfg.minmatch) {
        p.status = RD_NOWALK;
        return;
    }
    tot = p.total_len;
    if (R.flag[r] & 2048) p.status = RD_NOWALK;
}

// Any other read: its record in rec (MAXC words; the walk reads the first ncig + 1 of them: an indel
// looks at the operation after it, and the reference's record has the packed SEQ bytes there), with
// RULES (local realignment is on) rewritten by the CIGAR rules in *work.  rd: the read's bases and
// qualities.  False: refused (the caller counts it).  With RULES every lane of a wavefront runs this on
// the same LDS data on the device (see rx_search).
template <bool RULES>
__device__ inline bool prep_other(int64_t r, const ReadsDev& R, const Window& W, const Config& cfg, const ReadView& rd,
                                  PrepRec& p, uint32_t* rec, CigarWork* work, int& tot) {
    const int64_t co = R.cig_off[r];
    const int ncig = (int)(R.cig_off[r + 1] - co);
    const int nrec = ncig + ((p.lseq + 1) / 2 + 3) / 4 < MAXC ? ncig + ((p.lseq + 1) / 2 + 3) / 4 : MAXC;
    tot = 0;
    int idlen = 0;
    for (int i = 0; i < ncig; i++) {
        rec[i] = R.cigar[co + i];
        const int o = cop(rec[i]);
        if (o == OP_I || o == OP_D) idlen += clen(rec[i]);
    }
    // SEQ words: the rewrite adds at most two operations, and one word past the last is read
    auto seq_word = [&](int i) { return i < nrec ? packed_seq_word((const uint8_t*)rd.seq, p.lseq, i - ncig) : 0u; };
    const int filled = ncig + 4 < MAXC ? ncig + 4 : MAXC;
    for (int i = ncig; i < filled; i++) rec[i] = seq_word(i);
    int n_cigar = ncig;
    int position = p.position;
    if (RULES) {
        RefView rf{W.ref, W.ref_lo, W.ref_hi};
        int n_new = 0, fl = 0;
        if (modify_cigar_record(rf, rd, position, rec, nrec, ncig, idlen, n_new, fl, *work)) {
            n_cigar = n_new;
            p.flags |= 1;
        }
        p.flags |= fl;
        if (fl & 2) {  // rewrite text or words beyond capacity: refused as in prep_head
            p.status = RD_NOWALK;
            return false;
        }
    }
    if (n_cigar >= filled && n_cigar < MAXC) rec[n_cigar] = seq_word(n_cigar);
    // cleanupCigar: leading/trailing I become S until the first M/=/X
    {
        bool none = true;
        for (int i = 0; i < n_cigar && none; i++) {
            int o = cop(rec[i]);
            if (o == OP_I)
                rec[i] = (rec[i] & ~0xfu) | OP_S;
            else if (o == OP_M || o == OP_EQ || o == OP_X)
                none = false;
        }
        none = true;
        for (int i = n_cigar - 1; i >= 0 && none; i--) {
            int o = cop(rec[i]);
            if (o == OP_I)
                rec[i] = (rec[i] & ~0xfu) | OP_S;
            else if (o == OP_M || o == OP_EQ || o == OP_X)
                none = false;
        }
    }
    p.position = position;
    prep_tail(rec, n_cigar, R.flag[r], cfg, p, tot);
    return true;
}

// One read as a lane takes it: all of it, unless its CIGAR rules have to run (true: listed for a wavefront
// each, prep_other<true>)
__device__ __forceinline__ bool prep_lane(int64_t r, const ReadsDev& R, const Window& W, const Config& cfg,
                                          const uint8_t* dup, WalkCounters* ctr, uint32_t* cig, PrepRec& p, int& span,
                                          int& tot) {
    tot = 0;
    if (!prep_head(r, R, cfg, dup, ctr, p, span)) return false;
    const int64_t co = R.cig_off[r];
    uint32_t* const rec = cig + (size_t)r * MAXC;
    if (single_m_run(R.cigar + co, (int)(R.cig_off[r + 1] - co))) {
        uint32_t w[4] = {0u, 0u, 0u, 0u};
        prep_single_m(r, R, W, cfg, p, w, ctr, tot);
        // one store: the slot is 16-byte aligned, its fourth word is not read (at most 3 words and no indel)
        __builtin_memcpy(__builtin_assume_aligned(rec, 16), w, 16);
        return false;
    }
    if (cfg.performLocalRealignment) return true;
    const int64_t so = R.seq_off[r];
    (void)prep_other<false>(r, R, W, cfg, ReadView{(const char*)(R.bases + so), R.quals + so, p.lseq}, p, rec, nullptr, tot);
    return false;
}
static_assert(MAXC % 4 == 0, "16-byte slots");

__device__ inline void fill_row_one(DenseRow* rows, int i) {
    DenseRow z;
    for (int b = 0; b < 4; b++) {
        z.b[b].cnt = z.b[b].fwd = z.b[b].rev = z.b[b].hi = z.b[b].lo = 0;
        z.b[b].sum_tp = z.b[b].sum_q = z.b[b].sum_mq = z.b[b].sum_nm = 0;
        z.b[b].first_tpq = 0;
        z.b[b].flags = 0;
        z.b[b].min_ord = 0xffffffffu;
        z.b[b].last_tp = 0;
        z.b[b].pad[0] = z.b[b].pad[1] = z.b[b].pad[2] = 0;
    }
    z.cov = 0;
    z.rowflags = 0;
    z.first_touch = ~0ull;
    for (int k = 0; k < 4; k++) z.pad[k] = 0;
    rows[i] = z;
}

__device__ __forceinline__ int imax(int a, int b) { return a > b ? a : b; }

// Eight bytes of a read (n of them at s) from the 8k-th.  Nothing past the read is loaded: its last
// word is the last eight bytes, still to be shifted down by word_shift (where the word is used, so
// that nothing waits for it here).
__device__ __forceinline__ uint64_t read_word(const uint8_t* s, int n, int k) {
    uint64_t v = 0;
    if (n >= 8)
        __builtin_memcpy(&v, s + min(8 * k, n - 8), 8);
    else
        for (int j = 8 * k; j < n; j++) v |= (uint64_t)s[j] << (8 * (j - 8 * k));
    return v;
}
__device__ __forceinline__ int word_shift(int n, int k) { return n >= 8 ? 8 * imax(0, 8 * k - (n - 8)) : 0; }
// How many CIGAR words of a read the walk may look at
__device__ __forceinline__ int walk_cigar_words(const PrepRec& p) { return p.ncig + 1 < MAXC ? p.ncig + 1 : MAXC; }

// What a lane holds of a read before it goes to the wavefront's copy in LDS: one word of bases and
// of qualities and one of the CIGAR, so that the next read's loads are in flight while the current
// one is walked.
struct WalkFetch {
    uint64_t seq, qual;
    uint32_t cig;
};
__device__ __forceinline__ WalkFetch walk_fetch(const PrepRec& p, int64_t r, const uint8_t* bases, const uint8_t* quals,
                                               const uint32_t* cig, int k) {
    WalkFetch f{0, 0, 0};
    if (p.status != RD_PARSE) return f;
    if (p.lseq <= STAGE_LEN && 8 * k < p.lseq) {
        f.seq = read_word(bases + p.seq_off, p.lseq, k);
        f.qual = read_word(quals + p.seq_off, p.lseq, k);
    }
    if (k < walk_cigar_words(p)) f.cig = cig[(size_t)r * MAXC + k];
    return f;
}
__device__ __forceinline__ void walk_put(const PrepRec& p, const WalkFetch& f, WaveStage* st, int k) {
    if (p.lseq <= STAGE_LEN && 8 * k < p.lseq) {
        const int sh = word_shift(p.lseq, k);
        *reinterpret_cast<uint64_t*>(st->seq + 8 * k) = f.seq >> sh;
        *reinterpret_cast<uint64_t*>(st->qual + 8 * k) = f.qual >> sh;
    }
    if (k < walk_cigar_words(p)) st->cig[k] = f.cig;
}
static_assert(STAGE_LEN <= 8 * 64 && MAXC <= 64, "one word per lane");

// The smallest integer quality that is >= goodq (INT_MAX: none is)
__device__ __forceinline__ int goodq_threshold(double goodq) {
    if (!(goodq <= 1e6)) return 0x7fffffff;
    return goodq < -1e6 ? -1000000 : (int)ceil(goodq);
}
// a value that is the same on every lane, as a scalar
__device__ __forceinline__ int uniform(int v) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_readfirstlane(v);
#else
    return v;
#endif
}

// What walk_plain needs of the launch
struct PlainArgs {
    int goodq_i, goodq5_i;  // thresholds of goodq and goodq + 5
    int vext;
    int lo, hi;             // positions a read's bases may lie on: inside the tile, the dense window and,
                            // with the one after it, the reference window (hi exclusive)
    int Rs, Re;             // region
    int slo;                // position of walk_ref[0]
    int tile_lo;
    bool on;                // no option that drops part of a read is set
};
__device__ __forceinline__ PlainArgs plain_args(const Window& W, const Config& cfg, int tile_lo) {
    PlainArgs A;
    A.goodq_i = goodq_threshold(cfg.goodq);
    A.goodq5_i = goodq_threshold(cfg.goodq + 5);
    A.vext = cfg.vext;
    A.lo = imax(tile_lo, imax(W.dense_lo, W.ref_lo));
    A.hi = min(tile_lo + TILE_POS, min(W.dense_lo + W.dense_n, W.ref_hi));
    A.Rs = W.region_start;
    A.Re = W.region_end;
    A.slo = tile_lo - REF_BEFORE;
    A.tile_lo = tile_lo;
    A.on = cfg.trimBasesAfter == 0 && !cfg.uniqueModeAlignmentEnabled && !cfg.uniqueModeSecondInPairEnabled;
    return A;
}

// The plain bases of a staged read of one M run that lies inside the tile: what Walker::walk does for
// them, a base per lane, without the walker's state.  Returns how many bases it has done: all of them
// (the usual read), or those before the first one that Walker::plain_chunk would stop at too (done
// bases of the run, tseq key touches), or 0 for any other read.
// Nearly every read is of this kind, and the walk is bound by its instructions: through the walker,
// whose state spills scalar registers and whose conditions on the read are carried in lane masks, a
// 150-base read took 950 vector and 820 scalar instructions and 187 branches; k_walk on a 5 Mb contig at
// 60x 6.5 ms with every read through it, 4.55 with these here.
__device__ __forceinline__ int walk_plain(const PrepRec& p, int ord, const PlainArgs& A, int lane, int wave,
                                          unsigned& tseq) {
    const WaveStage* const st = &walk_stage[wave];
    const int ncig = uniform(p.ncig), lseq = uniform(p.lseq), position = uniform(p.position);
    const uint32_t word = (uint32_t)uniform((int)st->cig[0]);
    const int cel = clen(word);
    if (!A.on || ncig != 1 || cop(word) != OP_M || lseq > STAGE_LEN || cel > lseq || position < A.lo ||
        position + cel > A.hi)
        return 0;
    const int rlen1 = uniform(p.rlen1), nm = uniform(p.nm_eff);
    const unsigned add1 = (uniform(p.flag) & 0x10) ? TF_REV1 : 1u;
    const unsigned mapq = (unsigned)uniform(p.mapq) << 16;
    const char* const ref = walk_ref + (position - A.slo);
    int i = 0;
    while (i < cel) {
        const int span = min((int)warpSize, cel - i);
        const int j = i + lane;
        const bool act = lane < span;
        const int jc = act ? j : 0;
        const int pos = position + j;
        const unsigned ch = (unsigned char)st->seq[jc], rc = (unsigned char)ref[jc];
        const int qv = st->qual[jc];
        // the bits of A, C, G, T that differ, as 0..3, and back
        const unsigned x = (ch >> 1) & 3u;
        const int b = (int)(x ^ (x >> 1));
        const bool acgt = ((0x47544341u >> (8 * x)) & 0xffu) == ch, isN = ch == 'N';
        const bool in = pos >= A.Rs && pos <= A.Re;
        bool stop = act && !acgt && !isN;
        bool mnv = act && acgt && ch != rc && qv >= A.goodq_i && rc != 'N' && pos + 1 >= A.Rs && pos + 1 <= A.Re &&
                   j + 1 < cel;
        if (__ballot(mnv)) {
            if (mnv) {  // Walker::starts_mnv
                const char b1 = st->seq[j + 1], r1 = ref[j + 1];
                if (st->qual[j + 1] < A.goodq5_i || b1 == 'N' || r1 == 'N') {
                    mnv = false;
                } else if (r1 == b1) {
                    mnv = false;
                    for (int s = 1; s <= A.vext && j + 1 + s < cel; s++) {
                        if (ref[j + 1 + s] != st->seq[j + 1 + s]) {
                            mnv = st->qual[j + 1 + s] >= A.goodq5_i;
                            break;
                        }
                    }
                }
            }
            stop = stop || mnv;
        }
        const unsigned long long stops = __ballot(stop);
        const int f = stops ? __ffsll(stops) - 1 : span;
        const bool doit = lane < f && in && !isN;
        const unsigned long long md = __ballot(doit);
        if (doit) {
            const unsigned t = tseq + (unsigned)__popcll(md & ((1ull << lane) - 1ull));
            const int tp = min(j + 1, rlen1 - j);
            const int ti = pos - A.tile_lo;
            auto F = [&](int k) -> uint32_t* { return &walk_tile.f[k][b][ti]; };
            atomicMin(&walk_tile.first_touch[ti], ((unsigned long long)(unsigned)ord << 24) | (t & 0xffffffu));
            atomicAdd(F(TF_CNT), add1 + (qv >= A.goodq_i ? TF_HI1 : 0u));
            atomicAdd(F(TF_TP), (unsigned)tp);
            atomicAdd(F(TF_QMQ), (unsigned)qv | mapq);
            atomicAdd(F(TF_NM), (unsigned)nm);
            atomicMin(F(TF_MINORD), (unsigned)ord);
            const unsigned v = ((unsigned)tp << 8) | (unsigned)qv;
            atomicAnd(F(TF_AND), v);
            atomicOr(F(TF_OR), v);
            if (tp <= 0 || qv == 0) atomicOr(F(TF_CNT), TF_ZERO);
        }
        tseq += (unsigned)__popcll(md);
        i += f;
        if (f < span) break;
    }
    return i;
}

// A staged read (status RD_PARSE), walked by a whole wavefront (lane = this thread's lane, wave = its
// wavefront's index in the workgroup; see rv_walk.h).  Contributions to positions [tile_lo, tile_lo +
// TILE_POS) go to the workgroup's tile.  done, tseq: what walk_plain has done of it.
__device__ __forceinline__ void walk_staged(const PrepRec& p, int64_t r, const ReadsDev& R, const Window& W,
                                            const Config& cfg, const WalkSink& sink, int lane, int wave, int tile_lo,
                                            int done, unsigned tseq) {
    Walker w;
    w.lane = lane;
    w.leader = lane == 0;
    w.use_tile = true;
    w.tile_lo = tile_lo;
    w.ref.leader = lane == 0;
    w.cf = cfg;
    w.goodq_i = goodq_threshold(cfg.goodq);
    w.Rs = W.region_start;
    w.Re = W.region_end;
    w.chrLen = W.chr_len;
    w.ref.ref = W.ref;
    w.ref.lo = W.ref_lo;
    w.ref.hi = W.ref_hi;
    w.ref.ctr = sink.ctr;
    w.ref.slo = tile_lo - REF_BEFORE;
    w.ref.sn = REF_STAGE;
    w.S = sink;
    w.seq = (const char*)(R.bases + p.seq_off);
    w.qual = R.quals + p.seq_off;
    w.wave = wave;
    w.staged = p.lseq <= STAGE_LEN;
    w.lseq = p.lseq;
    w.qual_before0 = (uint8_t)p.qual_before0;
    w.rec_n = walk_cigar_words(p);
    w.n_cigar = p.ncig;
    w.ord = (int)r;
    w.evseq = 0;
    w.tseq = tseq;
    w.mapq = p.mapq;
    w.nm = p.nm_eff;
    w.dir = (p.flag & 0x10) != 0;
    w.position = p.position;
    w.bad = false;
    w.walk(p.rlen1, p.total_len, p.flag, p.same_contig != 0, p.mpos0 + 1, p.reflen, p.pos0, done);
}

// noPassingReads (reference src/VariationRealigner.cpp:1447-1498), one record: true when the record
// overlaps [start - 1, end) (0-based, as the region query does), carries no CIGAR deletion of
// exactly end - start bases, and its M + D span reaches more than two bases past both ends.
__device__ inline bool passes_one(const ReadsDev& R, int64_t i, int start, int end) {
    const int beg0 = R.pos0[i];
    if (beg0 >= end) return false;
    const uint32_t dq = ((uint32_t)(end - start) << 4) | (uint32_t)OP_D;
    int reflen_all = 0, al = 0;
    bool has = false;
    for (int64_t k = R.cig_off[i], k1 = R.cig_off[i + 1]; k < k1; k++) {
        const uint32_t w = R.cigar[k];
        const int o = (int)(w & 0xFu), l = (int)(w >> 4);
        if (o == OP_M || o == OP_D || o == OP_N || o == OP_EQ || o == OP_X) reflen_all += l;
        if (o == OP_M || o == OP_D) al += l;
        if (w == dq) has = true;
    }
    const int end0 = beg0 + (reflen_all > 0 ? reflen_all : 1);
    if (end0 <= start - 1 || has) return false;
    const int rs = beg0 + 1, re = rs + al;
    return re > end + 2 && rs < start - 2;
}

// Tile set-up and flush, strided over the workgroup's threads.
__device__ inline void tile_init(int tid, int nthreads, const Window& W, int tile_lo) {
    const int slo = tile_lo - REF_BEFORE;
    for (int k = tid; k < REF_STAGE; k += nthreads) {
        const int pos = slo + k;
        walk_ref[k] = (pos >= W.ref_lo && pos <= W.ref_hi) ? W.ref[pos - W.ref_lo] : '\0';
    }
    for (int k = tid; k < TF_N * 4 * TILE_POS; k += nthreads) {
        const int f = k / (4 * TILE_POS), r = k - f * 4 * TILE_POS;
        walk_tile.f[f][r / TILE_POS][r % TILE_POS] = (f == TF_MINORD || f == TF_AND) ? ~0u : 0u;
    }
    for (int k = tid; k < TILE_POS; k += nthreads) {
        walk_tile.cov[k] = 0;
        walk_tile.first_touch[k] = ~0ull;
    }
}

// Adds the tile into the dense rows.  What this costs is the number of cache lines its atomics go to
// (neighbouring positions' rows are 288 bytes apart, so each lane is a line of its own), so the nine
// sums of a base, next to each other in its row, are added by sixteen lanes of one instruction: a
// line per base, where a lane per base with 64-bit pairs of fields made five (k_walk on a 5 Mb contig at
// 60x 4.55 -> 3.28 ms with that, neighbouring tiles on one XCD and the compare-and-swap left out below).
// For the pstd/qstd state: the tile's AND/OR of its (position, quality) values covers pairs inside the
// workgroup, and comparing one tile value with the row's first value covers pairs across workgroups
// (not needed, and not waited for, where the tile's own values differ in both fields).  The tile
// value is the AND: exact in each field where the tile's values are all equal, and where they are
// not, that field's flag is already set, so a comparison against it can only set a flag that is set
// anyway.
#if defined(__HIP_DEVICE_COMPILE__)
constexpr int FLUSH_WAVE = 64, FLUSH_GROUP = 16;
#else
constexpr int FLUSH_WAVE = 1, FLUSH_GROUP = 1;
#endif
constexpr int FLUSH_SUMS = 9;
__device__ inline void tile_flush(int tile_lo, DenseRow* rows, int dense_lo, int dense_n, int tid, int nthreads) {
    const TileAcc* t = &walk_tile;
    const int lane = tid % FLUSH_WAVE, group = lane / FLUSH_GROUP;
    for (int k0 = tid - lane; k0 < 4 * TILE_POS; k0 += nthreads) {
        // one base, FLUSH_WAVE positions
        const int b = k0 / TILE_POS, i0 = k0 - b * TILE_POS, i = i0 + lane;
        const int ri = tile_lo + i - dense_lo;
        const bool in = ri >= 0 && ri < dense_n;
        if (b == 0 && in) {
            DenseRow& r = rows[ri];
            int cov = t->cov[i];
            for (int c = 0; c < 4; c++) {
                const unsigned cw = t->f[TF_CNT][c][i];
                cov += (int)((cw & 0x3ffu) + ((cw >> 10) & 0x3ffu));
            }
            if (cov) atomicAdd(&r.cov, cov);
            if (t->first_touch[i] != ~0ull) {
                atomicOr(&r.rowflags, 1u);
                atomicMin(&r.first_touch, t->first_touch[i]);
            }
        }
        const unsigned cw = in ? t->f[TF_CNT][b][i] : 0u;  // 0: no contribution to this base
        if (cw != 0) {
            DenseBase& d = rows[ri].b[b];
            atomicMin(&d.min_ord, t->f[TF_MINORD][b][i]);
            unsigned add = 1u | ((cw & TF_ZERO) ? 8u : 0u);
            const unsigned va = t->f[TF_AND][b][i], vo = t->f[TF_OR][b][i];
            if (va != ~0u || vo != 0u) {  // a pp/pq-updating contribution
                const unsigned diff = va ^ vo;
                if (diff >> 8) add |= 2u;
                if (diff & 0xffu) add |= 4u;
                if ((add & 6u) != 6u) {
                    const unsigned first = va + 1u;
                    const unsigned old = atomicCAS(&d.first_tpq, 0u, first);
                    if (old != 0u && old != first) {
                        const unsigned o = old - 1u;
                        if ((o >> 8) != (va >> 8)) add |= 2u;
                        if ((o & 0xffu) != (va & 0xffu)) add |= 4u;
                    }
                }
            }
            atomicOr(&d.flags, add);
        }
        for (unsigned long long m = __ballot(cw != 0); m;) {
            int e = -1;  // this group's position
            for (int g = 0; g < FLUSH_WAVE / FLUSH_GROUP; g++) {
                const int x = m ? __ffsll(m) - 1 : -1;
                e = g == group ? x : e;
                m &= m - 1;
            }
            if (e < 0) continue;
            DenseBase& d = rows[tile_lo + i0 + e - dense_lo].b[b];
            for (int f = lane % FLUSH_GROUP; f < FLUSH_SUMS; f += FLUSH_GROUP) {
                const unsigned w = t->f[f < 5 ? TF_CNT : f == 5 ? TF_TP : f == 8 ? TF_NM : TF_QMQ][b][i0 + e];
                const int fwd = (int)(w & 0x3ffu), rev = (int)((w >> 10) & 0x3ffu), hi = (int)((w >> 20) & 0x3ffu);
                const int v = f == 0   ? fwd + rev
                              : f == 1 ? fwd
                              : f == 2 ? rev
                              : f == 3 ? hi
                              : f == 4 ? fwd + rev - hi
                              : f == 6 ? (int)(w & 0xffffu)
                              : f == 7 ? (int)(w >> 16)
                                       : (int)w;
                if (v) atomicAdd(&d.cnt + f, v);
            }
        }
    }
}

// Insertion-anchor subtraction (parseCigar.cpp:1471-1490): the reference subtracts from the anchor
// base's entry only when that entry exists at that moment, i.e. when some read with an ordinal <=
// the inserting read created it (a creation by the same read always precedes its insertion).
__device__ inline void anchor_one(unsigned i, const Anchor* A, DenseRow* rows, int dense_lo, int dense_n, const Config& cfg) {
    Anchor a = A[i];
    int k = a.pos - dense_lo;
    if (k < 0 || k >= dense_n) return;
    DenseBase& d = rows[k].b[a.base];
    if (d.min_ord > (unsigned)a.ord) return;
    atomicSub(&d.cnt, 1);
    atomicSub(a.dir ? &d.rev : &d.fwd, 1);
    atomicSub(&d.sum_tp, a.tp);
    atomicSub(&d.sum_q, a.q);
    atomicSub(&d.sum_mq, a.mapq);
    atomicSub(&d.sum_nm, a.nmv);
    atomicSub((double)a.q >= cfg.goodq ? &d.hi : &d.lo, 1);
}


}  // namespace rv
