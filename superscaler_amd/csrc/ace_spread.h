// Scoring of SMALL batches: one plan (or single-stage query) per workgroup, its ops spread over the lanes.
//
// The large-batch kernel (ace_score_loop.h) gives a plan to a lane, which walks the op sequence: the right split when
// there are plans for every lane of the chip, but a lone wavefront then waits out one or two LDS latencies per op (about
// 220 ns: 71 us for one 315-op plan, behind the staging of 100 to 160 KB of tables that it reads a percent of).  Here
// the workgroup takes 256 ops at a time:
//   load   lane = op: its table entries, gathered from the rows in global memory (a plan touches 64 bytes per op; the
//          rows stay in L2), asked for before the chunk before is summed
//   write  ... into columns in LDS, one per accumulator, with the values that an accumulator does not take as 0.0
//          (x + 0.0 = x for the sums at hand, which start at +0.0)
//   seg    lane = op: an op that closes a run of recomputed pairs sums that run and writes it as a candidate of the peak
//   chain  lane = (stage, accumulator): the column's values of the stage, added in op order -- the reference's order of
//          additions, so the results are bit-identical to the other kernels'.  A dependent fp64 addition per op is what
//          bounds the kernel.
// and then lane = stage evaluates the stage tails (PlanState::finish), and lane 0 composes the plan.
//
// All phases are functions of (workgroup state, lane), so that the host build of the tests (ACE_HOST_EMU) can run the
// lanes of a phase one after the other.
#pragma once
#include "ace_score_loop.h"

constexpr int kSpreadLanes = 256;
constexpr int kSpreadPitch = kSpreadLanes + 2;      // doubles per column: columns start four banks apart
constexpr int kSpreadMaxOps = 16 * kSpreadLanes;    // a lane holds one 16-op group's stage starts
// LDS is what limits how many plans are on their way in a CU, and a kernel that mostly waits gains from every one of them: the
// table of pair kinds (up to 8 KB) is read where it is, and the per-group arrays are as long as the plan.  Six plans per CU
// instead of four; 3,001 plans, us per launch: 315 ops 35.6 -> 30.1, 523 ops 51.4 -> 45.0, 1,223 ops 89.7 -> 81.1.

// Columns: sums first, maxima after them.
template <bool BD, bool COLL> struct SpreadCols {
    static constexpr int FWD = 0, BWD = 1, RCS = 2, W = 3, A = 4, RSF = 5, RSB = 6, SAVED = 7, IDF = 8, IDB = 9;
    static constexpr int kSums = BD ? 10 : 8;
    static constexpr int RF = kSums, RB = kSums + 1, PEAK = kSums + 2, MC = kSums + 3;
    static constexpr int kMax = COLL ? 4 : 3;
    static constexpr int kCols = kSums + kMax;
};
// chains: sums of sixteen stages in the first three wavefronts, maxima in the fourth
static_assert(SpreadCols<true, true>::kSums * ACE_MAX_STAGES <= 192 && SpreadCols<true, true>::kMax * ACE_MAX_STAGES <= 64, "chain lanes");

struct SpreadShared {
    double *x;              // [kCols][kSpreadPitch] (+ 16)
    double *fin;            // [kCols][ACE_MAX_STAGES]
    double *stage_ms, *stage_mb;
    double *carry;          // [2] the running segment at the end of the chunk before, by chunk parity
    uint8_t *codes;         // [16 * G + 16]
    uint32_t *keep;         // [8] ops of the chunk that continue their segment, a bit each
    uint32_t *lut;          // [16] stage_lut of the plan's micro-batch size
    int32_t *bound;         // [18] first op of each stage, num_ops past the last
    uint16_t *starts;       // [G] stage starts of each 16-op group, a bit each
    uint16_t *count;        // [G] ... and their number
    uint16_t *prefix;       // [G] stage starts before the group
    int32_t *n_stages;
};

#ifdef ACE_HOST_EMU
inline
#else
__host__ __device__ __forceinline__
#endif
uint32_t ace_spread_layout(int cols, int G, unsigned char *lds, SpreadShared *s) {
    uint32_t o = 0;
    auto take = [&](uint32_t bytes) { const uint32_t at = o; o += (bytes + 15u) & ~15u; return lds + at; };
    s->x = reinterpret_cast<double *>(take((uint32_t)(cols * kSpreadPitch + 32) * 8u));
    s->fin = reinterpret_cast<double *>(take((uint32_t)(cols * ACE_MAX_STAGES) * 8u));
    s->stage_ms = reinterpret_cast<double *>(take(ACE_MAX_STAGES * 8u));
    s->stage_mb = reinterpret_cast<double *>(take(ACE_MAX_STAGES * 8u));
    s->carry = reinterpret_cast<double *>(take(16u));
    s->codes = take((uint32_t)G * 16u + 16u);
    s->keep = reinterpret_cast<uint32_t *>(take(32u));
    s->lut = reinterpret_cast<uint32_t *>(take(64u));
    s->bound = reinterpret_cast<int32_t *>(take(72u));
    s->starts = reinterpret_cast<uint16_t *>(take(2u * (uint32_t)G));
    s->count = reinterpret_cast<uint16_t *>(take(2u * (uint32_t)G));
    s->prefix = reinterpret_cast<uint16_t *>(take(2u * (uint32_t)G));
    s->n_stages = reinterpret_cast<int32_t *>(take(4u));
    return o;
}

// Per position, for this kernel: byte offset of the op's row in `rows`; kind of the (this op, next op) pair | bit 8: an
// ordinary op followed by a layer start | bit 9: an ordinary op.  Positions past the last op read zero.  (Host side.)
inline void ace_pos_spread(const ace_tables_t *t, ace_u2 *out, size_t entries) {
    const uint32_t row_bytes = (uint32_t)t->row_doubles * 8u;
    int w = 0;
    for (size_t i = 0; i < entries; ++i) {
        out[i] = ace_u2{0u, 0u};
        if (i >= (size_t)t->num_ops) continue;
        while (w + 1 < t->n_windows && (size_t)t->win_pos[w + 1] <= i) ++w;
        const uint32_t info = t->pos_info[i], slot_off = (info & 0xffu) * row_bytes;
        uint32_t type = 0;
        for (int r = t->win_row_begin[w]; r < t->win_row_begin[w + 1]; ++r)
            if (t->win_rows[2 * r + 1] == slot_off) type = t->win_rows[2 * r];
        out[i] = ace_u2{type * row_bytes, ((info >> 16) & 0xffu) | (((info >> 24) & 3u) << 8)};
    }
}

struct SpreadLane {
    // the op at hand
    ace_d2 h0, h1, h2;          // {fwd, bwd}, {weights, act}, {reserved fwd, bwd}
    double zf, zb, mf, mb;      // collectives of the pair with the op before: ms, MB occupied
    double idf, idb;
    uint32_t flags;             // SF_*
    // the chain at hand
    double acc;
};
enum { SF_LIVE = 1, SF_RC = 2, SF_LAST = 4, SF_PAIR = 8, SF_KEEP = 16, SF_PREV_ORDINARY = 32 };

// What every lane knows of the plan.
struct SpreadPlan {
    ace_u4 h;
    uint64_t glogs;
    uint32_t bidx, status;
    int lo, hi;                 // the ops of the plan (of the query)
};

template <bool RANGED> ACE_HD SpreadPlan spread_plan(const AceKernelArgs &a, long long plan) {
    SpreadPlan p;
    p.h = a.hdr[plan];
    p.glogs = (uint64_t)p.h.y | ((uint64_t)p.h.z << 32);
    p.bidx = (p.h.x >> 8) & 0xffu;
    p.status = 0;
    p.lo = 0;
    p.hi = a.g.N;
    if (p.bidx >= (uint32_t)a.g.n_mbs) { p.status = ACE_PLAN_MALFORMED; p.bidx = 0; }
    if (RANGED) {
        const ace_u2 r = a.range[plan];
        p.lo = (int)r.x;
        p.hi = (int)r.y;
        if (p.lo < 0 || p.hi > a.g.N || p.lo >= p.hi) { p.status = ACE_PLAN_MALFORMED; p.lo = 0; p.hi = 1; }
    }
    return p;
}

// ---- fetch: the plan's bytes and the small tables into LDS, stage starts per 16-op group -----------------------------------
template <bool RANGED> ACE_HD void spread_fetch(const AceKernelArgs &a, const SpreadShared &s, const SpreadPlan &p, long long plan, int cols, int tid) {
    const AceGeom &g = a.g;
    if (tid < g.G) {
        const ace_u4 cw = a.codes[(size_t)tid * g.P + plan];
        uint32_t w[4] = {cw.x, cw.y, cw.z, cw.w};
        uint32_t bits = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int left = g.N - (tid * 16 + 4 * j);              // code bytes of this word that belong to the plan
            w[j] &= left >= 4 ? 0xffffffffu : (left <= 0 ? 0u : ((1u << (8 * left)) - 1u));
            // bit 4 of each byte, gathered into four bits
            bits |= (((((w[j] >> 4) & 0x01010101u) * 0x01020408u) >> 24) & 15u) << (4 * j);
        }
        if (tid == 0) bits |= 1u;                                    // (a plan whose first op does not open a stage is malformed)
        reinterpret_cast<ace_u4 *>(s.codes)[tid] = ace_u4{w[0], w[1], w[2], w[3]};
        s.starts[tid] = (uint16_t)bits;
        s.count[tid] = (uint16_t)__builtin_popcount(bits);
    }
    if (tid == 0) {
        reinterpret_cast<ace_u4 *>(s.codes)[g.G] = ace_u4{0u, 0u, 0u, 0u};
        s.carry[0] = 0.0;
        s.carry[1] = 0.0;
    }
    if (tid < 16) s.lut[tid] = a.stage_lut[p.bidx * 16u + (uint32_t)tid];
    if (tid < 8) s.keep[tid] = 0u;
    if (tid < 18) s.bound[tid] = g.N;
    if (tid < cols) s.x[tid * kSpreadPitch + kSpreadLanes] = 0.0;
}

// ---- stages: where each stage begins -----------------------------------------------------------------------------------------
ACE_HD void spread_stages(const AceKernelArgs &a, const SpreadShared &s, int tid) {
    if (tid >= a.g.G) return;
    // stage starts before this group: the counts are added up two at a time (16 bits each; at most 4,096 in all)
    const uint32_t *pairs = reinterpret_cast<const uint32_t *>(s.count);
    uint32_t sum = 0;
    for (int j = 0; j < (tid >> 1); ++j) sum += pairs[j];
    uint32_t before = (sum & 0xffffu) + (sum >> 16);
    if (tid & 1) before += s.count[tid - 1];
    s.prefix[tid] = (uint16_t)before;
    uint32_t bits = s.starts[tid], k = before;
    while (bits && k < 18u) {
        s.bound[k++] = tid * 16 + __builtin_ctz(bits);
        bits &= bits - 1u;
    }
    if (tid == a.g.G - 1) *s.n_stages = (int32_t)(before + s.count[tid]);
}

// ---- load: the table entries of op c0 + tid ---------------------------------------------------------------------------------
template <bool BD, bool RANGED, bool COLL>
ACE_HD void spread_load(const AceKernelArgs &a, const SpreadShared &s, const SpreadPlan &p, int c0, int tid, SpreadLane &r) {
    const AceGeom &g = a.g;
    const int i = c0 + tid;
    r.flags = 0;
    if (i >= p.hi) return;
    const uint32_t byte = s.codes[i], nbyte = s.codes[i + 1], pbyte = i > 0 ? s.codes[i - 1] : 0u;
    const ace_u2 pos = a.pos_spread[i];
    const uint32_t prev = i > 0 ? a.pos_spread[i - 1].y : 0u;
    uint32_t stage = 0;
    bool first, last;
    if (RANGED) {
        first = i == p.lo;
        last = i + 1 == p.hi;
    } else {
        const int grp = i >> 4;
        stage = s.prefix[grp] + (uint32_t)__builtin_popcount(s.starts[grp] & ((2u << (i & 15)) - 1u)) - 1u;
        stage = stage < 15u ? stage : 15u;                  // (more than sixteen stages: refused in the end)
        first = i == 0 || ((byte >> 4) & 1u);
        last = i + 1 == p.hi || ((nbyte >> 4) & 1u);
    }
    const uint32_t pair = last ? 0u : pair_bit(byte, nbyte);
    const bool keep = pair && !((pos.y >> 8) & 1u);
    r.flags = SF_LIVE | (((byte >> 3) & 1u) ? SF_RC : 0) | (last ? SF_LAST : 0) | (pair ? SF_PAIR : 0) | (keep ? SF_KEEP : 0) |
              (((prev >> 9) & 1u) ? SF_PREV_ORDINARY : 0);
    const uint32_t glog = (uint32_t)(p.glogs >> (4u * stage)) & 15u;
    const uint32_t e = ace_mul24(s.lut[glog] & 15u, (uint32_t)g.C) + (byte & 7u);
    const unsigned char *row = reinterpret_cast<const unsigned char *>(a.rows) + pos.x;
    const ace_d2 *hot = reinterpret_cast<const ace_d2 *>(row + g.hot_off + e * ACE_HOT_STRIDE);
    r.h0 = hot[0];
    r.h1 = hot[1];
    r.h2 = hot[2];
    r.zf = r.zb = r.mf = r.mb = 0.0;
    if ((g.flags & ACE_F_RESHARDING) && !first) {           // (a stage's first op pays no resharding)
        const uint32_t gl = glog < (uint32_t)g.n_glog ? glog : 0u;
        const uint32_t id = a.pair_kinds[(prev & 0xffu) * g.rk_kind_stride + gl * 64u + (pbyte & 7u) * 8u + (byte & 7u)];
        const unsigned char *z = row + g.z_off + e * 8u;
        const uint32_t fo = (id & 15u) << g.z_shift, bo = (id >> 4) << g.z_shift;
        r.zf = *reinterpret_cast<const double *>(z + fo);
        r.zb = *reinterpret_cast<const double *>(z + bo);
        if (COLL) {
            r.mf = *reinterpret_cast<const double *>(z + fo + g.zm_delta);
            r.mb = *reinterpret_cast<const double *>(z + bo + g.zm_delta);
        }
    }
    if (BD) {
        // the "ideal" pass: tp = dp = 1, the diag of (micro_bs, 1 gpu)
        const uint32_t ie = ace_mul24(s.lut[0] & 15u, (uint32_t)g.C) + (byte & (uint32_t)(g.n_algo - 1));
        const ace_d2 v = *reinterpret_cast<const ace_d2 *>(row + g.hot_off + ie * ACE_HOT_STRIDE);
        r.idf = v.x;
        r.idb = v.y;
    }
}

// ---- write: into the columns --------------------------------------------------------------------------------------------------
template <bool BD, bool COLL> ACE_HD void spread_write(const SpreadShared &s, int tid, const SpreadLane &r) {
    typedef SpreadCols<BD, COLL> K;
    if (!(r.flags & SF_LIVE)) return;
    double *x = s.x + tid;
    auto put = [&](int col, double v) { x[col * kSpreadPitch] = v; };
    put(K::FWD, r.h0.x);
    put(K::BWD, r.h0.y);
    put(K::RCS, (r.flags & SF_RC) ? r.h0.x : 0.0);
    put(K::W, r.h1.x);
    put(K::A, r.h1.y);
    put(K::RSF, r.zf);
    put(K::RSB, r.zb);
    put(K::SAVED, (r.flags & SF_KEEP) ? r.h1.y : 0.0);
    if (BD) {
        put(K::IDF, r.idf);
        put(K::IDB, r.idb);
    }
    // the reserved maxima run over every op but the stage's last
    put(K::RF, (r.flags & SF_LAST) ? 0.0 : r.h2.x);
    put(K::RB, (r.flags & SF_LAST) ? 0.0 : r.h2.y);
    if (COLL) put(K::MC, ace_max(r.mf, r.mb));
    if (r.flags & SF_KEEP) {
#ifdef ACE_HOST_EMU
        s.keep[tid >> 5] |= 1u << (tid & 31);
#else
        atomicOr(&s.keep[tid >> 5], 1u << (tid & 31));
#endif
    }
}

// The running segment after op j of the chunk, which continues it: the activations of the ops that continue it, from the
// first of them on (`carry`: what the chunk before left, if they reach back to its end).
ACE_HD double spread_run(const SpreadShared &s, const double *act, double carry, int j) {
    int n = 0;
    for (int at = j; at >= 0;) {
        const uint32_t bit = (uint32_t)at & 31u;
        const uint32_t gaps = ~s.keep[at >> 5] << (31u - bit);          // the word's ops up to this one, this one on top
        const int ones = gaps ? __builtin_clz(gaps) : 32;
        const int mine = ones < (int)bit + 1 ? ones : (int)bit + 1;
        n += mine;
        if (mine <= (int)bit) break;
        at -= (int)bit + 1;
    }
    double run = n == j + 1 ? carry : 0.0;
    for (int k = j + 1 - n; k <= j; ++k) run += act[k];
    return run;
}

// ---- seg: candidates of the peak ----------------------------------------------------------------------------------------------
template <bool BD, bool COLL> ACE_HD void spread_seg(const SpreadShared &s, int tid, int parity, const SpreadLane &r) {
    typedef SpreadCols<BD, COLL> K;
    if (!(r.flags & SF_LIVE)) return;
    const double *act = s.x + K::A * kSpreadPitch;
    const double carry = s.carry[parity];
    double v = 0.0;
    if (!(r.flags & SF_KEEP)) {
        // the segment that the op before continued ends here: with this op's activations if the two form a pair, at all at
        // the stage's last op only behind an ordinary op
        if (!(r.flags & SF_LAST) || (r.flags & SF_PREV_ORDINARY)) {
            if (tid == 0) v = carry;
            else if ((s.keep[(tid - 1) >> 5] >> ((tid - 1) & 31)) & 1u) v = spread_run(s, act, carry, tid - 1);
        }
        if (r.flags & SF_PAIR) v += act[tid];
    }
    s.x[K::PEAK * kSpreadPitch + tid] = v;
    if (tid == kSpreadLanes - 1) s.carry[parity ^ 1] = (r.flags & SF_KEEP) ? spread_run(s, act, carry, tid) : 0.0;
}

// The values lo .. hi - 1 of a column (16-byte aligned; the one at kSpreadLanes is 0.0) added to `acc` in order (SUM), or their
// maximum with it.  A dependent addition takes a lone wavefront 3.5 ns, any other instruction about three, an LDS read 23: so
// values come in pairs, sixteen on their way while sixteen are added, in two sets of registers that take turns (nothing is
// moved), and the rest of a column as a block whose places past its end read the 0.0 (which changes neither a sum nor a maximum
// here: both start at +0.0).  Eight at a time, moved from set to set: 821 ops of one stage 25.4 us, now 18.7.
template <bool SUM> ACE_HD double spread_next(double acc, double v) { return SUM ? acc + v : ace_max(acc, v); }
template <bool SUM> ACE_HD double spread_column(const double *x, double acc, int lo, int hi, int zero) {
    int k = lo;
    if ((k & 1) && k < hi) acc = spread_next<SUM>(acc, x[k++]);
    if (k + 16 <= hi) {
        const ace_d2 *p = reinterpret_cast<const ace_d2 *>(x + k);
        ace_d2 v[8], u[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = p[j];
        for (;;) {
            // (reads past the column's end stay inside the columns and are not used)
#pragma unroll
            for (int j = 0; j < 8; ++j) u[j] = p[8 + j];
#pragma unroll
            for (int j = 0; j < 8; ++j) acc = spread_next<SUM>(spread_next<SUM>(acc, v[j].x), v[j].y);
            k += 16;
            if (k + 16 > hi) break;
            p += 16;
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = p[j];
#pragma unroll
            for (int j = 0; j < 8; ++j) acc = spread_next<SUM>(spread_next<SUM>(acc, u[j].x), u[j].y);
            k += 16;
            if (k + 16 > hi) break;
        }
    }
    while (k < hi) {
        double v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = x[k + j < hi ? k + j : zero];
#pragma unroll
        for (int j = 0; j < 8; ++j) acc = spread_next<SUM>(acc, v[j]);
        k += 8;
    }
    return acc;
}

// ---- chain: this chunk's share of the (stage, accumulator) of the lane ------------------------------------------------------
template <bool BD, bool RANGED, bool COLL>
ACE_HD void spread_chain(const SpreadShared &s, const SpreadPlan &p, int c0, int tid, SpreadLane &r) {
    typedef SpreadCols<BD, COLL> K;
    const bool sums = tid < 192;
    const int q = sums ? tid : tid - 192, per = sums ? K::kSums : K::kMax;
    const int stage = q / per, col = (sums ? 0 : K::kSums) + q % per;
    const int n = RANGED ? 1 : (*s.n_stages < ACE_MAX_STAGES ? *s.n_stages : ACE_MAX_STAGES);
    if (stage >= n) return;
    int lo = RANGED ? p.lo : s.bound[stage], hi = RANGED ? p.hi : s.bound[stage + 1];
    lo = (lo > c0 ? lo : c0) - c0;
    hi = (hi < c0 + kSpreadLanes ? hi : c0 + kSpreadLanes) - c0;
    const double *x = s.x + col * kSpreadPitch;
    const double acc = sums ? spread_column<true>(x, r.acc, lo, hi, kSpreadLanes) : spread_column<false>(x, r.acc, lo, hi, kSpreadLanes);
    r.acc = acc;
    s.fin[col * ACE_MAX_STAGES + stage] = acc;
}

// ---- tail: lane = stage ----------------------------------------------------------------------------------------------------------
template <bool BD, bool RANGED, bool COLL>
ACE_HD void spread_tail(const AceKernelArgs &a, const AceLds &lds, const SpreadShared &s, const SpreadPlan &p, double *rec, int tid) {
    typedef SpreadCols<BD, COLL> K;
    const int n = RANGED ? 1 : (*s.n_stages < ACE_MAX_STAGES ? *s.n_stages : ACE_MAX_STAGES);
    if (tid >= n) return;
    const AceGeom &g = a.g;
    const int lo = RANGED ? p.lo : s.bound[tid], hi = RANGED ? p.hi : s.bound[tid + 1];
    const uint32_t lut = s.lut[(uint32_t)(p.glogs >> (4 * tid)) & 15u];
    PlanState<BD, RANGED, false, COLL, true> st;
    st.S = (int)(p.h.x & 0xffu);
    st.bidx = p.bidx;
    st.cross = p.h.w;
    st.s = tid;
    st.sum_t = 0.0;
    st.max_t = 0.0;
    st.max_mem = 0.0;
    st.dc_v = ace_mul24(lut & 15u, (uint32_t)g.C);
    st.mrow = lut >> 16;
    st.ideal_start_v = ace_mul24(s.lut[0] & 15u, (uint32_t)g.C * ACE_START_STRIDE);
    st.start_lookups(g, lds, a.pos_spread[lo].x, s.codes[lo] & 7u);
    auto fin = [&](int col) { return s.fin[col * ACE_MAX_STAGES + tid]; };
    st.fwd = fin(K::FWD);
    st.bwd = fin(K::BWD);
    st.rcs = fin(K::RCS);
    st.W = fin(K::W);
    st.A = fin(K::A);
    st.rs_f = fin(K::RSF);
    st.rs_b = fin(K::RSB);
    st.saved = fin(K::SAVED);
    st.peak = fin(K::PEAK);
    st.rfm = fin(K::RF);
    st.rbm = fin(K::RB);
    st.mc = COLL ? fin(K::MC) : 0.0;
    st.run = 0.0;
    st.lastclose = false;
    if (BD) {
        st.id_fwd = fin(K::IDF);
        st.id_bwd = fin(K::IDB);
    }
    st.finish(g, lds, a.pos_spread[hi - 1].x, s.codes[hi - 1] & 7u, rec);
    s.stage_ms[tid] = st.sum_t;
    s.stage_mb[tid] = st.max_mem;
}

// ---- result: lane 0 --------------------------------------------------------------------------------------------------------------
template <bool BD, bool RANGED, bool COLL>
ACE_HD void spread_result(const AceKernelArgs &a, const SpreadShared &s, const SpreadPlan &p, long long out) {
    PlanState<BD, RANGED, false, COLL, true> st;
    st.S = (int)(p.h.x & 0xffu);
    st.s = RANGED ? 1 : *s.n_stages;
    st.status = p.status;
    if (!(s.codes[p.lo] & 0x10u)) st.status = ACE_PLAN_MALFORMED;       // the first op must open a stage
    const int n = st.s < ACE_MAX_STAGES ? st.s : ACE_MAX_STAGES;
    double sum = 0.0, mx = 0.0, mem = 0.0;
    for (int k = 0; k < n; ++k) {
        sum += s.stage_ms[k];
        mx = ace_max(mx, s.stage_ms[k]);
        mem = ace_max(mem, s.stage_mb[k]);
    }
    st.sum_t = sum;
    st.max_t = mx;
    st.max_mem = mem;
    double iter, peak;
    uint8_t feas, stat;
    st.result(a.g, a.nbm1[p.bidx], iter, peak, feas, stat);
    a.iter_ms[out] = iter;
    a.peak_mb[out] = peak;
    a.feasible[out] = feas;
    if (a.status) a.status[out] = stat;
}

// One workgroup.  SPREAD_PHASE runs a phase for every lane and waits for all of them.
#ifdef ACE_HOST_EMU
#define SPREAD_PHASE(...) for (int tid = 0; tid < kSpreadLanes; ++tid) { SpreadLane &r = lane[tid]; (void)r; __VA_ARGS__; }
#define SPREAD_NOWAIT SPREAD_PHASE
#else
#define SPREAD_PHASE(...) { __VA_ARGS__; } __syncthreads()
#define SPREAD_NOWAIT(...) { __VA_ARGS__; }
#endif
template <bool BD, bool RANGED, bool COLL>
ACE_HD void ace_spread_body(const AceKernelArgs &a, unsigned char *lds_raw, int tid_, long long plan) {
    typedef SpreadCols<BD, COLL> K;
    SpreadShared s;
    ace_spread_layout(K::kCols, a.g.G, lds_raw, &s);
#ifdef ACE_HOST_EMU
    static SpreadLane lane[kSpreadLanes];
    (void)tid_;
    AceLds lds = ace_make_lds(lds_raw, 0);
#else
    SpreadLane r;
    const int tid = tid_;
    AceLds lds = ace_make_lds(lds_raw, 0);
#endif
    lds.grows = reinterpret_cast<const unsigned char *>(a.rows);
    const SpreadPlan p = spread_plan<RANGED>(a, plan);
    const long long out = a.order ? (long long)a.order[plan] : plan;
    const bool active = out < a.g.P;
    const size_t rec_doubles = RANGED ? (size_t)ACE_STAGE_REC : (size_t)(ACE_MAX_STAGES * ACE_STAGE_REC);
    double *rec = (BD && a.stage_out && active) ? a.stage_out + (size_t)out * rec_doubles : nullptr;
    SPREAD_PHASE((spread_fetch<RANGED>(a, s, p, plan, K::kCols, tid)));
    if (!RANGED) { SPREAD_PHASE(spread_stages(a, s, tid)); }
    SPREAD_NOWAIT((r.acc = 0.0, spread_load<BD, RANGED, COLL>(a, s, p, p.lo, tid, r)));
    int parity = 0;
    for (int c0 = p.lo; c0 < p.hi; c0 += kSpreadLanes, parity ^= 1) {
        SPREAD_PHASE((spread_write<BD, COLL>(s, tid, r)));
        SPREAD_PHASE((spread_seg<BD, COLL>(s, tid, parity, r)));
        SPREAD_NOWAIT((spread_load<BD, RANGED, COLL>(a, s, p, c0 + kSpreadLanes, tid, r)));
        SPREAD_PHASE((spread_chain<BD, RANGED, COLL>(s, p, c0, tid, r)); if (tid < 8) s.keep[tid] = 0u);
    }
    SPREAD_PHASE((spread_tail<BD, RANGED, COLL>(a, lds, s, p, rec, tid)));
    SPREAD_NOWAIT(if (tid == 0 && active) (spread_result<BD, RANGED, COLL>(a, s, p, out)));
}
