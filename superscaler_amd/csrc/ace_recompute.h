// check_recompute (aceso_cost_model.py:822-872) for every stage of every plan of a batch, in one launch.
//
// One workgroup per plan, one wavefront per stage (its stages in turn).  The plan's code bytes and what the greedy loop
// reads again and again -- the activations of every op, twice (the raw table entry that sizes a group, and the one with the
// shared-buffer rule that the saved and peak activations are made of) -- stay in LDS from the first round to the last, so a
// round costs a few hundred instructions: pick the largest group (a reduction over its leaders, the groups' first ops),
// mark its ops, rebuild the masks, add the saved activations up in op order, take the maximum over the segments.  As
// launches per round (selection, gather of the plans still above the limit, single-stage queries, element-wise
// bookkeeping, a count of what is left read back by the host) the same loop took 6.5 ms for 16,384 plans of 523 ops; this launch
// takes 0.60 ms, bound by the latency of the additions in op order and of the exchanges between a round's phases.
//
// All sums run in op order, one rounding each: the recompute bits are those of the reference's loop.
// Lanes of a wavefront exchange values through LDS and through the reductions below; the host build of the tests
// (ACE_HOST_EMU) runs the 64 lanes of each phase one after the other.
#pragma once
#include "ace_spread.h"

constexpr int kRcWaves = 4;
constexpr int kRcMaxOps = 4000;          // LDS: 36 bytes per op

struct RcArgs {
    AceKernelArgs k;            // batch, tables, geometry
    const ace_u2 *pos;          // [N] previous | next op of the same type << 16 (0xffff / N: none); type | no-recompute flag << 16
    const double *act;          // raw activations [n_types][n_mbs][n_tp][n_algo]
    const uint8_t *status;      // [P] what scoring the batch said
    ace_u4 *codes_out;          // [G][P]
    int32_t *flags;             // [4], zeroed: RC_FLAG_*
    double limit, peak_backward;
};
// stage bits minus stage counts over the batch; a plan whose first op opens no stage; an op outside the profiled grid in
// a stage above the limit; a plan with a status
enum { RC_FLAG_COUNT = 0, RC_FLAG_FIRST = 1, RC_FLAG_GRID = 2, RC_FLAG_STATUS = 3 };

struct RcShared {
    double *act, *raw;          // [N]
    double *tmp;                // [N] weights, then the activations that a round saves
    double *sum;                // [N] at a group's first op: its size while it can still be chosen, else 0
    uint16_t *lead;             // [N] first op of the op's group
    uint32_t *keep;             // [kRcWaves][N / 32 + 2] ops that continue their segment, a bit each, from the stage's first op on
    uint8_t *codes;             // [16 * G + 16]
    uint32_t *lut;
    int32_t *bound;
    uint16_t *starts, *count, *prefix;
    int32_t *n_stages;
};

#ifdef ACE_HOST_EMU
inline
#else
__host__ __device__ __forceinline__
#endif
uint32_t ace_rc_layout(int N, int G, unsigned char *lds, RcShared *s) {
    uint32_t o = 0;
    auto take = [&](uint32_t bytes) { const uint32_t at = o; o += (bytes + 15u) & ~15u; return lds + at; };
    const uint32_t n8 = (uint32_t)N * 8u + 128u;        // (chains read up to sixteen values ahead)
    s->act = reinterpret_cast<double *>(take(n8));
    s->raw = reinterpret_cast<double *>(take(n8));
    s->tmp = reinterpret_cast<double *>(take(n8));
    s->sum = reinterpret_cast<double *>(take(n8));
    s->lead = reinterpret_cast<uint16_t *>(take((uint32_t)N * 2u));
    s->keep = reinterpret_cast<uint32_t *>(take((uint32_t)(kRcWaves * (N / 32 + 2)) * 4u));
    s->codes = take((uint32_t)G * 16u + 16u);
    s->lut = reinterpret_cast<uint32_t *>(take(64u));
    s->bound = reinterpret_cast<int32_t *>(take(72u));
    s->starts = reinterpret_cast<uint16_t *>(take(512u));
    s->count = reinterpret_cast<uint16_t *>(take(512u));
    s->prefix = reinterpret_cast<uint16_t *>(take(512u));
    s->n_stages = reinterpret_cast<int32_t *>(take(4u));
    return o;
}

// A wavefront's lanes: RC_EACH runs its body for every lane (`lane`, per-lane values `r`), then orders the wavefront's LDS
// accesses; the reductions leave their result in every lane's `r`.
struct RcLane { double a, b, c; int at, bad; };
#ifdef ACE_HOST_EMU
#define RC_EACH(...) for (int lane = 0; lane < 64; ++lane) { RcLane &r = rl[lane]; (void)r; __VA_ARGS__; }
#define RC_ATOMIC_OR(p, v) (*(p) |= (v))
#define RC_ATOMIC_ADD(p, v) (*(p) += (v))
inline void rc_max(RcLane *rl, double RcLane::*m) {
    double v = rl[0].*m;
    for (int j = 1; j < 64; ++j) v = ace_max(v, rl[j].*m);
    for (int j = 0; j < 64; ++j) rl[j].*m = v;
}
inline void rc_best(RcLane *rl) {       // largest a, the lowest `at` among equals
    RcLane v = rl[0];
    for (int j = 1; j < 64; ++j)
        if (rl[j].a > v.a || (rl[j].a == v.a && rl[j].at < v.at)) v = rl[j];
    for (int j = 0; j < 64; ++j) { rl[j].a = v.a; rl[j].at = v.at; }
}
inline int rc_any(RcLane *rl) {
    int v = 0;
    for (int j = 0; j < 64; ++j) v |= rl[j].bad;
    return v;
}
#define RC_R rl[0]
#define RC_MAX(m) rc_max(rl, &RcLane::m)
#define RC_BEST() rc_best(rl)
#define RC_ANY() rc_any(rl)
#define RC_FROM(m, from) (rl[from].m)
#else
#define RC_EACH(...) { __VA_ARGS__; } __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); __builtin_amdgcn_wave_barrier()
#define RC_ATOMIC_OR(p, v) atomicOr((p), (v))
#define RC_ATOMIC_ADD(p, v) atomicAdd((p), (v))
__device__ __forceinline__ void rc_max(double &v) {
    for (int off = 32; off > 0; off >>= 1) v = ace_max(v, __shfl_xor(v, off, 64));
}
__device__ __forceinline__ void rc_best(double &a, int &at) {
    for (int off = 32; off > 0; off >>= 1) {
        const double oa = __shfl_xor(a, off, 64);
        const int oi = __shfl_xor(at, off, 64);
        const bool other = oa > a || (oa == a && oi < at);
        a = other ? oa : a;
        at = other ? oi : at;
    }
}
#define RC_R r
#define RC_MAX(m) rc_max(r.m)
#define RC_BEST() rc_best(r.a, r.at)
#define RC_ANY() __any(r.bad)
#define RC_FROM(m, from) __shfl(r.m, from, 64)
#endif

ACE_HD double rc_chain(const double *x, int n) {
    double acc = 0.0;
    int k = 0;
    if (n >= 8) {
        double v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = x[j];
        for (; k + 8 <= n; k += 8) {
            double u[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) u[j] = x[k + 8 + j];
#pragma unroll
            for (int j = 0; j < 8; ++j) acc += v[j];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = u[j];
        }
    }
    for (; k < n; ++k) acc += x[k];
    return acc;
}

// The running segment after op j of the stage, which continues it.
ACE_HD double rc_run(const double *act, const uint32_t *keep, int j) {
    int n = 0;
    for (int at = j; at >= 0;) {
        const uint32_t bit = (uint32_t)at & 31u;
        const uint32_t gaps = ~keep[at >> 5] << (31u - bit);
        const int ones = gaps ? __builtin_clz(gaps) : 32;
        const int mine = ones < (int)bit + 1 ? ones : (int)bit + 1;
        n += mine;
        if (mine <= (int)bit) break;
        at -= (int)bit + 1;
    }
    double run = 0.0;
    for (int k = j + 1 - n; k <= j; ++k) run += act[k];
    return run;
}

// One stage: the ops [lo, hi) of the plan, `s` its index among `n_stages`.
template <bool COLL>
ACE_HD void rc_stage(const RcArgs &a, const RcShared &sh, const SpreadPlan &p, int s, int n_stages, int wave, int lane_) {
    const AceGeom &g = a.k.g;
    const int lo = sh.bound[s], hi = sh.bound[s + 1], len = hi - lo, nsb = n_stages - 1 - s;
    const uint32_t glog = (uint32_t)(p.glogs >> (4 * s)) & 15u, lut = sh.lut[glog], dc = ace_mul24(lut & 15u, (uint32_t)g.C);
    const unsigned char *rows = reinterpret_cast<const unsigned char *>(a.k.rows);
    uint32_t *keep = sh.keep + wave * (g.N / 32 + 2);
    double *act = sh.act + lo, *raw = sh.raw + lo, *tmp = sh.tmp + lo, *sum = sh.sum + lo;
    uint8_t *codes = sh.codes + lo;
    uint16_t *lead = sh.lead + lo;
#ifdef ACE_HOST_EMU
    static RcLane rl[64];
    (void)lane_;
#else
    RcLane r;
    const int lane = lane_;
#endif
    // ---- the stage's memory with no op recomputed (predict_stage_memory :514-539) ----
    RC_EACH(
        r.a = 0.0; r.b = 0.0; r.c = 0.0; r.bad = 0; r.at = 0;
        for (int j = lane; j < len; j += 64) {
            const uint32_t c = codes[j] & 7u;
            const unsigned char *row = rows + a.k.pos_spread[lo + j].x;
            const ace_d2 *hot = reinterpret_cast<const ace_d2 *>(row + g.hot_off + (dc + c) * ACE_HOT_STRIDE);
            const ace_d2 h1 = hot[1]; const ace_d2 h2 = hot[2];
            tmp[j] = h1.x;
            act[j] = h1.y;
            if (j + 1 < len) { r.a = ace_max(r.a, h2.x); r.b = ace_max(r.b, h2.y); }
            if (COLL && j > 0) {
                const uint32_t gl = glog < (uint32_t)g.n_glog ? glog : 0u;
                const uint32_t kind = a.k.pos_spread[lo + j - 1].y & 0xffu;
                const uint32_t id = a.k.pair_kinds[kind * g.rk_kind_stride + gl * 64u + (codes[j - 1] & 7u) * 8u + c];
                const unsigned char *z = row + g.z_off + (dc + c) * 8u + g.zm_delta;
                r.c = ace_max(r.c, *reinterpret_cast<const double *>(z + ((id & 15u) << g.z_shift)));
                r.c = ace_max(r.c, *reinterpret_cast<const double *>(z + ((id >> 4) << g.z_shift)));
            }
        });
    RC_MAX(a);
    RC_MAX(b);
    if (COLL) RC_MAX(c);
    const double rf = RC_R.a, rb = RC_R.b, mc = RC_R.c;
    RC_EACH(r.a = rc_chain((lane & 1) ? act : tmp, len));
    const double W = RC_FROM(a, 0), A = RC_FROM(a, 1);
    double reserved = 0.0;
    if (!(g.flags & ACE_F_NO_RESERVED)) {
        PlanState<false, false, false, COLL, true> st;
        st.rfm = rf; st.rbm = rb; st.W = W; st.mc = mc;
        reserved = st.reserved_term(g);
    }
    const double in = *reinterpret_cast<const double *>(rows + a.k.pos_spread[lo].x + g.start_off + (dc + (codes[0] & 7u)) * ACE_START_STRIDE);
    const double x = in + A;
    double mem = ((((W + W * g.main_params) + W) + W * g.optimizer) + x * (double)nsb) + x;
    mem = mem + reserved;
    mem = mem + a.peak_backward;
    if (!(mem - a.limit > 0.0)) return;

    // ---- op groups (:835-843) ----
    const uint32_t mrow = lut >> 16;
    RC_EACH(
        for (int j = lane; j < len; j += 64) {
            const uint32_t c = codes[j] & 7u; const uint32_t tp = c >> g.A_shift; const uint32_t al = c & (uint32_t)(g.n_algo - 1);
            uint32_t m = (mrow >> (4u * tp)) & 15u;
            if (tp >= (uint32_t)g.n_tp || m >= (uint32_t)g.n_mbs) { r.bad = 1; m = 0; }
            const uint32_t type = a.pos[lo + j].y & 0xffffu;
            raw[j] = a.act[((type * (uint32_t)g.n_mbs + m) * (uint32_t)g.n_tp + (tp < (uint32_t)g.n_tp ? tp : 0u)) * (uint32_t)g.n_algo + al] *
                     (double)(nsb + 1);
            sum[j] = 0.0;
        });
    RC_EACH(
        for (int j = lane; j < len; j += 64) {
            const ace_u2 e = a.pos[lo + j];
            const uint32_t before = e.x & 0xffffu;
            if (before != 0xffffu && (int)before >= lo) continue;
            double v = 0.0;
            for (int k = lo + j; k < hi; k = (int)(a.pos[k].x >> 16)) {
                v += raw[k - lo];
                lead[k - lo] = (uint16_t)j;
            }
            sum[j] = (e.y >> 16) ? 0.0 : v;
        });
    if (RC_ANY()) RC_EACH(if (lane == 0) RC_ATOMIC_OR(&a.flags[RC_FLAG_GRID], 1));

    // ---- the greedy loop (:849-868): every round takes one group out of `sum` ----
    double saved = 0.0, peak = 0.0;
    for (;;) {
        RC_EACH(
            r.a = 0.0; r.at = 0x7fffffff;
            for (int j = lane; j < len; j += 64) {
                const double v = sum[j];
                if (v > r.a) { r.a = v; r.at = j; }
            });
        RC_BEST();
        const double best = RC_R.a;
        const int T = RC_R.at;
        if (!(best > 0.0) || T + 1 >= len) return;           // nothing left (:804) or no op after the group's first (:805)
        const double exceed = mem - a.limit;
        int last = len;
        if (!(best < exceed)) {
            // the shortest prefix of the group that saves more than the excess (:812-816)
            double v = 0.0;
            for (int k = lo + T; k < hi && v <= exceed; k = (int)(a.pos[k].x >> 16)) {
                v += raw[k - lo];
                last = k - lo;
            }
        }
        const int also = lead[T + 1];
        RC_EACH(if (lane == 0) { sum[T] = 0.0; sum[also] = 0.0; }
                for (int j = lane; j < len; j += 64)
                    if ((int)lead[j] == T && j <= last) {
                        codes[j] |= 8u;
                        if (j + 1 < len) codes[j + 1] |= 8u;
                    }
                for (int j = lane; j <= (len >> 5); j += 64) keep[j] = 0u);
        // what the recompute bits save, and the largest segment (:394-449)
        RC_EACH(
            for (int j = lane; j < len; j += 64) {
                const bool pair = j + 1 < len && (codes[j] & codes[j + 1] & 8u);
                const bool cont = pair && !((a.k.pos_spread[lo + j].y >> 8) & 1u);
                tmp[j] = cont ? act[j] : 0.0;
                if (cont) RC_ATOMIC_OR(&keep[j >> 5], 1u << (j & 31));
            });
        RC_EACH(
            r.b = 0.0;
            for (int j = lane; j < len; j += 64) {
                if ((keep[j >> 5] >> (j & 31)) & 1u) continue;
                double v = 0.0;
                if (j > 0 && ((keep[(j - 1) >> 5] >> ((j - 1) & 31)) & 1u) &&
                    (j + 1 < len || ((a.k.pos_spread[lo + j - 1].y >> 9) & 1u)))
                    v = rc_run(act, keep, j - 1);
                if (j + 1 < len && (codes[j] & codes[j + 1] & 8u)) v += act[j];
                r.b = ace_max(r.b, v);
            }
            r.a = rc_chain(tmp, len));
        RC_MAX(b);
        const double new_saved = RC_R.a, new_peak = RC_R.b;
        mem = mem - (new_saved - saved) * (double)(nsb + 1);
        saved = new_saved;
        mem = mem + (new_peak - peak);
        peak = new_peak;
        if (!(mem - a.limit > 0.0)) return;
    }
}

ACE_HD void rc_fetch(const RcArgs &a, const RcShared &s, const SpreadPlan &p, long long plan, int tid) {
    const AceGeom &g = a.k.g;
    if (tid < g.G) {
        ace_u4 cw = a.k.codes[(size_t)tid * g.P + plan];
        cw = ace_u4{cw.x & 0xf7f7f7f7u, cw.y & 0xf7f7f7f7u, cw.z & 0xf7f7f7f7u, cw.w & 0xf7f7f7f7u};
        const uint32_t w[4] = {cw.x, cw.y, cw.z, cw.w};
        uint32_t bits = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) bits |= (((((w[j] >> 4) & 0x01010101u) * 0x01020408u) >> 24) & 15u) << (4 * j);
        const int left = g.N - tid * 16;
        if (left < 16) bits &= (1u << left) - 1u;            // (whatever stands behind the last op is no stage start)
        reinterpret_cast<ace_u4 *>(s.codes)[tid] = cw;
        s.starts[tid] = (uint16_t)bits;
        s.count[tid] = (uint16_t)__builtin_popcount(bits);
    } else
        s.count[tid] = 0;
    if (tid < 16) s.lut[tid] = a.k.stage_lut[p.bidx * 16u + (uint32_t)tid];
    if (tid < 18) s.bound[tid] = g.N;
}

#ifdef ACE_HOST_EMU
#define RC_PHASE(...) for (int tid = 0; tid < kSpreadLanes; ++tid) { __VA_ARGS__; }
#define RC_WAVES(...) for (int wave = 0; wave < kRcWaves; ++wave) { const int lane0 = 0; __VA_ARGS__; }
#else
#define RC_PHASE(...) { __VA_ARGS__; } __syncthreads()
#define RC_WAVES(...) { const int wave = tid >> 6, lane0 = tid & 63; __VA_ARGS__; } __syncthreads()
#endif
template <bool COLL> ACE_HD void ace_rc_body(const RcArgs &a, unsigned char *lds_raw, int tid_, long long plan) {
    const AceGeom &g = a.k.g;
    RcShared s;
    ace_rc_layout(g.N, g.G, lds_raw, &s);
    SpreadShared sp;            // (the part spread_stages works on)
    sp.starts = s.starts; sp.count = s.count; sp.prefix = s.prefix; sp.bound = s.bound; sp.n_stages = s.n_stages;
#ifdef ACE_HOST_EMU
    (void)tid_;
#else
    const int tid = tid_;
#endif
    const SpreadPlan p = spread_plan<false>(a.k, plan);
    RC_PHASE(rc_fetch(a, s, p, plan, tid));
    RC_PHASE(spread_stages(a.k, sp, tid));
    const int n = *s.n_stages, S = (int)(p.h.x & 0xffu);
    RC_PHASE(
        if (tid == 0) {
            if (n != S) RC_ATOMIC_ADD(&a.flags[RC_FLAG_COUNT], n - S);
            if (!(s.starts[0] & 1u)) RC_ATOMIC_OR(&a.flags[RC_FLAG_FIRST], 1);
            if (a.status[plan]) RC_ATOMIC_OR(&a.flags[RC_FLAG_STATUS], 1);
        });
    // (an inconsistent plan is reported and keeps its cleared bits)
    if (n == S && n <= ACE_MAX_STAGES && (s.starts[0] & 1u)) {
        RC_WAVES(for (int st = wave; st < n; st += kRcWaves) rc_stage<COLL>(a, s, p, st, n, wave, lane0));
    }
    RC_PHASE(if (tid < g.G) a.codes_out[(size_t)tid * g.P + plan] = reinterpret_cast<const ace_u4 *>(s.codes)[tid]);
}

// Per position: previous and next op of the same type, the type, whether its ops are never recomputed.  (Host side.)
inline void ace_rc_positions(const int32_t *type_of_pos, const uint8_t *norec, int N, int n_types, ace_u2 *out) {
    for (int i = 0; i < N; ++i) out[i] = ace_u2{0u, (uint32_t)type_of_pos[i] | ((uint32_t)(norec[type_of_pos[i]] != 0) << 16)};
    for (int t = 0; t < n_types; ++t) {
        uint32_t before = 0xffffu;
        for (int i = 0; i < N; ++i)
            if (type_of_pos[i] == t) {
                out[i].x = before | ((uint32_t)N << 16);
                if (before != 0xffffu) out[before].x = (out[before].x & 0xffffu) | ((uint32_t)i << 16);
                before = (uint32_t)i;
            }
    }
}
