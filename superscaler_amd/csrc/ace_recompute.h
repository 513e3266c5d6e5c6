// check_recompute (aceso_cost_model.py:822-872) for every stage of every plan of a batch, in one launch.
//
// One workgroup per plan: the memory of all stages first (a lane per op, then per stage), then a wavefront per stage above the limit, in
// turn.  What the greedy loop reads again and again -- the plan's code
// bytes, the activations, every op's type and the next op of that type -- stays in LDS from the first round to the last, so a round costs a
// few hundred instructions: pick the largest group (a reduction over the op types), mark its ops, put the activations that are
// saved one behind the other and add them up in op order, take the maximum over the segments.  As launches per round (selection,
// gather of the plans still above the limit, single-stage queries, element-wise bookkeeping, a count of what is left read back by the
// host) the same loop took 6.5 ms for 16,384 plans of 523 ops.
// Bound by latency -- a wavefront waits for LDS, for the trip to memory, for the addition before -- and by how many plans a CU has on
// their way.  16,384 plans of 523 ops (5.8 stages each, a quarter of them above the limit, three rounds), us:
//   596  a wavefront per stage, four of them, 36 bytes of LDS per op: 7 plans per CU, of whose 28 wavefronts five had something to do
//   301  two of them, 24 bytes (raw activations where the weights were; a size per type instead of one per op), 11 plans per CU; flags and
//        links in LDS; the saved activations one behind the other (no additions of 0.0); reductions without LDS
//   265  a segment per lane instead of an op per lane; 128 ops' entries asked for at once
//   244  all ops' entries at once, the sums of all stages side by side; wavefronts only for the stages above the limit
//
// All sums run in op order, one rounding each: the recompute bits are those of the reference's loop.
// Lanes of a wavefront exchange values through LDS and through the reductions below; the host build of the tests
// (ACE_HOST_EMU) runs the 64 lanes of each phase one after the other.
#pragma once
#include "ace_spread.h"

constexpr int kRcMaxOps = 4000;
constexpr int kRcLanes = 128;            // the most a workgroup has

struct RcArgs {
    AceKernelArgs k;            // batch, tables, geometry
    const ace_u2 *pos;          // [N] previous | next op of the same type << 16 (0xffff / N: none); type | no-recompute flag << 16 | group << 17
    int32_t groups = 0;         // types in use, numbered as groups (0: room for as many as there are ops)
    int32_t waves = 1;          // wavefronts of a workgroup
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
    double *act;                // [N] and a 0.0
    double *tmp;                // [N] weights, then raw activations, then the activations that a round saves, one behind the other; and a 0.0
    double *sum;                // [waves][groups] a group's size while it can still be chosen, else 0
    uint16_t *first;            // [waves][groups] its first op
    uint16_t *type, *next;      // [N] group | RC_LAST | RC_ORDINARY; next op of that type (N: none)
    uint8_t *codes;             // [16 * G + 16]
    uint32_t *lut;
    int32_t *bound;
    uint16_t *starts, *count, *prefix;
    int32_t *n_stages;
    // per stage: largest reserved sizes (forward, backward, of a collective) as their bits; input, weights, activations; its memory
    unsigned long long *reserved;
    double *in, *sums, *mem;
    int32_t groups;             // how many `sum` and `first` have room for
};
// an ordinary op with a layer start behind it; an ordinary op (group numbers are below kRcMaxOps)
enum { RC_GROUP = 0xfff, RC_LAST = 0x4000, RC_ORDINARY = 0x8000 };

#ifdef ACE_HOST_EMU
inline
#else
__host__ __device__ __forceinline__
#endif
uint32_t ace_rc_layout(int N, int G, int groups, int waves, unsigned char *lds, RcShared *s) {
    uint32_t o = 0;
    s->groups = groups ? groups : N;
    auto take = [&](uint32_t bytes) { const uint32_t at = o; o += (bytes + 15u) & ~15u; return lds + at; };
    const uint32_t n8 = (uint32_t)N * 8u + 128u;        // (chains read up to sixteen values ahead)
    s->act = reinterpret_cast<double *>(take(n8));
    s->tmp = reinterpret_cast<double *>(take(n8));
    s->sum = reinterpret_cast<double *>(take((uint32_t)(waves * s->groups) * 8u));
    s->first = reinterpret_cast<uint16_t *>(take((uint32_t)(waves * s->groups) * 2u));
    s->type = reinterpret_cast<uint16_t *>(take((uint32_t)N * 2u));
    s->next = reinterpret_cast<uint16_t *>(take((uint32_t)N * 2u));
    s->codes = take((uint32_t)G * 16u + 16u);
    s->lut = reinterpret_cast<uint32_t *>(take(64u));
    s->bound = reinterpret_cast<int32_t *>(take(72u));
    s->starts = reinterpret_cast<uint16_t *>(take((uint32_t)G * 2u));
    s->count = reinterpret_cast<uint16_t *>(take((uint32_t)G * 2u));
    s->prefix = reinterpret_cast<uint16_t *>(take((uint32_t)G * 2u));
    s->n_stages = reinterpret_cast<int32_t *>(take(4u));
    s->reserved = reinterpret_cast<unsigned long long *>(take(3u * ACE_MAX_STAGES * 8u));
    s->in = reinterpret_cast<double *>(take(ACE_MAX_STAGES * 8u));
    s->sums = reinterpret_cast<double *>(take(2u * ACE_MAX_STAGES * 8u));
    s->mem = reinterpret_cast<double *>(take(ACE_MAX_STAGES * 8u));
    return o;
}

// ... by the arguments of a launch: the kernel and whoever sizes its LDS read the same two members, which have a value if nobody set them.
#ifdef ACE_HOST_EMU
inline
#else
__host__ __device__ __forceinline__
#endif
uint32_t ace_rc_layout(const RcArgs &a, unsigned char *lds, RcShared *s) {
    return ace_rc_layout(a.k.g.N, a.k.g.G, a.groups, a.waves, lds, s);
}
// ... of one wavefront with room for a group per op: what arguments that say neither ask for.
inline uint32_t ace_rc_layout(int N, int G, unsigned char *lds, RcShared *s) { return ace_rc_layout(N, G, 0, 1, lds, s); }

// A wavefront's lanes: RC_EACH runs its body for every lane (`lane`, per-lane values `r`), then orders the wavefront's LDS
// accesses; the reductions leave their result in every lane's `r`.
struct RcLane { double a, b; int at, bad; };
#ifdef ACE_HOST_EMU
#define RC_EACH(...) for (int lane = 0; lane < 64; ++lane) { RcLane &r = rl[lane]; (void)r; __VA_ARGS__; }
#define RC_SAVED(to, ...) for (int j = 1; j < 64; ++j) rl[j].b = 0.0; { const int lane = 0; RcLane &r = rl[0]; to = __VA_ARGS__; }
#define RC_ATOMIC_OR(p, v) (*(p) |= (v))
#define RC_ATOMIC_ADD(p, v) (*(p) += (v))
#define RC_ATOMIC_MAX(p, v) (*(p) = *(p) > (v) ? *(p) : (v))
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
#define RC_SAVED(to, ...) RC_EACH(to = __VA_ARGS__)
#define RC_ATOMIC_OR(p, v) atomicOr((p), (v))
#define RC_ATOMIC_ADD(p, v) atomicAdd((p), (v))
#define RC_ATOMIC_MAX(p, v) atomicMax((p), (v))
// (values are not negative: lanes that nothing comes from give 0.0)
template <int CTRL> __device__ __forceinline__ double rc_dpp(double v) {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, 0xf, 0xf, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
__device__ __forceinline__ double rc_from(double v, int lane) {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, lane), hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), lane);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
// (what an instruction writes, another one reads across lanes two issue slots later at the earliest)
__device__ __forceinline__ double rc_larger(double a, double b) {
    double r;
    asm("v_max_f64 %0, %1, %2\n s_nop 1" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ void rc_max(double &v) {
    v = rc_larger(v, v);
    v = rc_larger(v, rc_dpp<0x111>(v));             // one, two, four and eight lanes before in the row of sixteen
    v = rc_larger(v, rc_dpp<0x112>(v));
    v = rc_larger(v, rc_dpp<0x114>(v));
    v = rc_larger(v, rc_dpp<0x118>(v));
    v = rc_larger(v, rc_dpp<0x142>(v));             // the last lane of the row before; of the first half
    v = rc_larger(v, rc_dpp<0x143>(v));
    v = rc_from(v, 63);
}
__device__ __forceinline__ void rc_best(double &a, int &at) {
    const double mine = a;
    rc_max(a);
    int best = 0x7fffffff;
    for (unsigned long long m = a > 0.0 ? __ballot(mine == a) : 0ull; m; m &= m - 1ull) {
        const int x = __builtin_amdgcn_readlane(at, __ffsll((long long)m) - 1);
        best = x < best ? x : best;
    }
    at = best;
}
#define RC_R r
#define RC_MAX(m) rc_max(r.m)
#define RC_BEST() rc_best(r.a, r.at)
#define RC_ANY() __any(r.bad)
#define RC_FROM(m, from) rc_from(r.m, from)
#endif

// The activations of the ops that continue their segment, one behind the other in `tmp` -- a segment's lie together --, and from the
// stage's last entry down what ends a segment (an op that does not continue the one that the op before did): RcEnd.  The two don't
// meet: every segment has an op that is not stored.  Returns how many activations and ends there are; `single` becomes the largest
// activation of a pair that is a segment by itself.
struct RcSaved { int n, ends; };
enum { RC_END_COUNTS = 1 << 28, RC_END_PAIR = 1 << 29 };    // behind the place of the segment's end (bits 0-15) and the op (16-27)
ACE_HD void rc_op(const uint8_t *codes, const uint16_t *type, int len, int j, bool &pair, bool &cont) {
    pair = j + 1 < len && (codes[j] & codes[j + 1] & 8u);
    cont = pair && !(type[j] & RC_LAST);
}
ACE_HD void rc_end(const uint16_t *type, double *tmp, int len, int j, bool pair, int n, int ends) {
    const bool counts = j + 1 < len || (type[j - 1] & RC_ORDINARY);
    *reinterpret_cast<uint32_t *>(tmp + (len - 1 - ends)) = (uint32_t)n | ((uint32_t)j << 16) | (counts ? RC_END_COUNTS : 0) | (pair ? RC_END_PAIR : 0);
}
ACE_HD RcSaved rc_saved(const uint8_t *codes, const uint16_t *type, const double *act, double *tmp, int len, int lane, double &single) {
    RcSaved s{0, 0};
    single = 0.0;
#ifdef ACE_HOST_EMU
    (void)lane;
    bool before = false;
    for (int j = 0; j < len; ++j) {
        bool pair, cont;
        rc_op(codes, type, len, j, pair, cont);
        if (before && !cont) rc_end(type, tmp, len, j, pair, s.n, s.ends++);
        else if (pair && !cont) single = ace_max(single, act[j]);
        if (cont) tmp[s.n++] = act[j];
        before = cont;
    }
#else
    unsigned long long carry = 0;
    for (int base = 0; base < len; base += 64) {
        const int j = base + lane;
        bool pair, cont;
        rc_op(codes, type, len, j, pair, cont);
        const unsigned long long m = __ballot(cont), ended = (m << 1 | carry) & ~m & __ballot(j < len);
        const int n = s.n + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        if (cont) tmp[n] = act[j];
        else if (ended >> lane & 1ull) rc_end(type, tmp, len, j, pair, n, s.ends + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(ended >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)ended, 0u)));
        else if (pair) single = ace_max(single, act[j]);
        s.n += __popcll(m);
        s.ends += __popcll(ended);
        carry = m >> 63;
    }
#endif
    return s;
}

// ---- the stages' memory with no op recomputed (predict_stage_memory :514-539), all of them at once ----
// The values of every op of the plan: several per lane in flight, the trips to memory are what this costs.
template <bool COLL> ACE_HD void rc_load(const RcArgs &a, const RcShared &s, const SpreadPlan &p, int n, int tid) {
    const AceGeom &g = a.k.g;
    const unsigned char *rows = reinterpret_cast<const unsigned char *>(a.k.rows);
    const int lanes = 64 * a.waves;
    auto stage_of = [&](int i) { return (int)s.prefix[i >> 4] + __builtin_popcount(s.starts[i >> 4] & ((2u << (i & 15)) - 1u)) - 1; };
    auto entry = [&](int i, int st) { return ace_mul24(s.lut[(uint32_t)(p.glogs >> (4 * st)) & 15u] & 15u, (uint32_t)g.C) + (s.codes[i] & 7u); };
    auto larger = [&](int what, int st, double x) {             // (a running maximum from 0.0)
        unsigned long long b;
        __builtin_memcpy(&b, &x, 8);
        if (x > 0.0) RC_ATOMIC_MAX(&s.reserved[what * ACE_MAX_STAGES + st], b);
    };
    constexpr int kAtOnce = 5;
    for (int i0 = tid; i0 < g.N; i0 += lanes * kAtOnce) {
        ace_d2 h1[kAtOnce], h2[kAtOnce];
#pragma unroll
        for (int q = 0; q < kAtOnce; ++q) {
            const int i = i0 + q * lanes < g.N ? i0 + q * lanes : i0;
            const ace_d2 *hot = reinterpret_cast<const ace_d2 *>(rows + a.k.pos_spread[i].x + g.hot_off + entry(i, stage_of(i)) * ACE_HOT_STRIDE);
            h1[q] = hot[1];
            h2[q] = hot[2];
        }
#pragma unroll
        for (int q = 0; q < kAtOnce; ++q) {
            const int i = i0 + q * lanes, st = i < g.N ? stage_of(i) : 0;
            if (i >= g.N) break;
            s.tmp[i] = h1[q].x;
            s.act[i] = h1[q].y;
            if (i + 1 < s.bound[st + 1]) {
                larger(0, st, h2[q].x);
                larger(1, st, h2[q].y);
            }
        }
    }
    if (COLL)
        for (int i = tid; i < g.N; i += lanes) {
            const int st = stage_of(i);
            if (i == s.bound[st]) continue;
            const uint32_t glog = (uint32_t)(p.glogs >> (4 * st)) & 15u, gl = glog < (uint32_t)g.n_glog ? glog : 0u;
            const uint32_t id = a.k.pair_kinds[(a.k.pos_spread[i - 1].y & 0xffu) * g.rk_kind_stride + gl * 64u + (s.codes[i - 1] & 7u) * 8u + (s.codes[i] & 7u)];
            const unsigned char *z = rows + a.k.pos_spread[i].x + g.z_off + entry(i, st) * 8u + g.zm_delta;
            larger(2, st, *reinterpret_cast<const double *>(z + ((id & 15u) << g.z_shift)));
            larger(2, st, *reinterpret_cast<const double *>(z + ((id >> 4) << g.z_shift)));
        }
    if (tid < n) {
        const int lo = s.bound[tid];
        s.in[tid] = *reinterpret_cast<const double *>(rows + a.k.pos_spread[lo].x + g.start_off + entry(lo, tid) * ACE_START_STRIDE);
    }
}

// Weights and activations in op order: a lane per stage and sum.
ACE_HD void rc_sums(const RcArgs &a, const RcShared &s, int n, int tid) {
    const int lane = tid & 63, stage = a.waves > 1 ? lane : lane >> 1, what = a.waves > 1 ? tid >> 6 : lane & 1;
    if (stage < n && what < 2) s.sums[what * ACE_MAX_STAGES + stage] = spread_column<true>(what ? s.act : s.tmp, 0.0, s.bound[stage], s.bound[stage + 1], a.k.g.N);
}

template <bool COLL> ACE_HD void rc_memory(const RcArgs &a, const RcShared &s, int n, int tid) {
    if (tid >= n) return;
    const AceGeom &g = a.k.g;
    const double W = s.sums[tid], A = s.sums[ACE_MAX_STAGES + tid];
    double reserved = 0.0;
    if (!(g.flags & ACE_F_NO_RESERVED)) {
        PlanState<false, false, false, COLL, true> st;
        auto largest = [&](int what) {
            double x;
            __builtin_memcpy(&x, &s.reserved[what * ACE_MAX_STAGES + tid], 8);
            return x;
        };
        st.rfm = largest(0); st.rbm = largest(1); st.W = W; st.mc = largest(2);
        reserved = st.reserved_term(g);
    }
    const double x = s.in[tid] + A;
    double mem = ((((W + W * g.main_params) + W) + W * g.optimizer) + x * (double)(n - 1 - tid)) + x;
    mem = mem + reserved;
    s.mem[tid] = mem + a.peak_backward;
}

// One stage above the limit: the ops [lo, hi) of the plan, `s` its index among `n_stages`.
ACE_HD void rc_stage(const RcArgs &a, const RcShared &sh, const SpreadPlan &p, int s, int n_stages, int wave, int lane_) {
    const AceGeom &g = a.k.g;
    const int lo = sh.bound[s], hi = sh.bound[s + 1], len = hi - lo, nsb = n_stages - 1 - s;
    const uint32_t lut = sh.lut[(uint32_t)(p.glogs >> (4 * s)) & 15u];
    double *act = sh.act + lo, *tmp = sh.tmp + lo, *sum = sh.sum + wave * sh.groups;
    uint8_t *codes = sh.codes + lo;
    uint16_t *first = sh.first + wave * sh.groups;
    const uint16_t *type = sh.type + lo;
    double mem = sh.mem[s];
#ifdef ACE_HOST_EMU
    static RcLane rl[64];
    (void)lane_;
#else
    RcLane r;
    const int lane = lane_;
#endif
    RC_EACH(r.a = 0.0; r.b = 0.0; r.bad = 0; r.at = 0);
    // ---- op groups (:835-843): the stage's ops of a type, each of the size of its raw activations ----
    const uint32_t mrow = lut >> 16;
    auto raw = [&](int j, int &bad) {
        const uint32_t c = codes[j] & 7u, tp = c >> g.A_shift, al = c & (uint32_t)(g.n_algo - 1);
        uint32_t m = (mrow >> (4u * tp)) & 15u;
        if (tp >= (uint32_t)g.n_tp || m >= (uint32_t)g.n_mbs) { bad = 1; m = 0; }
        const uint32_t ty = a.pos[lo + j].y & 0xffffu;
        return a.act[((ty * (uint32_t)g.n_mbs + m) * (uint32_t)g.n_tp + (tp < (uint32_t)g.n_tp ? tp : 0u)) * (uint32_t)g.n_algo + al] * (double)(nsb + 1);
    };
    RC_EACH(
        for (int t = lane; t < sh.groups; t += 64) sum[t] = 0.0;
        for (int j = lane; j < len; j += 64) tmp[j] = raw(j, r.bad));
    RC_EACH(
        for (int j = lane; j < len; j += 64) {
            const ace_u2 e = a.pos[lo + j];
            const uint32_t before = e.x & 0xffffu;
            if (before != 0xffffu && (int)before >= lo) continue;
            double v = 0.0;
            for (int k = lo + j; k < hi; k = sh.next[k]) v += sh.tmp[k];
            const int t = type[j] & RC_GROUP;
            first[t] = (uint16_t)j;
            sum[t] = ((e.y >> 16) & 1u) ? 0.0 : v;
        });
    if (RC_ANY()) RC_EACH(if (lane == 0) RC_ATOMIC_OR(&a.flags[RC_FLAG_GRID], 1));

    // ---- the greedy loop (:849-868): every round takes one group out of `sum` ----
    double saved = 0.0, peak = 0.0;
    for (int left = sh.groups; left >= 0; --left) {
        RC_EACH(
            r.a = 0.0; r.at = 0x7fffffff;
            for (int t = lane; t < sh.groups; t += 64) {
                const double v = sum[t];
                const int at = first[t];
                if (v > r.a || (v == r.a && v > 0.0 && at < r.at)) { r.a = v; r.at = at; }
            });
        RC_BEST();
        const double best = RC_R.a;
        const int T = RC_R.at;
        if (!(best > 0.0) || T + 1 >= len) return;           // nothing left (:804) or no op after the group's first (:805)
        const double exceed = mem - a.limit;
        const uint32_t group = type[T] & RC_GROUP, also = type[T + 1] & RC_GROUP;
        int last = len;
        if (!(best < exceed)) {
            // the shortest prefix of the group that saves more than the excess (:812-816)
            RC_EACH(int bad = 0; for (int j = lane; j < len; j += 64) if ((type[j] & RC_GROUP) == group) tmp[j] = raw(j, bad));
            double v = 0.0;
            for (int k = lo + T; k < hi && v <= exceed; k = sh.next[k]) {
                v += sh.tmp[k];
                last = k - lo;
            }
        }
        RC_EACH(if (lane == 0) { sum[group] = 0.0; sum[also] = 0.0; }
                for (int j = lane; j < len; j += 64)
                    if ((type[j] & RC_GROUP) == group && j <= last) {
                        codes[j] |= 8u;
                        if (j + 1 < len) codes[j + 1] |= 8u;
                    });
        // what the recompute bits save, and the largest segment (:394-449): the first lane adds up the former, the others a segment each
        RcSaved sv;
        RC_SAVED(sv, rc_saved(codes, type, act, tmp, len, lane, r.b));
        RC_EACH(
            for (int i = lane - 1; i < sv.ends; i += 63) {
                uint32_t e = 0; int from = 0;
                if (lane) {
                    e = *reinterpret_cast<const uint32_t *>(tmp + (len - 1 - i));
                    from = i ? (int)(*reinterpret_cast<const uint32_t *>(tmp + (len - i)) & 0xffffu) : 0;
                }
                double v = spread_column<true>(sh.tmp, 0.0, lo + from, lo + (lane ? (int)(e & 0xffffu) : sv.n), g.N);
                if (!lane) { r.a = v; break; }
                if (!(e & RC_END_COUNTS)) v = 0.0;
                if (e & RC_END_PAIR) v += act[(e >> 16) & 0xfffu];
                r.b = ace_max(r.b, v);
            });
        RC_MAX(b);
        const double new_saved = RC_FROM(a, 0), new_peak = RC_R.b;     // (the same in every lane: the rounds are the wavefront's)
        mem = mem - (new_saved - saved) * (double)(nsb + 1);
        saved = new_saved;
        mem = mem + (new_peak - peak);
        peak = new_peak;
        if (!(mem - a.limit > 0.0)) return;
    }
}

ACE_HD void rc_fetch(const RcArgs &a, const RcShared &s, const SpreadPlan &p, long long plan, int tid) {
    const AceGeom &g = a.k.g;
    const int lanes = 64 * a.waves;
    for (int q = tid; q < g.G; q += lanes) {
        ace_u4 cw = a.k.codes[(size_t)q * g.P + plan];
        cw = ace_u4{cw.x & 0xf7f7f7f7u, cw.y & 0xf7f7f7f7u, cw.z & 0xf7f7f7f7u, cw.w & 0xf7f7f7f7u};
        const uint32_t w[4] = {cw.x, cw.y, cw.z, cw.w};
        uint32_t bits = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) bits |= (((((w[j] >> 4) & 0x01010101u) * 0x01020408u) >> 24) & 15u) << (4 * j);
        const int left = g.N - q * 16;
        if (left < 16) bits &= (1u << left) - 1u;            // (whatever stands behind the last op is no stage start)
        reinterpret_cast<ace_u4 *>(s.codes)[q] = cw;
        s.starts[q] = (uint16_t)bits;
        s.count[q] = (uint16_t)__builtin_popcount(bits);
    }
    for (int i = tid; i < g.N; i += lanes) {
        const ace_u2 e = a.pos[i];
        s.type[i] = (uint16_t)((e.y >> 17) | (((a.k.pos_spread[i].y >> 8) & 3u) << 14));
        s.next[i] = (uint16_t)(e.x >> 16);
    }
    if (tid < 16) s.lut[tid] = a.k.stage_lut[p.bidx * 16u + (uint32_t)tid];
    if (tid < 18) s.bound[tid] = g.N;
    if (tid < 3 * ACE_MAX_STAGES) s.reserved[tid] = 0ull;
    if (tid == 0) { s.act[g.N] = 0.0; s.tmp[g.N] = 0.0; }
}

#ifdef ACE_HOST_EMU
#define RC_PHASE(...) for (int tid = 0; tid < 64 * a.waves; ++tid) { __VA_ARGS__; }
#define RC_WAVES(...) for (int wave = 0; wave < a.waves; ++wave) { const int lane0 = 0; __VA_ARGS__; }
#else
#define RC_PHASE(...) { __VA_ARGS__; } __syncthreads()
#define RC_WAVES(...) { const int wave = tid >> 6, lane0 = tid & 63; __VA_ARGS__; } __syncthreads()
#endif
template <bool COLL> ACE_HD void ace_rc_body(const RcArgs &a, unsigned char *lds_raw, int tid_, long long plan) {
    const AceGeom &g = a.k.g;
    RcShared s;
    ace_rc_layout(a, lds_raw, &s);
    SpreadShared sp;            // (the part spread_stages works on)
    sp.starts = s.starts; sp.count = s.count; sp.prefix = s.prefix; sp.bound = s.bound; sp.n_stages = s.n_stages;
#ifdef ACE_HOST_EMU
    (void)tid_;
#else
    const int tid = tid_;
#endif
    const SpreadPlan p = spread_plan<false>(a.k, plan);
    RC_PHASE(rc_fetch(a, s, p, plan, tid));
    RC_PHASE(for (int q = tid; q < g.G; q += 64 * a.waves) spread_stages(a.k, sp, q));
    const int n = *s.n_stages, S = (int)(p.h.x & 0xffu);
    RC_PHASE(
        if (tid == 0) {
            if (n != S) RC_ATOMIC_ADD(&a.flags[RC_FLAG_COUNT], n - S);
            if (!(s.starts[0] & 1u)) RC_ATOMIC_OR(&a.flags[RC_FLAG_FIRST], 1);
            if (a.status[plan]) RC_ATOMIC_OR(&a.flags[RC_FLAG_STATUS], 1);
        });
    // (an inconsistent plan is reported and keeps its cleared bits)
    if (n == S && n <= ACE_MAX_STAGES && (s.starts[0] & 1u)) {
        RC_PHASE(rc_load<COLL>(a, s, p, n, tid));
        RC_PHASE(rc_sums(a, s, n, tid));
        RC_PHASE(rc_memory<COLL>(a, s, n, tid));
        RC_WAVES(int turn = 0; for (int st = 0; st < n; ++st) if (s.mem[st] - a.limit > 0.0 && turn++ % a.waves == wave) rc_stage(a, s, p, st, n, wave, lane0));
    }
    RC_PHASE(for (int q = tid; q < g.G; q += 64 * a.waves) a.codes_out[(size_t)q * g.P + plan] = reinterpret_cast<const ace_u4 *>(s.codes)[q]);
}

// Per position: previous and next op of the same type, the type, whether its ops are never recomputed, its group -- the types in use
// in the order of their numbers; returns how many they are.  (Host side.)
inline int ace_rc_positions(const int32_t *type_of_pos, const uint8_t *norec, int N, int n_types, ace_u2 *out) {
    for (int i = 0; i < N; ++i) out[i] = ace_u2{0u, (uint32_t)type_of_pos[i] | ((uint32_t)(norec[type_of_pos[i]] != 0) << 16)};
    uint32_t groups = 0;
    for (int t = 0; t < n_types; ++t) {
        uint32_t before = 0xffffu;
        for (int i = 0; i < N; ++i)
            if (type_of_pos[i] == t) {
                out[i].x = before | ((uint32_t)N << 16);
                out[i].y |= groups << 17;
                if (before != 0xffffu) out[before].x = (out[before].x & 0xffffu) | ((uint32_t)i << 16);
                before = (uint32_t)i;
            }
        groups += before != 0xffffu ? 1u : 0u;
    }
    return (int)groups;
}

// Wavefronts of a workgroup: as few as share the stages above the limit among them, so that a CU has room for more plans (one / two / three:
// 299 / 244 / 269 us for 16,384 plans of 523 ops); one where the sizes of two wavefronts' groups would not fit in LDS.
inline int ace_rc_waves(int N, int G, int groups, uint32_t lds) {
    RcShared s;
    return ace_rc_layout(N, G, groups, 2, nullptr, &s) <= lds ? 2 : 1;
}
