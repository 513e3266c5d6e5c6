// Scoring of MID-SIZED batches (plain scoring, rows resident in LDS): a plan is walked by several lanes of different wavefronts.
//
// With fewer plans than the chip has lanes at four wavefronts per SIMD, what counts is how long one wavefront takes for the
// sequence.  In the kernel of large batches (ace_dense.h), whose tables these are, that is 220 ns per op for a lone wavefront: some
// 50 instructions of all kinds.  Here
//   * a plan's accumulators are divided: a "time" lane walks the ops for the compute, recompute and resharding sums, a
//     "memory" lane of another wavefront for weights, activations and the rest;
//   * the sequence is divided: a lane walks one of up to six parts of it.  A stage belongs to the part in which it starts,
//     whose lane walks on to the stage's end; how many stages start in the parts before is counted first.  A plan of few
//     stages gains nothing (its first part's lane walks nearly all ops, but hardly any of them ends a stage), one of many,
//     whose every op costs its wavefront twice the instructions, gains most: so the two balance;
//   * the tables go to LDS by LDS-direct loads, all in flight at once, while the workgroup deals its plans;
//   * the stages' tails are divided over the same lanes.
// No accumulator of a stage depends on another's or on an earlier stage's, so each is added up in op order as everywhere and
// the results are the same bits.
//
// Measured, us per launch, over the table compiler's rows (27 instructions per op and role, scalars of a position by v_readlane) ->
// over the dense tables:
//   plans      315 ops        523 ops       821 ops (no resharding)   1,251 ops
//    8,192     43.1 -> 31.9   67.3 -> 50.8   81.2 -> 67.1             107.3 -> 81.6
//   16,384     43.9 -> 33.1   68.4 -> 51.4   81.7 -> 67.5             112.1 -> 86.5
//   32,768     49.4 -> 37.3   80.1 -> 58.5   94.3 -> 73.9             149.4 -> 115.9
//   65,536     61.4 -> 44.3   106.7 -> 76.8  125.1 -> 88.0            209.8 -> 159.0
// Up to 16,384 plans the longest wavefront is what is waited for (the memory role of the first part: 250 cycles per op while the stages
// of its 64 plans end, 160 afterwards, for 24 instructions), from 65,536 on the SIMDs have two and more wavefronts to issue for all
// the time.
// Tables that are resident as the table compiler lays them out and not in the dense form have no such kernel any more: with resharding
// one constant byte names every row, so rows of more than 63 KB together go through windows (134 types of 16 entries, 134 ops: 10,000
// plans 31.5 -> 35.5 us, 24,576 37.4 -> 39.2, 65,536 54.8 -> 45.7) or, with more distinct sizes than the lists hold, over the table
// compiler's rows (10,000 32.5 -> 34.8, 24,576 36.6 -> 37.7, 65,536 45.8 -> 41.0); below 8,000 the kernel of small batches has them (28 against 31).
#pragma once
#include "ace_dense.h"

// Plans per workgroup: the number that fills the 256 CUs with one workgroup each (sixteen wavefronts of this many registers are all
// that a CU holds).  Above 256 plans per CU the kernel of large batches takes over (512 plans per workgroup here, in one part, against
// that: 100,000 plans of 523 ops 108 / 121 us and 131,072 115 / 122, but of 1,251 ops 269 / 226 and 318 / 239, of 821 126 / 117;
// 65,536 plans of 523 ops 77 / 117): 0.
inline int ace_duo_lanes(long long plans) {
    for (int L = 64; L <= 256; L *= 2)
        if (plans <= 256ll * L) return L;
    return 0;
}

#ifndef ACE_HOST_EMU
#include "ace_duo_loop_asm.inc"

#define ACE_DUO_RUN(TEXT)                                                                                                         \
    asm volatile(TEXT :                                                                                        \
                 : [glogs] "v"(glogs), [lut2] "v"(lut2), [zvrk] "v"(zvrk), [codeoff] "v"(code_off), [recoff] "v"(rec_off),        \
                   [codes] "s"(codes), [pos] "s"(pos), [n_ops] "s"(a.g.N), [recbase] "s"(rec_base),                          \
                   [gstride_lo] "s"((uint32_t)gstride), [gstride_hi] "s"((uint32_t)(gstride >> 32)), [wsstride] "s"(ws_stride),   \
                   [wspiece] "s"(ws_piece), [grp] "s"(grp), [cut] "s"(cut), [recnext] "v"(rec_next), [kv] "s"(d.kv)           \
                 : ACE_DUO_ASM_CLOBBERS)
// Walks one part of the lane's plan, from 16-op group `grp` on; the stages that start in front of position `cut` are parked, the
// first one at `rec_off`, the next at `rec_next` (kNoRecord: nowhere).  `role` is the same for the whole wavefront, and all 64
// lanes are active.
constexpr uint32_t kNoRecord = 0x80000000u;
__device__ __forceinline__ void duo_loop(const AceKernelArgs &a, const AceDenseArgs &d, uint32_t role, uint32_t grp, uint32_t cut, uint64_t glogs, uint32_t lut2,
                                         uint64_t zvrk, uint32_t code_off, const double *rec_base, uint32_t rec_off, uint32_t rec_next,
                                         uint32_t ws_stride, uint32_t ws_piece) {
    const uint64_t gstride = (uint64_t)(uint32_t)a.g.P * 16u;
    const unsigned char *codes = reinterpret_cast<const unsigned char *>(a.codes) + gstride * grp;
    const ace_u2 *pos = d.pos_duo + (size_t)(role ? (uint32_t)a.g.G + 1u + grp : grp) * 16u;
    if (a.g.flags & ACE_F_RESHARDING) {
        if (role == 0) ACE_DUO_RUN(ACE_DUO_ASM_TIME_RSH1);
        else ACE_DUO_RUN(ACE_DUO_ASM_MEMORY_RSH1);
    } else {
        if (role == 0) ACE_DUO_RUN(ACE_DUO_ASM_TIME_RSH0);
        else ACE_DUO_RUN(ACE_DUO_ASM_MEMORY_RSH0);
    }
}
#undef ACE_DUO_RUN

// The stashed stages first, first + step, ... (< n_st) of the lane's plan: `take(s, ms, MB)` gets what each came to.  What links a stage
// to the one before it (code and list of its first op) is that one's record word; the first stage's is `meta0`.  Three records in flight.
template <class Take>
__device__ __forceinline__ void duo_tails(const AceDenseArgs &d, const AceGeom &g, const AceLds &lds, DenseState &st, const unsigned char *rec, uint32_t stride,
                                          uint32_t piece, int first, int step, int n_st, uint32_t meta0, Take take) {
    DenseRecord r[3];
    auto fetch = [&](int s2, DenseRecord &x) {
        const unsigned char *p = rec + (size_t)s2 * stride;
#pragma unroll
        for (uint32_t j = 0; j < 4u; ++j) x.r[j] = *reinterpret_cast<const ace_d2 *>(p + j * piece);
        const ace_u2 t = *reinterpret_cast<const ace_u2 *>(p + 4u * piece);
        x.tail = ace_u4{t.x, t.y, s2 > 0 ? reinterpret_cast<const ace_u2 *>(p - stride + 4u * piece)->y : meta0, 0u};
    };
#pragma unroll
    for (int k = 0; k < 3; ++k)
        if (first + k * step < n_st) fetch(first + k * step, r[k]);
    for (int base = first; base < ACE_MAX_STAGES; base += 3 * step) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const int s2 = base + k * step;
            if (!__any(s2 < n_st)) return;
            if (s2 < n_st) {
                dense_tail(d, g, lds, st.bidx, (uint32_t)(st.glogs >> (4u * (uint32_t)s2)) & 15u, (uint32_t)s2, r[k], st);
                if (s2 + 3 * step < n_st) fetch(s2 + 3 * step, r[k]);
                take(s2, st.sum_t, st.max_mem);
            }
        }
    }
}

// Stage starts among the first `left` of eight op bytes.
__device__ __forceinline__ uint32_t starts_in(uint64_t bytes, int left) {
    const uint64_t m = left >= 8 ? ~0ull : left > 0 ? (1ull << (8 * left)) - 1ull : 0ull;
    return (uint32_t)__popcll(bytes & m & 0x1010101010101010ull);
}

// Which slice of 64 plans (the deepest first) and which part of the sequence each of a role's eight wavefronts walks, and the
// number of parts of each slice: four bits each, the first lowest (a part that the slice does not have: the wavefront idles).
// Consecutive wavefronts run on different SIMDs.  Measured, plans of 523 / 1,251 ops: with 64 plans, 5 / 6 / 8 parts 52.2 / 50.8 / 51.6 and
// 90.8 / 81.4 / 91.4 us (8,192 plans); with 128: 4 + 4 parts 58.7 and 116.3, 5 + 3 57.4 and 112.0 or, in another order of the wavefronts,
// 69.3 and 134.5 (32,768); with 256: 2 each 77.7 and 159.1, 3 + 2 + 2 + 1 77.7 and 178.0, 4 + 2 + 1 + 1 77.0 and 180.6 us (65,536).
template <int L> struct DuoDeal;
template <> struct DuoDeal<64> { static constexpr uint32_t v[3] = {0x00000000u, 0xff543210u, 0x6u}; };
template <> struct DuoDeal<128> { static constexpr uint32_t v[3] = {0x10101010u, 0x33221100u, 0x44u}; };
template <> struct DuoDeal<256> { static constexpr uint32_t v[3] = {0x32103210u, 0x11110000u, 0x2222u}; };

// One workgroup: L plans.  The LDS array starts at address 0 (the kernel has no other LDS variables).
template <int L>
__device__ __forceinline__ void ace_duo_body(const AceKernelArgs &a, const AceDenseArgs &d, unsigned char *lds_raw, int tid, long long block) {
    typedef DuoDeal<L> Deal;
    AceGeom g = a.g;
    g.out_off = 0u;                                                 // (what the evaluation indexes the outputs' addresses by)
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(tid >> 6), lane = (uint32_t)tid & 63u;
    // (the memory role's wavefronts in fours in reverse: a SIMD gets different slices of the two roles)
    const uint32_t role = wave >> 3, m = role ? (wave & 7u) ^ 3u : wave;
    const uint32_t slice = (Deal::v[0] >> (4u * m)) & 15u, part = (Deal::v[1] >> (4u * m)) & 15u, parts = (Deal::v[2] >> (4u * slice)) & 15u;
    const bool idle = part >= parts;
    const uint32_t grp = idle ? 0u : (part * (uint32_t)g.G + parts - 1u) / parts, grp_end = idle ? 0u : ((part + 1u) * (uint32_t)g.G + parts - 1u) / parts;
    dense_stage_image<kDuoBlock>(d, lds_raw, wave, lane);
    // Plans are dealt to the lanes by pipeline depth, like in ace_score_body: every op at which a lane closes a stage costs
    // its whole wavefront the stage-end code.
    unsigned int *cnt = reinterpret_cast<unsigned int *>(lds_raw + d.image16 * 16u);
    unsigned short *plan_of = reinterpret_cast<unsigned short *>(cnt + 32);
    unsigned short *starts = plan_of + L;                           // [role][wavefront's place in Deal][lane]
    uint32_t at = lane;                                             // the lane's place in the sorted workgroup
    if (L > 64) {
        if (tid < 32) cnt[tid] = 0u;
        const long long slot = block * L + tid;
        uint32_t depth = 0, rank = 0;                               // (slots past the batch: last)
        if (tid < L && slot < g.P) {
            depth = a.hdr[slot].x & 0xffu;
            depth = depth > 16u ? 16u : depth;
        }
        __syncthreads();
        if (tid < L) rank = atomicAdd(&cnt[16u - depth], 1u);
        __syncthreads();
        if (tid < L) {
            for (uint32_t b = 0; b < 16u - depth; ++b) rank += cnt[b];
            plan_of[rank] = (unsigned short)tid;
        }
        __syncthreads();
        at = (slice << 6) | lane;
    }
    const long long plan = block * L + (L > 64 ? (uint32_t)plan_of[at] : at);
    const bool in_batch = plan < g.P;
    const long long pl = in_batch ? plan : (long long)g.P - 1;      // plan this lane reads
    const long long out = a.order ? (long long)a.order[pl] : plan;
    const bool active = in_batch && out < g.P;
    const ace_u4 h = a.hdr[pl];
    // Stages that start in this part (every role counts half of its groups), in the parts before it, and altogether.
    uint32_t own = 0, before = 0, first = 0, n_st = 0;
    if (grp < grp_end) first = a.codes[(size_t)grp * g.P + pl].x & 0x1fu;
    {
        const uint32_t mid = (grp + grp_end + 1u) >> 1, end = role ? grp_end : mid;
        for (uint32_t k0 = role ? mid : grp; k0 < end; k0 += 8u) {
            ace_u4 c[8];
#pragma unroll
            for (uint32_t k = 0; k < 8u; ++k) c[k] = a.codes[(size_t)(k0 + k < end ? k0 + k : k0) * g.P + pl];
#pragma unroll
            for (uint32_t k = 0; k < 8u; ++k) {
                const int left = k0 + k < end ? g.N - 16 * (int)(k0 + k) : 0;       // (bytes past the last op are anything)
                own += starts_in((uint64_t)c[k].y << 32 | c[k].x, left) + starts_in((uint64_t)c[k].w << 32 | c[k].z, left - 8);
            }
        }
        starts[(role * 8u + m) * 64u + lane] = (unsigned short)own;
        __syncthreads();
#pragma unroll
        for (uint32_t k = 0; k < 8u; ++k) {
            if (((Deal::v[0] >> (4u * k)) & 15u) != slice) continue;
            const uint32_t p = (Deal::v[1] >> (4u * k)) & 15u, n = (uint32_t)starts[k * 64u + lane] + (uint32_t)starts[(8u + k) * 64u + lane];
            if (p < part) before += n;
            if (p == part) own = n;
            n_st += n;
        }
    }
    const uint32_t code0 = a.codes[pl].x & 0x1fu;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                 // the tables
    __syncthreads();

    const AceLds lds = ace_make_lds(lds_raw, 0u);
    DenseState st;
    st.init(g, lds, h, ace_u2{0u, 0u});
    double *rec_base = a.stage_ws + (size_t)block * ACE_MAX_STAGES * L * ACE_WS_REC;
    constexpr uint32_t kStride = L * ACE_WS_REC * 8u, kPiece = L * 16u;
    // the part's first position is in stage `before` (it starts there), or in the one before that
    const bool opens = part == 0u || (first & 0x10u) != 0u, any = part == 0u || own != 0u;
    const uint32_t here = before + (opens ? 1u : 0u);                // one more than the index of that stage
    // Issue priority to the longest walk of a slice, the first part's; without resharding the time role's step is half the memory's, whose
    // walks go first then (65,536 plans of 821 ops 93.7 -> 88.0 us, 16,384 68.4 -> 67.5; with resharding 1,251 ops lose 0.7 % by it).
    // No priorities: 523 ops, 32,768 plans 58.6 -> 64.0.
    if (part == 0u && (role || (g.flags & ACE_F_RESHARDING))) __builtin_amdgcn_s_setprio(3);
    else if (part == 0u) __builtin_amdgcn_s_setprio(2);
    else if (role && !(g.flags & ACE_F_RESHARDING)) __builtin_amdgcn_s_setprio(1);
    if (grp < grp_end && __any(any)) {
        const uint32_t shift = here > 1u ? 4u * (here - 1u) : 0u, lut = d.lut_off + st.bidx * 128u, to = at * 16u + role * 2u * kPiece;
        const uint64_t glogs = shift < 64u ? st.glogs >> shift : 0ull;
        duo_loop(a, d, role, grp, part + 1u < parts ? 16u * grp_end : 0x7fffffffu, glogs >> 1, lut, lds.ld<uint64_t>(lut + ((uint32_t)glogs & 15u) * 8u),
                    (uint32_t)pl * 16u, rec_base, opens ? to + before * kStride : kNoRecord, any ? to + here * kStride : kNoRecord, kStride, kPiece);
    }
    __builtin_amdgcn_s_setprio(0);
    __syncthreads();                                                // all pieces of the records
    // Stage tails: every lane evaluates its role's half of every `parts`-th stage and leaves the stage times / the largest
    // stage memory in places of the records that only this lane reads; then one lane per plan puts the plan together.
    double *rec = rec_base + (size_t)at * 2;
    const int n_live = (int)(n_st < ACE_MAX_STAGES ? n_st : ACE_MAX_STAGES);
    const uint32_t meta0 = ((code0 & 7u) << 8) | (d.first_in << 24);
    const unsigned char *recs = reinterpret_cast<const unsigned char *>(rec);
    if (idle) {
    } else if (role) {
        double most = 0.0;
        duo_tails(d, g, lds, st, recs, kStride, kPiece, (int)part, (int)parts, n_live, meta0, [&](int, double, double mb) { most = ace_max(most, mb); });
        rec[(size_t)part * (kStride / 8u) + 2u * (kPiece / 8u)] = most;
    } else
        duo_tails(d, g, lds, st, recs, kStride, kPiece, (int)part, (int)parts, n_live, meta0, [=](int s, double t, double) { rec[(size_t)s * (kStride / 8u)] = t; });
    __syncthreads();
    if (role || part) return;
    // (all loads before the first use: one trip to memory)
    double t[ACE_MAX_STAGES], sum = 0.0, mx = 0.0, mem = 0.0;
#pragma unroll
    for (int s = 0; s < ACE_MAX_STAGES; ++s) {
        t[s] = 0.0;
        if (s < n_live) t[s] = rec[(size_t)s * (kStride / 8u)];
    }
    double pm[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        pm[k] = 0.0;
        if (k < (int)parts) pm[k] = rec[(size_t)k * (kStride / 8u) + 2u * (kPiece / 8u)];
    }
#pragma unroll
    for (int s = 0; s < ACE_MAX_STAGES; ++s) {
        sum += t[s];                                            // (stage times are sums from +0.0: adding 0.0 changes nothing)
        mx = ace_max(mx, t[s]);
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) mem = ace_max(mem, pm[k]);
    st.s = (int)n_st;
    st.sum_t = sum; st.max_t = mx; st.max_mem = mem;
    if (!(code0 & 0x10u)) st.status = ACE_PLAN_MALFORMED;            // the first op must open a stage
    double iter, peak;
    uint8_t feas, stat;
    st.result(g, a.nbm1[st.bidx], iter, peak, feas, stat);
    if (active) {
        a.iter_ms[out] = iter;
        a.peak_mb[out] = peak;
        a.feasible[out] = feas;
        if (a.status) a.status[out] = stat;
    }
}
#endif
