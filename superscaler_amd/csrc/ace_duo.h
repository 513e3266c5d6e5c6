// Scoring of MID-SIZED batches (plain scoring, rows resident in LDS): a plan is walked by several lanes of different wavefronts.
//
// With fewer plans than the chip has lanes at four wavefronts per SIMD, what counts is how long one wavefront takes for the
// sequence.  In the kernel of large batches (ace_score_loop.h) that is 250 ns per op for a lone wavefront: 35 vector
// instructions, a scalar one for each of them, and two LDS latencies that nothing else on the SIMD covers.  Here
//   * a plan's accumulators are divided: a "time" lane walks the ops for the compute, recompute and resharding sums, a
//     "memory" lane of another wavefront for weights, activations and the rest;
//   * the sequence is divided: a lane walks one of up to six parts of it.  A stage belongs to the part in which it starts,
//     whose lane walks on to the stage's end; how many stages start in the parts before is counted first.  A plan of few
//     stages gains nothing (its first part's lane walks nearly all ops, but hardly any of them ends a stage), one of many,
//     whose every op costs its wavefront twice the instructions, gains most: so the two balance;
//   * the op loop (gen_duo_loop_asm.py) asks for everything it reads two to four ops ahead;
//   * the rows go to LDS by LDS-direct loads, all in flight at once, while the workgroup deals its plans;
//   * the stages' tails are divided over the same lanes.
// No accumulator of a stage depends on another's or on an earlier stage's, so each is added up in op order as everywhere and
// the results are the same bits.
//
// Measured, us per launch, before (one lane per plan, 256 lanes per workgroup) -> now:
//   plans      315 ops        523 ops       821 ops (no resharding)   1,251 ops
//    8,192     65.6 -> 43.8   131.8 -> 68.5   136.7 -> 83.7           254.4 -> 109.1
//   16,384     66.0 -> 47.3   131.3 -> 72.4   136.9 -> 87.0           258.6 -> 117.1
//   32,768     67.0 -> 53.2   135.3 -> 85.7   140.1 -> 98.5           259.0 -> 160.7
//   65,536     70.8 -> 65.9   139.5 -> 114.4  142.7 -> 130.1          264.9 -> 228.6
// Up to 16,384 plans the longest wavefront is what is waited for (about 220 cycles per op, of which 110 are the issue of its
// 27 instructions), from 65,536 on the SIMDs have two and more wavefronts to issue for all the time.
#pragma once
#include "ace_score_loop.h"

// Plans per workgroup: the number that fills the 256 CUs with one workgroup each (the rows take most of a CU's LDS).  Above
// 256 plans per CU the kernel of large batches is the faster one (ace_many.h; 131,072 plans of 523 ops: 141 us, 512 plans per
// workgroup here 162; 65,536 plans: 114 us here, 134 there): 0.
inline int ace_duo_lanes(long long plans) {
    for (int L = 64; L <= 256; L *= 2)
        if (plans <= 256ll * L) return L;
    return 0;
}
constexpr int kDuoBlock = 1024;     // lanes of a workgroup: eight wavefronts per role
// LDS of the workgroup beyond the tables: the deal of the plans keeps its bins, its permutation and the parts' stage counts
// where the small tables go.
inline uint32_t ace_duo_lds(const AceGeom &g, uint32_t lds_bytes, int L) {
    const uint32_t deal = g.rk_lds_off + 128u + 2u * (uint32_t)L + 2u * (uint32_t)kDuoBlock;
    return deal > lds_bytes ? deal : lds_bytes;
}

#ifndef ACE_HOST_EMU
#include "ace_duo_loop_asm.inc"

// The rows, as one block from LDS address 0 on (a.flat_rows16 > 0): 1 KB per wavefront and load.
template <int BLOCK> __device__ __forceinline__ void duo_rows(const AceKernelArgs &a, unsigned char *lds_raw, uint32_t wave, uint32_t lane) {
    typedef const void __attribute__((address_space(1))) *gptr;
    typedef void __attribute__((address_space(3))) *lptr;
    const uint32_t n = (uint32_t)a.flat_rows16;
    const unsigned char *src = reinterpret_cast<const unsigned char *>(a.rows);
    for (uint32_t at = wave * 64u; at < n; at += BLOCK)
        if (at + lane < n) __builtin_amdgcn_global_load_lds((gptr)(src + (size_t)(at + lane) * 16u), (lptr)(lds_raw + at * 16u), 16, 0, 0);
}

#define ACE_DUO_RUN(TEXT)                                                                                                         \
    asm volatile(TEXT :                                                                                        \
                 : [glogs] "v"(glogs), [lut2] "v"(lut2), [codeoff] "v"(code_off), [recoff] "v"(rec_off), [zerop] "v"(zero_pair),  \
                   [codes] "s"(codes), [pos] "s"(pos), [n_ops] "s"(a.g.N), [recbase] "s"(rec_base),                          \
                   [gstride_lo] "s"((uint32_t)gstride), [gstride_hi] "s"((uint32_t)(gstride >> 32)), [wsstride] "s"(ws_stride),   \
                   [wspiece] "s"(ws_piece), [grp] "s"(grp), [cut] "s"(cut), [recnext] "v"(rec_next)                                 \
                 : ACE_DUO_ASM_CLOBBERS)
// Walks one part of the lane's plan, from 16-op group `grp` on; the stages that start in front of position `cut` are parked, the
// first one at `rec_off`, the next at `rec_next` (kNoRecord: nowhere).  `role` is the same for the whole wavefront, and all 64
// lanes are active.
constexpr uint32_t kNoRecord = 0x80000000u;
__device__ __forceinline__ void duo_loop(const AceKernelArgs &a, uint32_t role, uint32_t grp, uint32_t cut, uint64_t glogs, uint32_t lut2,
                                         uint32_t code_off, uint32_t zero_pair, const double *rec_base, uint32_t rec_off,
                                         uint32_t rec_next, uint32_t ws_stride, uint32_t ws_piece) {
    const uint64_t gstride = (uint64_t)(uint32_t)a.g.P * 16u;
    const unsigned char *codes = reinterpret_cast<const unsigned char *>(a.codes) + gstride * grp;
    const ace_u4 *pos = a.pos4 + (size_t)grp * 16u;
    if (role == 0) {
        if (a.g.flags & ACE_F_RESHARDING) ACE_DUO_RUN(ACE_DUO_ASM_TIME_RSH1);
        else ACE_DUO_RUN(ACE_DUO_ASM_TIME_RSH0);
    } else {
        if (a.g.flags & ACE_F_NO_RESERVED) ACE_DUO_RUN(ACE_DUO_ASM_MEMORY_NONE);
        else if (a.g.flags & ACE_F_RESERVED_MIN) ACE_DUO_RUN(ACE_DUO_ASM_MEMORY_MIN);
        else ACE_DUO_RUN(ACE_DUO_ASM_MEMORY_MAX);
    }
}
#undef ACE_DUO_RUN

// Stage starts among the first `left` of eight op bytes.
__device__ __forceinline__ uint32_t starts_in(uint64_t bytes, int left) {
    const uint64_t m = left >= 8 ? ~0ull : left > 0 ? (1ull << (8 * left)) - 1ull : 0ull;
    return (uint32_t)__popcll(bytes & m & 0x1010101010101010ull);
}

// Which slice of 64 plans (the deepest first) and which part of the sequence each of a role's eight wavefronts walks, and the
// number of parts of each slice: four bits each, the first lowest (a part that the slice does not have: the wavefront idles).
// Consecutive wavefronts run on different SIMDs.  Measured with 64 plans: 4 / 5 / 6 / 8 parts 76.0 / 75.2 / 72.4 / 72.9 us
// (16,384 plans, 523 ops); with 128: 4 + 4 parts 85.7, 5 + 3 87.4, 3 + 3 88.8 us (32,768); with 256: 2 each 114.4, 3 + 2 + 2 + 1
// 118.0, 1 each 139.0 us (65,536).
template <int L> struct DuoDeal;
template <> struct DuoDeal<64> { static constexpr uint32_t v[3] = {0x00000000u, 0xff543210u, 0x6u}; };
template <> struct DuoDeal<128> { static constexpr uint32_t v[3] = {0x10101010u, 0x33221100u, 0x44u}; };
template <> struct DuoDeal<256> { static constexpr uint32_t v[3] = {0x32103210u, 0x11110000u, 0x2222u}; };

// One workgroup: L plans.  The LDS array starts at address 0 (the kernel has no other LDS variables).
template <int L> __device__ __forceinline__ void ace_duo_body(const AceKernelArgs &a, unsigned char *lds_raw, int tid, long long block) {
    typedef DuoDeal<L> Deal;
    const AceGeom &g = a.g;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(tid >> 6), lane = (uint32_t)tid & 63u;
    // (the memory role's wavefronts in fours in reverse: a SIMD gets different slices of the two roles)
    const uint32_t role = wave >> 3, m = role ? (wave & 7u) ^ 3u : wave;
    const uint32_t slice = (Deal::v[0] >> (4u * m)) & 15u, part = (Deal::v[1] >> (4u * m)) & 15u, parts = (Deal::v[2] >> (4u * slice)) & 15u;
    const bool idle = part >= parts;
    const uint32_t grp = idle ? 0u : (part * (uint32_t)g.G + parts - 1u) / parts, grp_end = idle ? 0u : ((part + 1u) * (uint32_t)g.G + parts - 1u) / parts;
    duo_rows<kDuoBlock>(a, lds_raw, wave, lane);
    // Plans are dealt to the lanes by pipeline depth, like in ace_score_body: every op at which a lane closes a stage costs
    // its whole wavefront the stage-end code.
    unsigned int *cnt = reinterpret_cast<unsigned int *>(lds_raw + g.rk_lds_off);
    unsigned short *plan_of = reinterpret_cast<unsigned short *>(lds_raw + g.rk_lds_off + 128);
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
    __syncthreads();
    stage_small_tables<kDuoBlock, true>(a, lds_raw, tid);
    // (a word no block of the pair-kind table uses: what the loop reads for a stage's first op)
    const uint32_t zero_pair = g.pk32_lds_off + 64u * 4u;
    if (tid == 0) *reinterpret_cast<uint32_t *>(lds_raw + zero_pair) = 0u;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                 // the rows
    __syncthreads();

    const AceLds lds = ace_make_lds(lds_raw, 0u);
    PlanState<false, false, true> st;
    st.init(g, lds, h, ace_u2{0u, 0u});
    double *rec_base = a.stage_ws + (size_t)block * ACE_MAX_STAGES * L * ACE_WS_REC;
    constexpr uint32_t kStride = L * ACE_WS_REC * 8u, kPiece = L * 16u;
    // the part's first position is in stage `before` (it starts there), or in the one before that
    const bool opens = part == 0u || (first & 0x10u) != 0u, any = part == 0u || own != 0u;
    const uint32_t here = before + (opens ? 1u : 0u);                // one more than the index of that stage
    if (part == 0u) __builtin_amdgcn_s_setprio(3);                  // (the longest walk of a slice: 78.3 -> 72.9 us, 16,384 plans of 523 ops)
    if (grp < grp_end && __any(any)) {
        const uint32_t shift = here > 1u ? 4u * (here - 1u) : 0u;
        duo_loop(a, role, grp, part + 1u < parts ? 16u * grp_end : 0x7fffffffu, shift < 64u ? st.glogs >> shift : 0ull,
                 g.lut2a_lds_off + st.bidx * 128u, (uint32_t)pl * 16u, zero_pair, rec_base,
                 opens ? at * 16u + before * kStride : kNoRecord, any ? at * 16u + here * kStride : kNoRecord, kStride, kPiece);
    }
    __builtin_amdgcn_s_setprio(0);
    __syncthreads();                                                // all pieces of the records
    // Stage tails: every lane evaluates its role's half of every `parts`-th stage and leaves the stage times / the largest
    // stage memory in places of the records that only this lane reads; then one lane per plan puts the plan together.
    double *rec = rec_base + (size_t)at * 2;
    const int n_live = (int)(n_st < ACE_MAX_STAGES ? n_st : ACE_MAX_STAGES);
    st.ws_stride = kStride / 16u;
    st.ws_piece = kPiece / 16u;
    const uint32_t code0 = a.codes[pl].x & 0x1fu, row0 = a.pos_info[0] & 0xffu;
    if (idle) {
    } else if (role) {
        st.replay_some(g, lds, rec, (int)part, (int)parts, n_live, code0 & 7u, row0, [](int, double) {});
        rec[(size_t)part * (kStride / 8u) + 2u * (kPiece / 8u)] = st.max_mem;
    } else
        st.replay_some(g, lds, rec, (int)part, (int)parts, n_live, code0 & 7u, row0,
                       [=](int s, double t) { rec[(size_t)s * (kStride / 8u)] = t; });
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
