// Scoring of LARGE batches where the assembly op loop runs: the kernel of ace_score_loop.h (a plan per lane, up to sixteen
// wavefronts per workgroup and CU) with workgroups of as many plans as make an even share.  For tables that do not fit the dense
// form (ace_dense.h): more distinct costs or sizes than its lists hold.  They come here from what the kernel of small batches leaves
// (ace_route.h): the kernel of mid-sized batches (ace_duo.h) walks dense tables alone.
//
// The rows fill a CU's LDS, so the workgroups of a batch run in rounds of 256, and with 1,024 plans each a batch of 200,000
// leaves a fifth of the CUs idle and the last 37,856 plans of one of 300,000 take a second round of their own.  Here a
// workgroup takes 64 * slices plans, at most 1,024, so that the rounds the batch needs are all full.  (One workgroup per CU
// that stages once and walks several rounds, with or without a barrier between them, was slower: 1,048,576 plans of 523 ops
// 757 / 797 us instead of 729.)  Rows that are resident are staged by LDS-direct loads; windowed rows are fetched while the
// loop walks, by all sixteen wavefronts: those without plans do nothing else.
// Measured, us per launch, before -> now (tables of five graphs that the dense form has taken over since):
//   plans      315 ops          523 ops          821 ops          1,251 ops
//   100,000   132.4 -> 69.1    263.9 -> 136.5   272.4 -> 139.8   517.1 -> 293.0     (two rounds of 256-lane workgroups before)
//   131,072    88.9 -> 71.2    163.4 -> 141.4   161.7 -> 142.9   422.6 -> 305.1
//   200,003    94.3 -> 86.5    174.9 -> 169.1   172.8 -> 170.2   456.6 -> 416.6
//   300,000   178.0 -> 152.7   338.6 -> 297.2   326.0 -> 310.3   864.7 -> 740.2
//   600,000   275.3 -> 258.8   525.7 -> 507.6   505.6 -> 497.6  1328.8 -> 1185.7
//   windowed, 134 ops: 8,192 plans 76.8 -> 45.9, 65,536 84.9 -> 57.5, 131,072 86.0 -> 66.5, 300,000 172.8 -> 139.0
// and the same for whole rounds.  What bounds it is the issue of vector instructions (the op loop) up to the batch's last op,
// and then the records coming back from memory.
#pragma once
#include "ace_duo.h"

// Slices of 64 plans per workgroup.
inline uint32_t ace_many_slices(long long plans) {
    const long long fullest = ((plans + 63) / 64 + 255) / 256;       // slices of the batch on the fullest CU
    const long long rounds = (fullest + 15) / 16;
    return (uint32_t)((fullest + rounds - 1) / rounds);
}

#ifndef ACE_HOST_EMU
// The rows, as one block from LDS address 0 on (a.flat_rows16 > 0): 1 KB per wavefront and load.
template <int BLOCK> __device__ __forceinline__ void many_rows(const AceKernelArgs &a, unsigned char *lds_raw, uint32_t wave, uint32_t lane) {
    typedef const void __attribute__((address_space(1))) *gptr;
    typedef void __attribute__((address_space(3))) *lptr;
    const uint32_t n = (uint32_t)a.flat_rows16;
    const unsigned char *src = reinterpret_cast<const unsigned char *>(a.rows);
    for (uint32_t at = wave * 64u; at < n; at += BLOCK)
        if (at + lane < n) __builtin_amdgcn_global_load_lds((gptr)(src + (size_t)(at + lane) * 16u), (lptr)(lds_raw + at * 16u), 16, 0, 0);
}

// Windowed rows: the fetches of a wavefront without plans, in step with the loops of the others (see fetch_event of
// gen_score_loop_asm.py and setup_windowed_asm).  As many events as they have: every barrier is met.
__device__ __forceinline__ void many_fetch(const AceKernelArgs &a, unsigned char *lds_raw, uint32_t wave, uint32_t lane) {
    typedef const void __attribute__((address_space(1))) *gptr;
    typedef void __attribute__((address_space(3))) *lptr;
    for (int e = 0; e < a.n_fetch; ++e) {
        const ace_u4 *rec = a.win_dma + ((size_t)e * 16u + wave) * 5u;
        const ace_u4 head = rec[0];
        const unsigned char *rows = reinterpret_cast<const unsigned char *>(((uint64_t)head.w << 32) | head.z);
        const uint32_t n = (head.y >> 8) & 15u;
        const ace_u2 *load = reinterpret_cast<const ace_u2 *>(rec + 1);
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n s_barrier" ::: "memory");
        for (uint32_t k = 0; k < n; ++k) {
            const uint32_t from = (uint32_t)__builtin_amdgcn_readfirstlane((int)load[k].x), to = (uint32_t)__builtin_amdgcn_readfirstlane((int)load[k].y);
            __builtin_amdgcn_global_load_lds((gptr)(rows + from + lane * 16u), (lptr)(lds_raw + to), 16, 0, 0);
        }
        if (head.y & 1u) asm volatile("s_waitcnt vmcnt(0)\n s_barrier" ::: "memory");
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// One workgroup of 1,024 lanes.
template <bool WIN> __device__ __forceinline__ void ace_many_body(const AceKernelArgs &a, uint32_t slices, unsigned char *lds_raw, int tid, long long block) {
    constexpr int kLanes = 1024;
    const AceGeom &g = a.g;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(tid >> 6), lane = (uint32_t)tid & 63u;
    const uint32_t lanes = 64u * slices;
    if (!WIN) many_rows<kLanes>(a, lds_raw, wave, lane);
    // Deal: counting sort of the plans by pipeline depth, the deepest first (see ace_score_body), where the small tables go.
    // Sorted slice q goes to wavefront q in rows of four, every second row reversed: each SIMD gets the same mix.
    // (Windowed rows: the deeper its plans, the higher a wavefront's issue priority -- it has the most instructions to issue and
    // the others wait for it at every window.)
    unsigned int *cnt = reinterpret_cast<unsigned int *>(lds_raw + g.rk_lds_off);
    unsigned short *plan_of = reinterpret_cast<unsigned short *>(lds_raw + g.rk_lds_off + 128);
    const uint32_t q = (wave & 4u) ? wave ^ 3u : wave;
    if (tid < 32) cnt[tid] = 0u;
    const long long slot = block * lanes + tid;
    uint32_t depth = 0, rank = 0;                                   // (slots past the batch: last)
    if ((uint32_t)tid < lanes && slot < g.P) {
        depth = a.hdr[slot].x & 0xffu;
        depth = depth > 16u ? 16u : depth;
    }
    __syncthreads();
    if ((uint32_t)tid < lanes) rank = atomicAdd(&cnt[16u - depth], 1u);
    __syncthreads();
    if ((uint32_t)tid < lanes) {
        for (uint32_t b = 0; b < 16u - depth; ++b) rank += cnt[b];
        plan_of[rank] = (unsigned short)tid;
    }
    __syncthreads();
    const uint32_t at = (q << 6) | lane;
    const long long plan = block * lanes + (q < slices ? (uint32_t)plan_of[at] : 0u);
    __syncthreads();
    const bool in_batch = plan < g.P;
    const long long pl = in_batch ? plan : (long long)g.P - 1;      // plan this lane reads
    const long long out = a.order ? (long long)a.order[pl] : plan;
    const bool active = in_batch && out < g.P;
    const ace_u4 h = a.hdr[pl];
    const uint32_t first = a.codes[pl].x & 0x1fu;
    stage_small_tables<kLanes, true>(a, lds_raw, tid);
    if (!WIN && g.pace_lds_off && tid < 32) reinterpret_cast<uint32_t *>(lds_raw + g.pace_lds_off)[tid] = 0u;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                 // the rows
    __syncthreads();
    if (q >= slices) {
        if (WIN) many_fetch(a, lds_raw, wave, lane);
        return;
    }

    AceLds lds = ace_make_lds(lds_raw, 0u);
    lds.grows = reinterpret_cast<const unsigned char *>(a.rows);
    PlanState<false, false, true, false, WIN> st;
    st.init(g, lds, h, ace_u2{0u, 0u});
    st.row_ids = a.pos_types;
    if (!(first & 0x10u)) st.status = ACE_PLAN_MALFORMED;            // the first op must open a stage
    const uint32_t stride = lanes * (ACE_WS_REC * 8u), rec_off = at * (ACE_WS_REC * 8u);
    st.ws_stride = stride / 16u;
    double *rec_base = a.stage_ws + (size_t)block * ACE_MAX_STAGES * lanes * ACE_WS_REC;
    const int n_st = (int)ace_score_loop_asm<WIN>(a, g, st.glogs, g.lut2a_lds_off + st.bidx * 128u, (uint32_t)pl * 16u, rec_base, rec_off,
                                                  stride, 3u - (q >> 2), wave);
    if (WIN) {
        AceGeom gr = g;                                             // (row offsets as the rows lie in global memory)
        gr.row_bytes = (uint32_t)a.row_doubles * 8u;
        st.replay_all(gr, lds, rec_base + rec_off / 8u, n_st, first & 7u, a.pos_types[0] & 0xffu);
    } else
        st.replay_all(g, lds, rec_base + rec_off / 8u, n_st, first & 7u, a.pos_info[0] & 0xffu);
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
