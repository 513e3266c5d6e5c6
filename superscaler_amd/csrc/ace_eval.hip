// MI355X (gfx950) batched plan evaluator: kernels and C ABI (see include/ace_eval.h).
//
// Scoring, by the size of the batch (ace_route.h holds the rule):
//   ace_spread.h      small batches, and most batches of stage records and single-stage queries: a plan per workgroup, its ops
//                     over the lanes
//   ace_duo.h         mid-sized batches, every row resident: a plan walked by several lanes
//   ace_dense.h       large batches: a plan per lane, over tables in a denser form, rows resident or in windows
//   ace_many.h        large batches on tables that do not fit that form: a plan per lane
//   ace_score_loop.h  what these leave, in C++: a plan per lane
// With a plan per lane, all lanes of a workgroup walk the op sequence in lockstep, so the op type at each step is wave-uniform:
// the row of profiled values for that type sits in LDS at a scalar base address and each lane only adds its own (micro-batch,
// tp, algo) offset -- at most n_tp*n_algo distinct, consecutive entries per sub-table, i.e. LDS reads without bank conflicts.
// Plan bytes are stored plan-minor ([16-op group][plan][16 bytes]) so a wavefront's load covers 1 KiB of consecutive HBM.
// When the rows of all op types do not fit in LDS the op sequence is cut into windows, whose rows are staged in turn.
// Whatever the kernel, every plan's sums run sequentially in op order in fp64, which reproduces the reference's Python floats
// bit for bit.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstring>
#include <algorithm>
#include <mutex>
#include <new>
#include <vector>

#include "ace_edit_kernels.h"
#include "ace_grid.h"
#include "ace_keyset.h"
#include "ace_pack.h"
#include "ace_moves_host.h"
#include "ace_score_loop.h"
#include "ace_spread.h"
#include "ace_duo.h"
#include "ace_many.h"
#include "ace_dense.h"
#include "ace_route.h"
#include "ace_recompute.h"

// Scratch of ace_score_batch_static: the deferred-stage-tail records of up to ACE_STATIC_MAX_PLANS plans, in the layout of whichever kernel
// takes them (that of the dense tables is the largest).  Every GPU the library runs on holds
// its own copy of this array until the process ends.  In host code the array's name is only a stand-in for
// hipGetSymbolAddress(): kernels get the per-device pointer that call returned (static_scratch_ptr), never the name.
constexpr size_t kStaticBytes = (size_t)ACE_STATIC_MAX_PLANS * kDensePlan;
static_assert(kDensePlan >= kWsPlan, "the larger of the two");
static __device__ __align__(256) double scratch[kStaticBytes / sizeof(double)];

namespace {

#ifndef ACE_BLOCK
#define ACE_BLOCK 1024
#endif
constexpr int kBlock = ACE_BLOCK;        // lanes (= plans) per workgroup: 16 wavefronts, 4 per SIMD
constexpr int kSmallBlock = 256;         // ... for small batches: 4 wavefronts, 1 per SIMD
#ifndef ACE_SMALL_BATCH_BLOCKS
#define ACE_SMALL_BATCH_BLOCKS 128
#endif
constexpr int kSmallBatchBlocks = ACE_SMALL_BATCH_BLOCKS;   // batches of fewer than this many kBlock workgroups use kSmallBlock
constexpr uint32_t kMaxLds = 160 * 1024;  // CDNA4 LDS per workgroup
constexpr size_t kHostIoBytes = 1 << 20;  // page-locked buffers of ace_score_host, each way
static_assert(ACE_STATIC_MAX_PLANS % ACE_BLOCK == 0, "the static scratch holds whole workgroups");

thread_local char g_hip_err[256] = "";

constexpr int kMaxDevices = 64;
double *g_static_ptr[kMaxDevices];     // device address of `scratch` by device ordinal; filled once per device
std::mutex g_static_mutex;

// f() where host memory may run out (no exception leaves a C entry)
template <class F> static int or_enomem(F f) {
    try {
        return f();
    } catch (const std::bad_alloc &) {
        return ACE_ENOMEM;
    }
}

#define ACE_HIP(call)                                                                          \
    do {                                                                                       \
        hipError_t e_ = (call);                                                                \
        if (e_ != hipSuccess) {                                                                \
            snprintf(g_hip_err, sizeof(g_hip_err), "%s failed: %s", #call, hipGetErrorString(e_)); \
            return ACE_EHIP;                                                                   \
        }                                                                                      \
    } while (0)

// BD / RANGED / WIN / DEFER: see ace_score_body (ace_score_loop.h), which holds the whole kernel.
// BLOCK: kBlock lanes for large batches; kSmallBlock for batches that would otherwise occupy only a
// few CUs (a workgroup keeps a CU to itself either way: the tables fill its LDS): the walk over the
// op sequence is sequential per wavefront, so a small batch finishes soonest with one wavefront per
// SIMD on as many CUs as it can reach.
// COLL: tables compiled with consider_collective_memory (large workgroups only: a switch few callers set).
template <bool BD, bool RANGED, bool WIN, bool DEFER, int BLOCK, bool COLL = false>
__global__ __launch_bounds__(BLOCK) void ace_score_kernel(const AceKernelArgs a) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    ace_score_body<BD, RANGED, WIN, DEFER, BLOCK, COLL>(a, lds_raw, 0u, (int)threadIdx.x, (long long)blockIdx.x, gridDim.x);
}

// Small batches: a plan (or single-stage query) per workgroup, see ace_spread.h.
template <bool BD, bool RANGED, bool COLL>
__global__ __launch_bounds__(kSpreadLanes) void ace_spread_kernel(const AceKernelArgs a) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    ace_spread_body<BD, RANGED, COLL>(a, lds_raw, (int)threadIdx.x, (long long)blockIdx.x);
}
// Mid-sized batches: several lanes per plan, see ace_duo.h.
template <int L> __global__ __launch_bounds__(kDuoBlock) void ace_duo_kernel(const AceKernelArgs a, const AceDenseArgs d) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    ace_duo_body<L>(a, d, lds_raw, (int)threadIdx.x, (long long)blockIdx.x);
}
// Large batches on the assembly loop, see ace_many.h.
template <bool WIN> __global__ __launch_bounds__(1024) void ace_many_kernel(const AceKernelArgs a, const uint32_t slices) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    ace_many_body<WIN>(a, slices, lds_raw, (int)threadIdx.x, (long long)blockIdx.x);
}
// ... over dense tables, see ace_dense.h.
template <bool WIN, int LANES> __global__ __launch_bounds__(LANES, 4)
void ace_dense_kernel(const AceKernelArgs a, const AceDenseArgs d, const uint32_t slices) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    ace_dense_body<WIN, LANES>(a, d, slices, lds_raw, (int)threadIdx.x, (long long)blockIdx.x);
}
template <bool COLL> __global__ __launch_bounds__(kRcLanes, 6) void ace_rc_kernel(const RcArgs a, const long long first) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    ace_rc_body<COLL>(a, lds_raw, (int)threadIdx.x, first + (long long)blockIdx.x);
}

// ------------------------------------------------------------------------------------------
// top-k: radix select on the order-preserving 64-bit image of the iteration time, then a
// gather of everything below the k-th key plus the lowest-indexed ties, then a small sort.
// ------------------------------------------------------------------------------------------
constexpr int kTopBlock = 256;
constexpr int kRadixBits = 11;
constexpr int kRadix = 1 << kRadixBits;
constexpr int kPasses = 6;               // 6 * 11 = 66 >= 64 key bits
constexpr unsigned long long kInfKey = 0xffffffffffffffffull;

struct TopkState {                     // lives in the caller's workspace
    unsigned long long prefix;         // key bits fixed so far (from the top)
    unsigned long long thr;            // final k-th smallest key
    unsigned int k_rem;                // how many still to pick inside the current bucket
    unsigned int n_feasible;
    unsigned int n_less;               // entries with key < thr
    unsigned int n_out_less;           // atomic cursor for the gather of "< thr"
    unsigned int n_ties;               // atomic cursor for tie candidates
    unsigned int pad;
};

__device__ __forceinline__ unsigned long long time_key(double t, uint8_t feasible) {
    // positive doubles order like their bit patterns; infeasible or NaN plans sort last
    if (!feasible || !(t == t)) return kInfKey;
    if (t == 0.0) t = 0.0;          // (-0.0 compares equal to 0.0 in the reference's float order: one key for both)
    unsigned long long b = (unsigned long long)__double_as_longlong(t);
    return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}

__device__ __forceinline__ int pass_shift(int pass) {
    int s = 64 - kRadixBits * (pass + 1);
    return s < 0 ? 0 : s;
}
__device__ __forceinline__ int pass_bits(int pass) {
    int hi = 64 - kRadixBits * pass;
    int lo = pass_shift(pass);
    return hi - lo;
}

__global__ void topk_init(TopkState *st, unsigned int *hist, int k) {
    for (int j = threadIdx.x; j < kRadix; j += blockDim.x) hist[j] = 0;
    if (threadIdx.x == 0) {
        st->prefix = 0; st->thr = 0; st->k_rem = (unsigned)k; st->n_feasible = 0;
        st->n_less = 0; st->n_out_less = 0; st->n_ties = 0; st->pad = 0;
    }
}

__global__ __launch_bounds__(kTopBlock) void topk_hist(const double *t, const uint8_t *f, size_t n, int pass,
                                                       const TopkState *st, unsigned int *hist) {
    __shared__ unsigned int lh[kRadix];
    for (int j = threadIdx.x; j < kRadix; j += kTopBlock) lh[j] = 0;
    __syncthreads();
    const int shift = pass_shift(pass);
    const int bits = pass_bits(pass);
    const unsigned long long prefix = st->prefix;
    const int hi_shift = shift + bits;   // bits above this are already fixed
    for (size_t i = (size_t)blockIdx.x * kTopBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kTopBlock) {
        unsigned long long key = time_key(t[i], f[i]);
        bool match = hi_shift >= 64 ? true : ((key >> hi_shift) == (prefix >> hi_shift));
        if (match) atomicAdd(&lh[(unsigned)((key >> shift) & ((1ull << bits) - 1))], 1u);
    }
    __syncthreads();
    for (int j = threadIdx.x; j < kRadix; j += kTopBlock)
        if (lh[j]) atomicAdd(&hist[j], lh[j]);
}

__global__ __launch_bounds__(kTopBlock) void topk_pick(TopkState *st, unsigned int *hist, int pass) {
    // single workgroup: find the bucket holding the k_rem-th entry of the current prefix, descend into it
    constexpr int kPer = kRadix / kTopBlock;          // buckets per lane
    __shared__ unsigned int part[kTopBlock];
    const int tid = threadIdx.x;
    unsigned int loc[kPer];
    unsigned int sum = 0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) { loc[j] = hist[tid * kPer + j]; sum += loc[j]; }
    part[tid] = sum;
    __syncthreads();
    for (int off = 1; off < kTopBlock; off <<= 1) {   // inclusive scan of the per-lane sums
        unsigned int v = tid >= off ? part[tid - off] : 0u;
        __syncthreads();
        part[tid] += v;
        __syncthreads();
    }
    const unsigned int rem = st->k_rem;
    const unsigned int incl = part[tid], excl = incl - sum;
    const unsigned int total = part[kTopBlock - 1];
    const int shift = pass_shift(pass);
    __syncthreads();
    bool mine = excl < rem && rem <= incl;            // exactly one lane when total >= rem
    if (total < rem) mine = (tid == kTopBlock - 1);   // fewer entries than asked for: take the last bucket
    if (mine) {
        unsigned int acc = excl;
        int b = tid * kPer;
        if (total >= rem) {
            for (int j = 0; j < kPer; ++j) {
                if (acc + loc[j] >= rem) { b = tid * kPer + j; break; }
                acc += loc[j];
            }
        } else {
            const int nb = 1 << pass_bits(pass);
            b = nb - 1;
            acc = total - hist[b];
        }
        st->prefix |= ((unsigned long long)b) << shift;
        st->k_rem = rem - acc;
        st->n_less += acc;
        if (pass == kPasses - 1) st->thr = st->prefix;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kPer; ++j) hist[tid * kPer + j] = 0;
}

struct Cand { unsigned long long key; long long idx; };

__global__ __launch_bounds__(kTopBlock) void topk_gather(const double *t, const uint8_t *f, size_t n, TopkState *st,
                                                         Cand *less, Cand *ties, unsigned int cap_less, unsigned int cap_ties) {
    const unsigned long long thr = st->thr;
    for (size_t i = (size_t)blockIdx.x * kTopBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kTopBlock) {
        unsigned long long key = time_key(t[i], f[i]);
        if (key == kInfKey) continue;
        if (key < thr) {
            unsigned int p = atomicAdd(&st->n_out_less, 1u);
            if (p < cap_less) less[p] = Cand{key, (long long)i};
        } else if (key == thr) {
            unsigned int p = atomicAdd(&st->n_ties, 1u);
            if (p < cap_ties) ties[p] = Cand{key, (long long)i};
        }
    }
}

// When more ties than fit were seen, pick the lowest-indexed ones: one workgroup reads the input in index order, 8,192
// entries per step (512 consecutive ones per wavefront, the loads of the next step in flight), ranks the entries equal to
// the k-th key by wavefront ballots and one exchange of the wavefronts' counts through LDS, and stops as soon as it has
// enough.  Exact whatever the number of ties.
constexpr int kTieBlock = 1024;
__global__ __launch_bounds__(kTieBlock) void topk_ties_exact(const double *t, const uint8_t *f, size_t n, TopkState *st,
                                                             Cand *ties, unsigned int want) {
    constexpr int kCh = 8;                                      // a wavefront's share of a step: kCh * 64 consecutive entries
    constexpr size_t kStep = (size_t)kCh * kTieBlock;
    __shared__ unsigned int s_cnt[16];
    const unsigned long long thr = st->thr;
    // nothing to redo unless the gather overflowed its tie buffer (every lane reads the same value;
    // it is only rewritten after the last barrier below)
    if (st->n_ties <= want || thr == kInfKey) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const size_t mine = (size_t)wave * (kCh * 64) + (size_t)lane;   // entry c of this lane in a step: start + mine + c * 64
    unsigned int found = 0;
    // (the entries of the step after the current one are asked for before the current one is ranked)
    double nt[kCh];
    uint8_t nf[kCh];
#pragma unroll
    for (int c = 0; c < kCh; ++c) {
        const size_t i = mine + (size_t)c * 64;
        nt[c] = 0.0; nf[c] = 0;
        if (i < n) { nt[c] = t[i]; nf[c] = f[i]; }
    }
    for (size_t start = 0; start < n && found < want; start += kStep) {
        unsigned long long mask[kCh];
        unsigned int wave_total = 0;
#pragma unroll
        for (int c = 0; c < kCh; ++c) {
            const size_t i = start + mine + (size_t)c * 64;
            mask[c] = __ballot(i < n && time_key(nt[c], nf[c]) == thr);
            wave_total += (unsigned int)__popcll(mask[c]);
        }
#pragma unroll
        for (int c = 0; c < kCh; ++c) {
            const size_t i = start + kStep + mine + (size_t)c * 64;
            if (i < n) { nt[c] = t[i]; nf[c] = f[i]; }
        }
        if (lane == 0) s_cnt[wave] = wave_total;
        __syncthreads();
        unsigned int before = found, total = 0;
        for (int w = 0; w < 16; ++w) { const unsigned int v = s_cnt[w]; before += w < wave ? v : 0u; total += v; }
#pragma unroll
        for (int c = 0; c < kCh; ++c) {
            const unsigned int rank = before + (unsigned int)__popcll(mask[c] & ((1ull << lane) - 1ull));
            if (((mask[c] >> lane) & 1ull) && rank < want) ties[rank] = Cand{thr, (long long)(start + mine + (size_t)c * 64)};
            before += (unsigned int)__popcll(mask[c]);
        }
        found += total;                                        // (the same for every lane)
        __syncthreads();
    }
    if (tid == 0) st->n_ties = found < want ? found : want;
}

// Sort the candidates (key asc, index asc) in one workgroup (bitonic, in global memory for
// sizes beyond LDS) and write the first k.
__global__ __launch_bounds__(1024) void topk_finish(TopkState *st, Cand *less, Cand *ties, unsigned int cap_ties, int k,
                                                    Cand *buf, unsigned int buf_pow2, long long *out_idx, double *out_val,
                                                    int *out_count) {
    const unsigned int n_less = st->n_less;
    unsigned int n_ties = st->n_ties < cap_ties ? st->n_ties : cap_ties;
    const unsigned int total = n_less + n_ties;
    for (unsigned int j = threadIdx.x; j < buf_pow2; j += blockDim.x) {
        Cand c{kInfKey, 0x7fffffffffffffffll};
        if (j < n_less) c = less[j];
        else if (j < total) c = ties[j - n_less];
        buf[j] = c;
    }
    __syncthreads();
    for (unsigned int size = 2; size <= buf_pow2; size <<= 1) {
        for (unsigned int stride = size >> 1; stride > 0; stride >>= 1) {
            for (unsigned int j = threadIdx.x; j < buf_pow2; j += blockDim.x) {
                unsigned int partner = j ^ stride;
                if (partner > j) {
                    Cand x = buf[j], y = buf[partner];
                    bool up = (j & size) == 0;
                    bool gt = x.key > y.key || (x.key == y.key && x.idx > y.idx);
                    if (gt == up) { buf[j] = y; buf[partner] = x; }
                }
            }
            __syncthreads();
        }
    }
    unsigned int cnt = total < (unsigned)k ? total : (unsigned)k;
    for (unsigned int j = threadIdx.x; j < (unsigned)k; j += blockDim.x) {
        if (j < cnt) {
            Cand c = buf[j];
            unsigned long long b = c.key;
            b = (b >> 63) ? (b & 0x7fffffffffffffffull) : ~b;
            out_idx[j] = c.idx;
            out_val[j] = __longlong_as_double((long long)b);
        } else {
            out_idx[j] = -1;
            out_val[j] = __longlong_as_double(0x7ff0000000000000ll);
        }
    }
    if (threadIdx.x == 0 && out_count) *out_count = (int)cnt;
}

// ------------------------------------------------------------------------------------------
// top-k, short form (k <= 256): workgroups of 1,024 lanes select the k best of a stretch of the input each, one workgroup the
// k best of what they found (up to 16,384 entries: that workgroup alone).  A selection keeps its entries in registers.  Up to
// kBoundMaxK it bounds the k-th key by the best ones of the lanes and ranks what lies below (short_bound); where that is too much, and
// for larger k, it is a radix select on the 96-bit order (key, index) -- so ties fall to the lower index --, starting below the bits that
// all keys share, cut short as soon as the bucket that holds the k-th entry is small enough to be ranked as it is.  Exact for any
// input, whatever its order and however many keys are equal: no list that overflows is used.
// Bound by the latency of the two selections -- their own code's way into the instruction cache, a trip to memory, the barriers --, not
// by reading the input.  Kernel trace behind the scoring kernel, us, radix select alone -> with the bound, k = 64: 4,096 entries
// 9.1 -> 6.0; 65,536 entries 9.3 + 7.3 -> 6.7 + 4.6; 262,144 entries 8.6 + 8.9 -> 6.8 + 5.6; 2^20 entries 16.0 + 16.6 -> 11.4 + 8.5; k = 1,
// 8,192 entries 9.8 -> 4.8.  Where the times spread over more powers of two (lognormal), a call, us: k = 64, 262,144 entries 37 -> 15, k = 160
// 50 -> 34.
// ------------------------------------------------------------------------------------------
constexpr int kShortMaxK = 256;
constexpr unsigned kShortMaxEntries = 16384;     // entries one workgroup selects from: sixteen per lane
constexpr unsigned kShortBucket = 512;           // bucket entries that fit the histogram's LDS as (key, index) pairs

// Which of the kRadix buckets of `hist` (LDS) holds the rem-th entry (1-based), counting buckets in order: returns the
// bucket, the entries before it in `before` and the total in `total` to every lane of the 1024-lane workgroup (no bucket:
// total < rem, and the return value is meaningless).  Two buckets per lane, wavefront scans, one exchange through LDS.
__device__ __forceinline__ unsigned int short_pick(const unsigned int *hist, unsigned int rem, unsigned int *wsum /* [16 + 3] */,
                                                   unsigned int &before, unsigned int &total) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const unsigned int h0 = hist[2 * tid], h1 = hist[2 * tid + 1];
    unsigned int incl = h0 + h1;
    for (int off = 1; off < 64; off <<= 1) {
        const unsigned int v = __shfl_up(incl, off, 64);
        if (lane >= off) incl += v;
    }
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    unsigned int base = 0, all = 0;
    for (int w2 = 0; w2 < 16; ++w2) {
        const unsigned int v = wsum[w2];
        if (w2 < wave) base += v;
        all += v;
    }
    incl += base;
    const unsigned int excl = incl - (h0 + h1);
    if (all >= rem && excl < rem && rem <= incl) {       // exactly one lane
        const bool second = excl + h0 < rem;
        wsum[16] = 2 * tid + (second ? 1 : 0);
        wsum[17] = excl + (second ? h0 : 0u);
    }
    __syncthreads();
    const unsigned int bucket = wsum[16];
    before = wsum[17];
    total = all;
    __syncthreads();                                       // (wsum is reused by the next call)
    return bucket;
}

// Rank in (key, index) order of entry tid / parts of `list` (LDS, cnt <= 1,024 / parts entries) for every entry at once:
// `parts` neighbouring lanes compare an entry with a part of the others each; every one of them gets the rank.
template <int parts> __device__ __forceinline__ unsigned int short_rank(const Cand *list, unsigned int cnt, Cand &me) {
    const unsigned int i = threadIdx.x / parts, part = threadIdx.x % parts;
    me = list[i < cnt ? i : 0u];
    unsigned int rank = 0;
#pragma unroll 8
    for (unsigned int j = part; j < cnt; j += parts) {
        const Cand o = list[j];
        rank += o.key < me.key || (o.key == me.key && o.idx < me.idx) ? 1u : 0u;
    }
#pragma unroll
    for (int off = 1; off < parts; off <<= 1) rank += __shfl_xor(rank, off, 64);
    return i < cnt ? rank : ~0u;
}

struct ShortShared {
    union {
        unsigned int hist[kRadix];
        Cand bucket[kShortBucket];               // after the passes
    };
    Cand win[kShortMaxK];
    __align__(16) unsigned int mins[256];        // short_bound
    unsigned int wsum[20];
    unsigned long long wref[16];
    unsigned int nfin, cur, nwin, nbucket, bound;
};

// Few entries that hold the k smallest (k <= kBoundMaxK) of the workgroup's, into s.bucket in no order; returns how many (more than
// kShortBucket: too many, s.bucket is not filled).  Every four neighbouring lanes give the smallest of their entries' leading 32 bits; the
// k-th smallest of these 256 bounds the k-th key, and what lies at or below it is taken: of random keys in random order some
// 256 ln(256 / (256 - k)).  That is 251 for k = 160, and ranking them costs their square: a call for 4,096 / 262,144 entries takes
// 15 / 34 us there (radix select: 26 / 47), with k = 200 29 / 60 (27 / 48).
// What a selection of 4,096 entries waits for is its own code, run once: some 250 cycles for every 64 bytes of it.  So this is
// short and has three barriers; the radix selection below takes what it cannot (many equal keys, the best ones all together).
constexpr int kBoundMaxK = 160;
template <int kPer>
__device__ __forceinline__ unsigned int short_bound(ShortShared &s, const unsigned long long (&rk)[kPer], const unsigned int (&ri)[kPer], int k) {
    const unsigned int tid = threadIdx.x;
    unsigned int mn = ~0u;
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        const unsigned int h = (unsigned int)(rk[q] >> 32);
        mn = h < mn ? h : mn;
    }
    unsigned int o = (unsigned int)__builtin_amdgcn_mov_dpp((int)mn, 0xb1, 0xf, 0xf, true);      // (lane ^ 1)
    mn = o < mn ? o : mn;
    o = (unsigned int)__builtin_amdgcn_mov_dpp((int)mn, 0x4e, 0xf, 0xf, true);                   // (lane ^ 2)
    mn = o < mn ? o : mn;
    if (!(tid & 3u)) s.mins[tid >> 2] = mn;
    if (tid == 0) { s.nbucket = 0; s.bound = 0; }
    __syncthreads();
    unsigned int rank = 0;
    const ace_u4 *m = reinterpret_cast<const ace_u4 *>(s.mins) + (tid & 3u);
#pragma unroll 4
    for (unsigned int j = 0; j < 64u; j += 4u) {
        const ace_u4 v = m[j];
        rank += (v.x < mn ? 1u : 0u) + (v.y < mn ? 1u : 0u) + (v.z < mn ? 1u : 0u) + (v.w < mn ? 1u : 0u);
    }
    rank += (unsigned int)__builtin_amdgcn_mov_dpp((int)rank, 0xb1, 0xf, 0xf, true);
    rank += (unsigned int)__builtin_amdgcn_mov_dpp((int)rank, 0x4e, 0xf, 0xf, true);
    if (!(tid & 3u) && rank < (unsigned int)k) atomicMax(&s.bound, mn);
    __syncthreads();
    const unsigned int bound = s.bound;
#pragma unroll
    for (int q = 0; q < kPer; ++q)
        if ((unsigned int)(rk[q] >> 32) <= bound && rk[q] != kInfKey) {
            const unsigned int p = atomicAdd(&s.nbucket, 1u);
            if (p < kShortBucket) s.bucket[p] = Cand{rk[q], (long long)ri[q]};
        }
    __syncthreads();
    const unsigned int cnt = s.nbucket;
    if (cnt > kShortBucket) __syncthreads();                   // (read by all before the radix selection clears it)
    return cnt;
}

// `take(rank, entry)` for every entry of `list` (LDS, cnt <= 512 entries): as many neighbouring lanes compare an entry with a part of the
// others each as there are lanes for it (at most sixteen).
template <class Take> __device__ __forceinline__ void short_ranked(const Cand *list, unsigned int cnt, Take take) {
    const unsigned int shift = cnt <= 64u ? 4u : cnt <= 128u ? 3u : cnt <= 256u ? 2u : 1u, parts = 1u << shift;
    const unsigned int i = threadIdx.x >> shift;
    if (i >= cnt) return;
    const Cand me = list[i];
    unsigned int rank = 0;
#pragma unroll 2
    for (unsigned int j = threadIdx.x & (parts - 1u); j < cnt; j += parts) {
        const Cand o = list[j];
        rank += o.key < me.key || (o.key == me.key && o.idx < me.idx) ? 1u : 0u;
    }
#pragma unroll 1
    for (unsigned int off = 1; off < parts; off <<= 1) rank += __shfl_xor(rank, off, 64);
    if (!(threadIdx.x & (parts - 1u))) take(rank, me);
}

// The k smallest of the workgroup's entries (kPer per lane; kInfKey: none) in (key, index) order, into s.win in no order;
// returns how many there are (k, or all of them).
template <int kPer>
__device__ __forceinline__ unsigned int short_select(ShortShared &s, const unsigned long long (&rk)[kPer], const unsigned int (&ri)[kPer], int k) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid == 0) { s.nfin = 0; s.cur = 0; s.nwin = 0; s.nbucket = 0; }
    // how many keys there are, and which bits vary among them: the highest bit in which any key differs from one of
    // them (the first one in lane order), one 32-bit maximum over the workgroup
    unsigned long long mine = kInfKey;
    unsigned int wave_cnt = 0;
#pragma unroll
    for (int q = kPer - 1; q >= 0; --q) {
        const bool fin = rk[q] != kInfKey;
        if (fin) mine = rk[q];
        wave_cnt += (unsigned int)__popcll(__ballot(fin));
    }
    const unsigned long long has = __ballot(mine != kInfKey);
    const unsigned long long wave_ref = __shfl(mine, has ? __ffsll((long long)has) - 1 : 0, 64);
    __syncthreads();                                           // (the counters are zero)
    if (lane == 0) {
        s.wref[wave] = wave_ref;
        if (wave_cnt) atomicAdd(&s.nfin, wave_cnt);
    }
    __syncthreads();
    const unsigned int nfin = s.nfin;
    const bool all = nfin <= (unsigned)k;
    int cur = 0, icur = 32, small_shift = 0;
    unsigned long long prefix = 0;
    unsigned int iprefix = 0, rem = (unsigned)k;
    bool small = false;
    if (!all) {
        unsigned long long ref = kInfKey;
        for (int w2 = 15; w2 >= 0; --w2) {
            const unsigned long long v = s.wref[w2];
            if (v != kInfKey) ref = v;
        }
        int hb = 0;
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            const unsigned long long x = rk[q] == kInfKey ? 0ull : rk[q] ^ ref;
            const int b = x ? 64 - __clzll((long long)x) : 0;
            hb = b > hb ? b : hb;
        }
        for (int off = 32; off > 0; off >>= 1) {
            const int o = __shfl_xor(hb, off, 64);
            hb = o > hb ? o : hb;
        }
        if (lane == 0 && hb) atomicMax(&s.cur, (unsigned int)hb);
        __syncthreads();
        cur = (int)s.cur;                                      // the low `cur` key bits vary
        prefix = cur >= 64 ? 0ull : (ref >> cur) << cur;
        // key digits from the highest varying bit down, then index digits among the entries with the selected key
        while (!small && (cur > 0 || icur > 0)) {
            for (int j = tid; j < kRadix; j += 1024) s.hist[j] = 0;
            __syncthreads();
            const bool on_key = cur > 0;
            const int top = on_key ? cur : icur;
            const int bits = top < kRadixBits ? top : kRadixBits, shift = top - bits;
#pragma unroll
            for (int q = 0; q < kPer; ++q) {
                const unsigned long long key = rk[q];
                if (key == kInfKey) continue;
                if (on_key) {
                    if (cur >= 64 || (key >> cur) == (prefix >> cur))
                        atomicAdd(&s.hist[(unsigned)((key >> shift) & ((1ull << bits) - 1ull))], 1u);
                } else if (key == prefix) {
                    if (icur >= 32 || (ri[q] >> icur) == (iprefix >> icur)) atomicAdd(&s.hist[(ri[q] >> shift) & ((1u << bits) - 1u)], 1u);
                }
            }
            __syncthreads();
            unsigned int before, total;
            const unsigned int b = short_pick(s.hist, rem, s.wsum, before, total);
            (void)total;
            rem -= before;
            if (on_key) {
                prefix |= (unsigned long long)b << shift;
                cur = shift;
                if (s.hist[b] <= kShortBucket) { small = true; small_shift = shift; }
            } else {
                iprefix |= b << shift;
                icur = shift;
            }
            __syncthreads();                                   // (hist[b] read by all before the next pass clears it)
        }
    }
    // gather the winners (the bucket's entries go where the histogram was)
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        const unsigned long long key = rk[q];
        if (key == kInfKey) continue;
        bool wins = true;
        if (small) {
            // the key bits from small_shift up are fixed: below the bucket -> a winner; in it -> ranked below
            const unsigned long long hk = key >> small_shift, hp = prefix >> small_shift;
            wins = hk < hp;
            if (hk == hp) {
                const unsigned int p = atomicAdd(&s.nbucket, 1u);
                if (p < kShortBucket) s.bucket[p] = Cand{key, (long long)ri[q]};
            }
        } else if (!all) wins = key < prefix || (key == prefix && ri[q] <= iprefix);
        if (wins) {
            const unsigned int p = atomicAdd(&s.nwin, 1u);
            if (p < (unsigned)kShortMaxK) s.win[p] = Cand{key, (long long)ri[q]};
        }
    }
    __syncthreads();
    unsigned int nwin = s.nwin;
    if (small) {
        // the `rem` smallest (key, index) of the bucket join the winners, each at its rank
        const unsigned int nb = s.nbucket < kShortBucket ? s.nbucket : kShortBucket;
        static_assert(kShortBucket * 2 <= 1024, "two lanes per entry");
        Cand me;
        const unsigned int rank = short_rank<2>(s.bucket, nb, me);
        if (!(tid & 1) && rank < rem && nwin + rank < (unsigned)kShortMaxK) s.win[nwin + rank] = me;
        nwin += rem;
        __syncthreads();
    }
    return nwin < (unsigned)k ? nwin : (unsigned)k;
}

// The k best of each stretch of 1,024 * kPer entries: cand[k * workgroup ...], kInfKey behind the last one.
template <int kPer>
__global__ __launch_bounds__(1024) void topk_local(const double *t, const uint8_t *f, size_t n, int k, int spread, Cand *cand) {
    __shared__ ShortShared s;
    unsigned long long rk[kPer];
    unsigned int ri[kPer];
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        const size_t i = ((size_t)blockIdx.x * kPer + q) * 1024 + threadIdx.x;
        rk[q] = i < n ? time_key(t[i], f[i]) : kInfKey;
        ri[q] = (unsigned int)i;
    }
    if (k <= kBoundMaxK) {
        const unsigned int cnt = short_bound<kPer>(s, rk, ri, k);
        if (cnt <= kShortBucket) {
            // (where short_bound of the last launch, 2^spread entries per lane, finds the best ones of all stretches with different
            // four lanes: its bound is close then.  In the order of their ranks it let 256 of 1,024 entries through for k = 64)
            Cand *out = cand + (size_t)blockIdx.x * k;
            if (cnt < (unsigned)k) {
                for (unsigned int j = threadIdx.x; j < (unsigned)k; j += 1024) out[j] = Cand{kInfKey, 0x7fffffffffffffffll};
                __syncthreads();
            }
            const unsigned int A = (unsigned)k >> 2, rot = ((blockIdx.x * (unsigned)k >> 10) * A) >> spread;
            short_ranked(s.bucket, cnt, [&](unsigned int rank, const Cand &c) {
                if (rank >= (unsigned)k) return;
                unsigned int slot = rank;
                if (rank < 4u * A) {
                    const unsigned int b = (rank >= A ? 1u : 0u) + (rank >= 2u * A ? 1u : 0u) + (rank >= 3u * A ? 1u : 0u);
                    unsigned int at = rank - b * A + rot;
                    if (at >= A) at -= A;
                    slot = 4u * at + b;
                }
                out[slot] = c;
            });
            return;
        }
    }
    const unsigned int nwin = short_select<kPer>(s, rk, ri, k);
    for (unsigned int j = threadIdx.x; j < (unsigned)k; j += 1024)
        cand[(size_t)blockIdx.x * k + j] = j < nwin ? s.win[j] : Cand{kInfKey, 0x7fffffffffffffffll};
}

// The k best of all: of the input itself (cand == nullptr) or of the m entries that topk_local left.
template <int kPer>
__global__ __launch_bounds__(1024) void topk_final(const double *t, const uint8_t *f, const Cand *cand, unsigned int m, int k,
                                                   long long *out_idx, double *out_val, int *out_count) {
    __shared__ ShortShared s;
    const int tid = threadIdx.x;
    unsigned long long rk[kPer];
    unsigned int ri[kPer];
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        const unsigned int i = (unsigned int)q * 1024u + (unsigned int)tid;
        rk[q] = kInfKey;
        ri[q] = i;
        if (i < m) {
            if (cand) {
                const Cand c = cand[i];
                rk[q] = c.key;
                ri[q] = (unsigned int)c.idx;
            } else
                rk[q] = time_key(t[i], f[i]);
        }
    }
    const Cand *list = s.bucket;
    unsigned int cnt = k <= kBoundMaxK ? short_bound<kPer>(s, rk, ri, k) : ~0u;
    if (cnt > kShortBucket) {
        cnt = short_select<kPer>(s, rk, ri, k);
        list = s.win;
    }
    // the winners in ascending (key, index) order
    short_ranked(list, cnt, [&](unsigned int rank, const Cand &c) {
        if (rank >= (unsigned)k) return;
        unsigned long long b = c.key;
        b = (b >> 63) ? (b & 0x7fffffffffffffffull) : ~b;
        out_idx[rank] = c.idx;
        out_val[rank] = __longlong_as_double((long long)b);
    });
    const unsigned int found = cnt < (unsigned)k ? cnt : (unsigned)k;
    for (unsigned j = found + tid; j < (unsigned)k; j += 1024) {
        out_idx[j] = -1;
        out_val[j] = __longlong_as_double(0x7ff0000000000000ll);
    }
    if (tid == 0 && out_count) *out_count = (int)found;
}

// Entries per workgroup of topk_local for n entries (0: topk_final alone): short stretches while the selection from what they
// leave stays short too (4,096 entries), longer ones while it fits one workgroup, or none at all (~0u).
unsigned int short_stretch(size_t n, int k) {
    if (k > kShortMaxK || n > 0xffffffffull) return ~0u;
    if (n <= kShortMaxEntries) return 0;
    const auto found = [&](size_t per) { return (n + per - 1) / per * (size_t)k; };
    if (found(4096) <= 4096) return 4096;
    if (found(8192) <= kShortMaxEntries) return 8192;
    if (found(16384) <= kShortMaxEntries) return 16384;
    return ~0u;
}

unsigned int next_pow2(unsigned int v) {
    unsigned int p = 1;
    while (p < v) p <<= 1;
    return p;
}

}  // namespace

struct ace_handle {
    int device;
    AceGeom geom;
    int32_t n_windows, row_doubles, rk_bytes, stg_words, num_types;
    uint32_t lds_bytes;
    // device copies
    double *d_rows;
    uint32_t *d_pos_info;
    ace_u2 *d_pos_spread;      // per position, for the kernel of small batches (null: more ops than it takes)
    uint32_t *d_pos_types;     // d_pos_info with row indices in place of LDS slots (windowed rows, at most 256 of them; else null)
    ace_u4 *d_pos4;            // per position, for the assembly op loop (null when its pair-kind table has no room in LDS)
    int32_t n_fetch;           // fetch events of d_win_dma
    ace_u4 *d_win_dma;         // windowed rows: what the assembly op loop fetches its windows by (setup_windowed_asm), or null
    AceGeom geom_wa;           // ... and the LDS layout of the kernel that runs it
    uint32_t lds_bytes_wa;
    AceDenseArgs dense;        // tables of ace_dense.h (device addresses; image null: they do not fit that form)
    uint32_t dense_lds;
    int dense_lanes;           // of a workgroup of large batches
    unsigned char *d_dense_rows;   // ... windowed: the rows
    uint8_t *d_pair_kinds;
    uint32_t *d_stage_lut;
    double *d_nbm1;
    int32_t *d_win_pos, *d_win_row_begin;
    uint32_t *d_win_rows;
    int32_t flat_rows16;       // see AceKernelArgs
    ace_u2 *d_rc_pos;          // check_recompute's tables (ace_recompute_prepare), or null
    int32_t rc_groups, rc_waves;   // ... see RcArgs
    double *d_rc_act;
    unsigned char *host_in, *host_out;   // page-locked buffers of ace_score_host (null until the first call)
    struct StepBuffers *step;  // of ace_search_step (null until the first call)
    double *d_stage_ws;        // grow-only workspace for deferred stage tails
    size_t stage_ws_plans, stage_ws_bytes;     // the most plans it was asked for, its size
    AceRouteTables route;      // what the tables allow (ace_route.h)
    int stage_ws_fixed;        // ace_reserve(..., fixed): a larger batch is an error instead of a reallocation
    std::mutex host_calls;     // held by ace_score_host and ace_search_step from their first to their last use of host_in, host_out and
                               // step: the next call, of another thread, must find the transfers of the one before ended
    std::mutex workspace;      // held from the look at d_stage_ws to the launch that uses it: another thread's larger batch replaces it
};

struct StepOut { long long idx; double iter_ms, peak_mb; int32_t count; };
struct StepBuffers {
    std::vector<uint8_t> t_codes;
    std::vector<uint32_t> t_hdr;
    unsigned char *host, *dev;          // page-locked: StepOut, then what goes up; both grow only
    size_t host_bytes, dev_bytes;
};
__global__ void step_out_kernel(const long long *idx, const double *val, const int32_t *count, const double *peak, StepOut *out) {
    const int32_t n = *count;
    *out = StepOut{*idx, *val, n > 0 ? peak[*idx] : 0.0, n};
}

// The bodies of these kernels live in ace_edit_kernels.h (shared with the host build of the tests).
__global__ __launch_bounds__(256) void apply_moves_kernel(const ace_u4 *tmpl_codes, const ace_u4 *tmpl_hdr, int n_templates,
                                                          const ace_u4 *moves, unsigned long long n, int G, int a_shift,
                                                          ace_u4 *codes_out, ace_u4 *hdr_out, unsigned long long *key_out, unsigned long long first) {
    apply_moves_body((first + blockIdx.x) * 256 + threadIdx.x, tmpl_codes, tmpl_hdr, n_templates, moves, n, G, a_shift,
                     codes_out, hdr_out, key_out);
}

__global__ __launch_bounds__(256) void group_keys_kernel(const ace_u4 *codes, const ace_u4 *hdr, unsigned long long n, int G, int N,
                                                         unsigned long long *keys) {
    group_keys_body((unsigned long long)blockIdx.x * 256 + threadIdx.x, codes, hdr, n, G, N, keys);
}

__global__ __launch_bounds__(256) void gather_plans_kernel(const ace_u4 *codes_in, const ace_u4 *hdr_in, const uint32_t *perm,
                                                           unsigned long long n, int G, ace_u4 *codes_out, ace_u4 *hdr_out, unsigned long long first) {
    gather_plans_body((first + blockIdx.x) * 256 + threadIdx.x, codes_in, hdr_in, perm, n, G, codes_out, hdr_out);
}

__global__ __launch_bounds__(kPackLanes, 4) void pack_plans_kernel(const PackArgs a, const long long first) {
    __shared__ PackShared s;
    ace_pack_body(a, s, (int)threadIdx.x, first + (long long)blockIdx.x);
}

__global__ __launch_bounds__(kPackLanes) void unpack_plans_kernel(const PackArgs a, const long long first) {
    __shared__ PackShared s;
    ace_unpack_body(a, s, (int)threadIdx.x, first + (long long)blockIdx.x);
}

__global__ void rc_groups_kernel(RcTables t, int n, const int32_t *q_plan, const int32_t *q_lo, const int32_t *q_hi,
                                 const int32_t *q_nsb, const uint32_t *q_mrow, double *sum_size, int32_t *first_pos,
                                 int32_t *bad) {
    rc_groups_body((int)(blockIdx.x * blockDim.x + threadIdx.x), t, n, q_plan, q_lo, q_hi, q_nsb, q_mrow, sum_size, first_pos, bad);
}

__global__ void rc_select_kernel(RcTables t, uint8_t *codes_rw, int n, const int32_t *q_plan, const int32_t *q_lo,
                                 const int32_t *q_hi, const int32_t *q_nsb, const uint32_t *q_mrow, const double *sum_size,
                                 const int32_t *first_pos, uint8_t *recomputed, const double *mem, double memory_limit,
                                 uint8_t *alive) {
    rc_select_body((int)(blockIdx.x * blockDim.x + threadIdx.x), t, codes_rw, n, q_plan, q_lo, q_hi, q_nsb, q_mrow, sum_size,
                   first_pos, recomputed, mem, memory_limit, alive);
}

extern "C" {

int ace_abi_version(void) { return ACE_ABI_VERSION; }

const char *ace_strerror(int code) {
    switch (code) {
        case ACE_OK: return "ok";
        case ACE_EINVAL: return "invalid argument";
        case ACE_ETOOBIG: return "table row larger than LDS";
        case ACE_EHIP: return "HIP runtime error";
        case ACE_ENOMEM: return "out of memory";
        case ACE_EVERSION: return "ABI version mismatch";
        case ACE_EFIXED: return "the batch needs a larger workspace than the one fixed with ace_reserve";
        default: return "unknown error";
    }
}

const char *ace_last_hip_error(void) { return g_hip_err; }

static int upload(void **dst, const void *src, size_t bytes, size_t alloc_bytes = 0) {
    *dst = nullptr;
    if (alloc_bytes < bytes) alloc_bytes = bytes;
    if (alloc_bytes == 0) alloc_bytes = 16;
    ACE_HIP(hipMalloc(dst, alloc_bytes));
    if (alloc_bytes > bytes) ACE_HIP(hipMemset(*dst, 0, alloc_bytes));
    if (src && bytes) ACE_HIP(hipMemcpy(*dst, src, bytes, hipMemcpyHostToDevice));
    return ACE_OK;
}

}  // extern "C"

template <bool BD, bool RANGED, bool WIN, bool DEFER> static int allow_big_lds() {
    ACE_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&ace_score_kernel<BD, RANGED, WIN, DEFER, kBlock>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxLds));
    ACE_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&ace_score_kernel<BD, RANGED, WIN, DEFER, kSmallBlock>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxLds));
    if (!DEFER)
        ACE_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&ace_score_kernel<BD, RANGED, WIN, false, kBlock, true>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxLds));
    return ACE_OK;
}

static int allow_duo_lds() {
    ACE_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&ace_duo_kernel<64>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxLds));
    ACE_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&ace_duo_kernel<128>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxLds));
    ACE_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&ace_duo_kernel<256>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxLds));
    return ACE_OK;
}

template <bool WIN> static int allow_many_lds() {
    ACE_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&ace_many_kernel<WIN>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxLds));
    return ACE_OK;
}

static int allow_dense_lds() {
    ACE_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&ace_dense_kernel<false, kDenseLanes>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kDenseLds));
    ACE_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&ace_dense_kernel<false, kDenseWinLanes>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kDenseWinLds));
    ACE_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&ace_dense_kernel<true, kDenseWinLanes>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kDenseWinLds));
    return ACE_OK;
}

// Per op position, what the assembly form of the op loop (ace_score_loop_asm.inc) reads with scalar loads: the LDS
// address of the position's row at its hot sub-table and at its collective-cost tables, the LDS address of the
// 32-bit pair-kind block of the (this op, next op) pair, and two flags (bit 0: the rule "ordinary op followed by a layer
// start" does NOT apply here, bit 1: ordinary op).  Positions past the last op point at row 0 and pair kind 0.
static int upload_pos4(ace_handle *h, const ace_tables_t *t, size_t pos_entries, uint32_t pk32_off) {
    h->d_pos4 = nullptr;
    if (!pk32_off || t->n_windows != 1) return ACE_OK;       // (windowed rows: setup_windowed_asm)
    ace_u4 *p4 = new (std::nothrow) ace_u4[pos_entries];
    if (!p4) return ACE_ENOMEM;
    const uint32_t row_bytes = (uint32_t)t->row_doubles * 8u, kind_stride = (uint32_t)t->n_glog * ACE_PK32_BLOCK;   // (words of the 32-bit table per pair kind)
    for (size_t i = 0; i < pos_entries; ++i) {
        const uint32_t info = i < (size_t)t->num_ops ? t->pos_info[i] : 0u;
        const uint32_t row = (info & 0xffu) * row_bytes;
        p4[i].x = row + (uint32_t)t->hot_off * 8u;
        p4[i].y = row + (uint32_t)t->z_off * 8u;
        p4[i].z = pk32_off + ((info >> 16) & 0xffu) * kind_stride * 4u;
        // (rows as the evaluation of the stage tails indexes them: LDS slots)
        const uint32_t ids = info & 0xffffu;
        p4[i].w = (((info >> 24) & 1u) ^ 1u) | (((info >> 25) & 1u) << 1) | (ids << 8);
    }
    const int rc = upload((void **)&h->d_pos4, p4, pos_entries * sizeof(ace_u4));
    delete[] p4;
    return rc;
}

static int upload_pos_spread(ace_handle *h, const ace_tables_t *t, size_t pos_entries) {
    h->d_pos_spread = nullptr;
    if (t->num_ops > kSpreadMaxOps || (uint64_t)t->num_types * (uint64_t)t->row_doubles * 8u > 0xffffffffull) return ACE_OK;
    std::vector<ace_u2> ps(pos_entries);
    ace_pos_spread(t, ps.data(), pos_entries);
    return upload((void **)&h->d_pos_spread, ps.data(), pos_entries * sizeof(ace_u2));
}

// Windowed rows: the position descriptors with each row's index in `rows` where its LDS slot is.
static int upload_pos_types(ace_handle *h, const ace_tables_t *t, size_t pos_entries) {
    h->d_pos_types = nullptr;
    if (t->n_windows <= 1 || t->num_types > 256) return ACE_OK;
    uint32_t *pt = new (std::nothrow) uint32_t[pos_entries];
    if (!pt) return ACE_ENOMEM;
    ace_pos_types(t, pt, pos_entries);
    const int rc = upload((void **)&h->d_pos_types, pt, pos_entries * 4);
    delete[] pt;
    return rc;
}

// Windowed rows, for the assembly op loop.  That loop reads only the hot sub-table and the collective-cost tables of a
// row (the boundary sub-tables are read from global memory when the stage tails are evaluated), so it keeps its own,
// denser windows: per row those two parts back to back, consecutive windows in alternate halves of the region in front of
// the small tables, so that a window is fetched while the one before it is walked.  Built here: the LDS layout
// (h->geom_wa), the per-position table (h->d_pos4) and the fetch records (h->d_win_dma): per fetch event and wavefront
// (sixteen) 80 bytes = {first position of the window after the one being entered, bit 0: wait for the fetch (else it
// completes before the next event) | number of loads << 8, address of the rows} and eight LDS-direct loads {byte offset
// in the rows, LDS address} of 1 KB each.  Events: 0 fetches window 0 and waits, 1 fetches window 1, and entering window
// w >= 1 fetches window w + 1 (the last one fetches window w - 1 again, into the half nobody reads).
// Leaves the handle without them (plain scoring then takes the C++ loop) where the layout does not work out.
static int setup_windowed_asm(ace_handle *h, const ace_tables_t *t, size_t pos_entries, int32_t rk_bytes, int32_t stg_words) {
    h->d_win_dma = nullptr;
    if (t->n_windows <= 1 || !h->d_pos_types || (t->flags & ACE_F_COLLECTIVE_MEM) || t->num_ops >= 32768) return ACE_OK;
    if ((int64_t)(t->n_z > 0 ? t->n_z : 1) * t->z_table_doubles * 8 > 65536) return ACE_OK;
    const uint64_t row_bytes = (uint64_t)t->row_doubles * 8u;
    if ((uint64_t)t->num_types * row_bytes > 0xffffffffull) return ACE_OK;
    if (!(t->hot_off < t->start_off && t->start_off <= t->z_off && t->z_off <= t->row_doubles)) return ACE_OK;
    const uint32_t hot_len = (uint32_t)(t->start_off - t->hot_off) * 8u, z_len = (uint32_t)(t->row_doubles - t->z_off) * 8u;
    if (hot_len < 1024u || (z_len != 0u && z_len < 1024u) || (hot_len & 15u) || (z_len & 15u)) return ACE_OK;
    const uint32_t crow = hot_len + z_len;
    // the most rows per half that leave room for the small tables
    uint32_t slots = 127, stg_off = 0, lut2_off = 0, pk32_off = 0, lut2a_off = 0, lds_end = 0;
    for (; slots >= 5u; --slots) {
        lut2a_off = (ace_lds_pk32(ace_lds_layout(2u * slots * crow, (uint32_t)rk_bytes, (uint32_t)stg_words, &stg_off, &lut2_off),
                                  (uint32_t)rk_bytes, &pk32_off) + 15u) & ~15u;
        lds_end = lut2a_off + (uint32_t)stg_words * 8u;
        if (lds_end <= kMaxLds) break;
    }
    if (slots < 5u) return ACE_OK;
    const int N = t->num_ops;
    std::vector<uint32_t> types(pos_entries);
    ace_pos_types(t, types.data(), pos_entries);
    // windows end at multiples of 4 ops (or at the last op) and hold at most `slots` different rows
    std::vector<int> win_start;
    std::vector<std::vector<uint32_t>> win_types;
    for (int i = 0; i < N;) {
        std::vector<uint32_t> seen;
        int good = -1;
        size_t good_n = 0;
        for (int j = i; j < N;) {
            const uint32_t ty = types[j] & 0xffu;
            if (std::find(seen.begin(), seen.end(), ty) == seen.end()) {
                if (seen.size() >= slots) break;
                seen.push_back(ty);
            }
            ++j;
            if (j == N || (j & 3) == 0) { good = j; good_n = seen.size(); }
        }
        if (good < 0) return ACE_OK;
        seen.resize(good_n);
        win_start.push_back(i);
        win_types.push_back(seen);
        i = good;
    }
    const int n_w = (int)win_start.size();
    if (n_w < 2) return ACE_OK;
    auto row_addr = [&](int w, uint32_t ty) {
        const std::vector<uint32_t> &v = win_types[w];
        return (uint32_t)((w & 1) * slots + (uint32_t)(std::find(v.begin(), v.end(), ty) - v.begin())) * crow;
    };
    // the per-position table
    std::vector<ace_u4> p4(pos_entries);
    const uint32_t kind_stride = (uint32_t)t->n_glog * ACE_PK32_BLOCK;
    for (size_t i = 0, w = 0; i < pos_entries; ++i) {
        if (i >= (size_t)N) { p4[i] = ace_u4{0u, hot_len, pk32_off, 0u}; continue; }
        while ((int)w + 1 < n_w && (size_t)win_start[w + 1] <= i) ++w;
        const uint32_t info = t->pos_info[i], at = row_addr((int)w, types[i] & 0xffu);
        p4[i] = ace_u4{at, at + hot_len, pk32_off + ((info >> 16) & 0xffu) * kind_stride * 4u,
                       (((info >> 24) & 1u) ^ 1u) | (((info >> 25) & 1u) << 1) | ((types[i] & 0xffffu) << 8)};
    }
    // the loads of each window, dealt to the wavefronts in turn (the last load of a part ends with the part: it may
    // overlap the one before it)
    std::vector<std::vector<ace_u2>> loads(n_w);
    for (int w = 0; w < n_w; ++w)
        for (uint32_t ty : win_types[w]) {
            const uint32_t at = row_addr(w, ty), src = (uint32_t)(ty * row_bytes);
            for (int part = 0; part < 2; ++part) {
                const uint32_t len = part ? z_len : hot_len, from = src + (uint32_t)(part ? t->z_off : t->hot_off) * 8u;
                for (uint32_t off = 0; off < len; off += 1024u) {
                    const uint32_t o = off + 1024u <= len ? off : len - 1024u;
                    loads[w].push_back(ace_u2{from + o, at + (part ? hot_len : 0u) + o});
                }
            }
        }
    for (int w = 0; w < n_w; ++w)
        if (loads[w].size() > 16u * 8u) return ACE_OK;
    const int n_ev = n_w + 1;
    std::vector<ace_u4> blob((size_t)n_ev * 16u * 5u, ace_u4{0u, 0u, 0u, 0u});
    const uint64_t rows_at = (uint64_t)(uintptr_t)h->d_rows;
    for (int e = 0; e < n_ev; ++e) {
        const int entering = e < 2 ? 0 : e - 1;                        // the window walked after this event
        int fetch = e == 0 ? 0 : entering + 1;
        if (fetch >= n_w) fetch = entering - 1;
        const uint32_t nextwin = entering + 1 < n_w ? (uint32_t)win_start[entering + 1] : 0x7fffffffu;
        for (uint32_t v = 0; v < 16u; ++v) {
            ace_u4 *rec = &blob[((size_t)e * 16u + v) * 5u];
            uint32_t d[16] = {0};
            uint32_t n = 0;
            for (size_t c = v; c < loads[fetch].size(); c += 16u, ++n) { d[2 * n] = loads[fetch][c].x; d[2 * n + 1] = loads[fetch][c].y; }
            rec[0] = ace_u4{nextwin, (e == 0 ? 1u : 0u) | (n << 8), (uint32_t)rows_at, (uint32_t)(rows_at >> 32)};
            for (int q = 0; q < 4; ++q) rec[1 + q] = ace_u4{d[4 * q], d[4 * q + 1], d[4 * q + 2], d[4 * q + 3]};
        }
    }
    int rc = upload((void **)&h->d_win_dma, blob.data(), blob.size() * sizeof(ace_u4));
    if (rc == ACE_OK) rc = upload((void **)&h->d_pos4, p4.data(), p4.size() * sizeof(ace_u4));
    if (rc != ACE_OK) return rc;
    h->n_fetch = n_ev;
    h->geom_wa = h->geom;
    h->geom_wa.rk_lds_off = 2u * slots * crow;
    h->geom_wa.stg_lds_off = stg_off; h->geom_wa.lut2_lds_off = lut2_off; h->geom_wa.pk32_lds_off = pk32_off; h->geom_wa.pace_lds_off = 0; h->geom_wa.lut2a_lds_off = lut2a_off;
    h->lds_bytes_wa = lds_end;
    return ACE_OK;
}

// The dense tables, where the handle's fit that form.
static int setup_dense(ace_handle *h, const ace_tables_t *t, size_t pos_entries) {
    AceDenseTables d;
    ace_dense_build(t, pos_entries, d);
    if (!d.ok) return ACE_OK;
    h->dense = d.args;
    int rc = upload((void **)&h->dense.pos, d.pos.data(), d.pos.size() * sizeof(ace_u4));
    if (rc == ACE_OK) rc = upload((void **)&h->dense.pos_duo, d.pos_duo.data(), d.pos_duo.size() * sizeof(ace_u2));
    if (rc == ACE_OK) rc = upload((void **)&h->dense.image, d.image.data(), d.image.size());
    if (rc == ACE_OK && !d.windows.empty()) {
        rc = upload((void **)&h->d_dense_rows, d.rows.data(), d.rows.size());
        if (rc != ACE_OK) return rc;
        const std::vector<uint32_t> ev = dense_events(d, (uint64_t)(uintptr_t)h->d_dense_rows);
        rc = upload((void **)&h->dense.events, ev.data(), ev.size() * 4);
        h->dense.n_events = (uint32_t)d.windows.size() + 1u;
    }
    if (rc != ACE_OK) return rc;
    h->dense_lds = d.lds;
    h->dense_lanes = d.lanes;
    return ACE_OK;
}

// The assembly loop over the table compiler's rows: LDS of a workgroup, or 0 where it cannot walk them.
static uint32_t many_lds(const ace_handle_t *h) {
    const bool win = h->n_windows > 1;
    if (win ? !h->d_win_dma : !(h->d_pos4 && h->geom.lut2a_lds_off && h->flat_rows16 > 0)) return 0;
    const uint32_t tables = win ? h->lds_bytes_wa : h->lds_bytes, deal = (win ? h->geom_wa : h->geom).rk_lds_off + 128u + 2u * 1024u, lds = deal > tables ? deal : tables;
    return lds <= kMaxLds ? lds : 0;
}
static AceRouteTables route_tables(const ace_handle_t *h) {
    AceRouteTables t;
    t.ops = h->geom.N;
    t.spread = h->d_pos_spread != nullptr;
    t.dense = h->dense.image != nullptr;
    t.dense_windows = h->dense.events ? (int32_t)h->dense.n_events - 1 : 0;
    t.dense_lanes = h->dense_lanes;
    t.many = many_lds(h) != 0;
    t.windows = h->n_windows;
    t.deferred = (h->n_windows == 1 || h->d_pos_types) && h->geom.N < 32768 && !(h->geom.flags & ACE_F_COLLECTIVE_MEM);
    return t;
}

// The device address of `scratch` on the current device (looked up once per device).
static int static_scratch_ptr(double **out) {
    int dev = -1;
    ACE_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return ACE_EINVAL;
    std::lock_guard<std::mutex> lock(g_static_mutex);
    if (!g_static_ptr[dev]) {
        void *p = nullptr;
        ACE_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) return ACE_EHIP;
        g_static_ptr[dev] = static_cast<double *>(p);
    }
    *out = g_static_ptr[dev];
    return ACE_OK;
}

extern "C" {

int ace_create(const ace_tables_t *t, ace_handle_t **out) {
    if (!t || !out) return ACE_EINVAL;
    *out = nullptr;
    if (t->abi_version != ACE_ABI_VERSION) return ACE_EVERSION;
    if (t->num_ops <= 0 || t->num_types <= 0 || t->n_mbs <= 0 || t->n_mbs > 15 || t->n_tp <= 0 || t->n_tp > 4 ||
        (t->n_algo != 1 && t->n_algo != 2) || t->n_diag <= 0 || t->n_diag > 14 || t->n_glog <= 0 || t->n_glog > 16 ||
        t->n_z < 0 || t->n_z == 1 || t->n_z > 15 || ((t->flags & ACE_F_RESHARDING) && t->n_z < 2) || t->z_table_doubles <= 0 || (t->z_table_doubles & (t->z_table_doubles - 1)) || t->n_pair_kinds <= 0 || t->n_pair_kinds > 255 || t->row_doubles <= 0 ||
        (t->row_doubles & 1) || t->n_windows <= 0 || t->lds_row_bytes <= 0 || (t->lds_row_bytes & 15) ||
        !t->rows || !t->pos_info || !t->pair_kinds || !t->stage_lut || !t->nb_minus_1 || !t->win_pos ||
        !t->win_row_begin || !t->win_rows)
        return ACE_EINVAL;
    const int C = t->n_tp * t->n_algo;
    // sub-tables must lie inside a row and be 16-byte aligned
    const int64_t hot_end = (int64_t)t->hot_off + (int64_t)(t->n_diag + 1) * C * 6;
    const int64_t start_end = (int64_t)t->start_off + (int64_t)t->n_diag * C * 3;
    const int64_t out_end = (int64_t)t->out_off + (int64_t)t->n_mbs * t->n_tp * t->n_algo * 2;
    if ((t->flags & ACE_F_COLLECTIVE_MEM) && !(t->flags & ACE_F_RESHARDING)) return ACE_EINVAL;
    const int64_t z_end = (int64_t)t->z_off + (int64_t)t->n_z * t->z_table_doubles * ((t->flags & ACE_F_COLLECTIVE_MEM) ? 2 : 1);
    if (t->z_table_doubles < t->n_diag * C) return ACE_EINVAL;
    if ((t->hot_off & 1) || (t->start_off & 1) || (t->out_off & 1) || (t->z_off & 1) || t->hot_off < 0 ||
        t->start_off < 0 || t->out_off < 0 || t->z_off < 0 ||
        hot_end > t->row_doubles || start_end > t->row_doubles || out_end > t->row_doubles || z_end > t->row_doubles)
        return ACE_EINVAL;
    const int64_t row_bytes = (int64_t)t->row_doubles * 8;
    if (row_bytes > t->lds_row_bytes || t->lds_row_bytes > (int32_t)kMaxLds) return ACE_ETOOBIG;
    const int32_t rk_bytes = t->n_pair_kinds * t->n_glog * 64;
    const int32_t stg_words = t->n_mbs * 16;
    const uint32_t rk_off = (uint32_t)t->lds_row_bytes;
    uint32_t stg_off, lut2_off;
    uint32_t lds_bytes = ace_lds_layout(rk_off, (uint32_t)rk_bytes, (uint32_t)stg_words, &stg_off, &lut2_off);
    if (lds_bytes > kMaxLds) return ACE_ETOOBIG;
    // the assembly loop's pair-kind table, where the table has room and its entries can hold the offsets (otherwise plain
    // scoring takes the C++ form of the loop)
    uint32_t pk32_off = 0, pace_off = 0, lut2a_off = 0;
    if (t->n_windows == 1) {                               // (windowed rows: setup_windowed_asm lays LDS out anew)
        uint32_t off;
        const uint32_t end = ace_lds_pk32(lds_bytes, (uint32_t)rk_bytes, &off);
        // (behind it: the loop's arrival counters and its own per-(micro-batch, stage size) offset pairs)
        if (end + 128u + (uint32_t)stg_words * 8u + 16u <= kMaxLds && ((int64_t)(t->n_z > 0 ? t->n_z : 1) * t->z_table_doubles * 8) <= 65536) {
            pk32_off = off;
            pace_off = (end + 15u) & ~15u;
            lut2a_off = pace_off + 128u;
            lds_bytes = lut2a_off + (uint32_t)stg_words * 8u;
        }
    }
    // (the in-kernel sort keeps its bins and its permutation in the first 128 + 2 * kBlock bytes of LDS before the
    // tables are staged there: tiny tables still get that much)
    const uint32_t lds_floor = 128u + 2u * (uint32_t)kBlock;
    const uint32_t lds_alloc = lds_bytes < lds_floor ? lds_floor : lds_bytes;
    // window tables: window starts are multiples of 4 ops; every referenced row must fit the
    // resident region; every position's row offsets must point at a row start inside it
    const int32_t n_win_rows = t->win_row_begin[t->n_windows];
    if (t->win_pos[0] != 0 || t->win_row_begin[0] != 0 || n_win_rows <= 0) return ACE_EINVAL;
    for (int w = 0; w < t->n_windows; ++w) {
        if (t->win_pos[w + 1] <= t->win_pos[w] || t->win_row_begin[w + 1] < t->win_row_begin[w] || (t->win_pos[w] & 3))
            return ACE_EINVAL;
    }
    if (t->win_pos[t->n_windows] < t->num_ops) return ACE_EINVAL;
    for (int r = 0; r < n_win_rows; ++r) {
        if (t->win_rows[2 * r] >= (uint32_t)t->num_types) return ACE_EINVAL;
        if ((int64_t)t->win_rows[2 * r + 1] + row_bytes > t->lds_row_bytes || (t->win_rows[2 * r + 1] & 15u)) return ACE_EINVAL;
    }
    for (int i = 0; i <= t->num_ops; ++i) {
        const uint32_t pi = t->pos_info[i];
        if ((int64_t)((pi & 0xffu) + 1) * row_bytes > t->lds_row_bytes || (int64_t)(((pi >> 8) & 0xffu) + 1) * row_bytes > t->lds_row_bytes ||
            ((pi >> 16) & 0xffu) >= (uint32_t)t->n_pair_kinds)
            return ACE_EINVAL;
    }
    for (int j = 0; j < stg_words; ++j) {
        // the diag of every (micro-batch, stage size) pair must exist (n_diag = the all-NaN one)
        if ((t->stage_lut[j] & 0xffffu) > (uint32_t)t->n_diag) return ACE_EINVAL;
    }
    for (int j = 0; j < rk_bytes; ++j) {
        const uint32_t lim = t->n_z ? (uint32_t)t->n_z : 1u;
        if ((t->pair_kinds[j] & 15u) >= lim || (uint32_t)(t->pair_kinds[j] >> 4) >= lim) return ACE_EINVAL;
    }

    ace_handle *h = new (std::nothrow) ace_handle();       // (all zeros)
    if (!h) return ACE_ENOMEM;
    AceGeom &g = h->geom;
    g.N = t->num_ops; g.P = 0; g.G = (t->num_ops + 15) / 16;
    g.C = C; g.A_shift = t->n_algo == 2 ? 1 : 0;
    g.n_mbs = t->n_mbs; g.n_tp = t->n_tp; g.n_algo = t->n_algo; g.n_glog = t->n_glog; g.n_pair_kinds = t->n_pair_kinds;
    g.hot_off = (uint32_t)t->hot_off * 8u; g.start_off = (uint32_t)t->start_off * 8u;
    g.out_off = (uint32_t)t->out_off * 8u; g.z_off = (uint32_t)t->z_off * 8u;
    g.z_shift = 3;
    while ((1 << (g.z_shift - 3)) < t->z_table_doubles) ++g.z_shift;
    g.zm_delta = (uint32_t)t->n_z << g.z_shift;
    g.rk_lds_off = rk_off; g.stg_lds_off = stg_off; g.lut2_lds_off = lut2_off; g.pk32_lds_off = pk32_off; g.pace_lds_off = pace_off; g.lut2a_lds_off = lut2a_off;
    g.rk_kind_stride = (uint32_t)(t->n_glog * 64);
    g.row_bytes = (uint32_t)row_bytes;
    g.flags = t->flags; g.main_params = t->main_params; g.optimizer = t->optimizer;
    g.mem_limit = 0.0; g.strict = 0;
    h->n_windows = t->n_windows; h->row_doubles = t->row_doubles; h->rk_bytes = rk_bytes; h->stg_words = stg_words;
    // rows resident, slot r of LDS holding row r: the kernels stage them as one block
    h->flat_rows16 = 0;
    if (t->n_windows == 1 && (row_bytes & 15) == 0) {
        bool flat = true;
        for (int r = 0; r < n_win_rows; ++r)
            flat = flat && t->win_rows[2 * r] == (uint32_t)r && t->win_rows[2 * r + 1] == (uint32_t)(r * row_bytes);
        if (flat) h->flat_rows16 = (int32_t)(n_win_rows * row_bytes / 16);
    }
    h->num_types = t->num_types; h->lds_bytes = lds_alloc;
    const size_t pos_entries = (size_t)((t->num_ops + 15) / 16) * 16 + 16;
    int rc;
    double *scratch_here = nullptr;
    if ((rc = hipGetDevice(&h->device) == hipSuccess ? ACE_OK : ACE_EHIP) ||
        (rc = static_scratch_ptr(&scratch_here)) ||
        // (zeros behind the last row: a code byte that names no profiled entry may point a few entries past its row)
        (rc = upload((void **)&h->d_rows, t->rows, (size_t)t->num_types * row_bytes, (size_t)t->num_types * row_bytes + 4096u)) ||
        (rc = upload((void **)&h->d_pos_info, t->pos_info, (size_t)(t->num_ops + 1) * 4, pos_entries * 4)) ||
        (rc = upload_pos4(h, t, pos_entries, pk32_off)) ||
        (rc = upload_pos_types(h, t, pos_entries)) || (rc = or_enomem([&] { return upload_pos_spread(h, t, pos_entries); })) ||
        (rc = upload((void **)&h->d_pair_kinds, t->pair_kinds, (size_t)rk_bytes)) ||
        (rc = upload((void **)&h->d_stage_lut, t->stage_lut, (size_t)stg_words * 4)) ||
        (rc = upload((void **)&h->d_nbm1, t->nb_minus_1, (size_t)t->n_mbs * 8)) ||
        (rc = upload((void **)&h->d_win_pos, t->win_pos, (size_t)(t->n_windows + 1) * 4)) ||
        (rc = upload((void **)&h->d_win_row_begin, t->win_row_begin, (size_t)(t->n_windows + 1) * 4)) ||
        (rc = upload((void **)&h->d_win_rows, t->win_rows, (size_t)n_win_rows * 8)) ||
        (rc = or_enomem([&] { return setup_windowed_asm(h, t, pos_entries, rk_bytes, stg_words); })) ||
        (rc = or_enomem([&] { return setup_dense(h, t, pos_entries); })) ||
        (rc = allow_big_lds<false, false, false, false>()) || (rc = allow_big_lds<false, false, true, false>()) ||
        (rc = allow_big_lds<false, false, false, true>()) || (rc = allow_big_lds<false, false, true, true>()) ||
        (rc = allow_big_lds<true, false, false, false>()) || (rc = allow_big_lds<true, false, true, false>()) ||
        (rc = allow_duo_lds()) || (rc = allow_many_lds<false>()) || (rc = allow_many_lds<true>()) || (rc = allow_dense_lds()) ||
        (rc = allow_big_lds<true, true, false, false>()) || (rc = allow_big_lds<true, true, true, false>())) {
        ace_destroy(h);
        return rc;
    }
    h->route = route_tables(h);
    *out = h;
    return ACE_OK;
}

void ace_destroy(ace_handle_t *h) {
    if (!h) return;
    (void)hipFree(h->d_rows); (void)hipFree(h->d_pos_info); (void)hipFree(h->d_pos_types); (void)hipFree(h->d_pos_spread);
    (void)hipFree(h->d_pair_kinds);
    if (h->d_pos4) (void)hipFree(h->d_pos4);
    if (h->d_win_dma) (void)hipFree(h->d_win_dma);
    for (const void *p : {(const void *)h->dense.image, (const void *)h->dense.pos, (const void *)h->dense.pos_duo, (const void *)h->dense.events, (const void *)h->d_dense_rows})
        if (p) (void)hipFree(const_cast<void *>(p));
    (void)hipFree(h->d_stage_lut); (void)hipFree(h->d_nbm1); (void)hipFree(h->d_win_pos);
    (void)hipFree(h->d_win_row_begin); (void)hipFree(h->d_win_rows);
    if (h->d_rc_pos) (void)hipFree(h->d_rc_pos);
    if (h->d_rc_act) (void)hipFree(h->d_rc_act);
    if (h->host_in) (void)hipHostFree(h->host_in);
    if (h->host_out) (void)hipHostFree(h->host_out);
    if (h->d_stage_ws) (void)hipFree(h->d_stage_ws);
    if (h->step) {
        if (h->step->host) (void)hipHostFree(h->step->host);
        if (h->step->dev) (void)hipFree(h->step->dev);
        delete h->step;
    }
    delete h;
}

static int fill_args(ace_handle_t *h, const ace_batch_t *b, double memory_limit, int strict, double *d_iter_ms,
                     double *d_peak_mb, uint8_t *d_feasible, uint8_t *d_status, double *d_stage_out, AceKernelArgs *a) {
    if (!h || !b || !b->d_codes || !b->d_hdr || !d_iter_ms || !d_peak_mb || !d_feasible) return ACE_EINVAL;
    if (b->n_plans == 0 || b->n_plans > 0x7fffffffull) return ACE_EINVAL;
    if (((uintptr_t)b->d_codes & 15u) || ((uintptr_t)b->d_hdr & 15u) || ((uintptr_t)b->d_range & 7u) || ((uintptr_t)b->d_order & 3u))
        return ACE_EINVAL;
    if (b->d_range && !d_stage_out) return ACE_EINVAL;   // single-stage queries are read from their stage record
    a->g = h->geom;
    a->g.P = (int32_t)b->n_plans;
    a->g.mem_limit = memory_limit;
    a->g.strict = strict ? 1 : 0;
    a->codes = reinterpret_cast<const ace_u4 *>(b->d_codes);
    a->hdr = reinterpret_cast<const ace_u4 *>(b->d_hdr);
    a->range = reinterpret_cast<const ace_u2 *>(b->d_range);
    a->order = b->d_order;
    a->rows = h->d_rows; a->pos_info = h->d_pos_info; a->pos_types = h->d_pos_types; a->pos4 = h->d_pos4; a->win_dma = h->d_win_dma; a->n_fetch = h->n_fetch; a->pos_spread = h->d_pos_spread; a->pair_kinds = h->d_pair_kinds; a->stage_lut = h->d_stage_lut;
    a->nbm1 = h->d_nbm1; a->win_pos = h->d_win_pos; a->win_row_begin = h->d_win_row_begin; a->win_rows = h->d_win_rows;
    a->n_windows = h->n_windows; a->row_doubles = h->row_doubles; a->rk_bytes = h->rk_bytes; a->stg_words = h->stg_words;
    a->flat_rows16 = h->flat_rows16;
    a->iter_ms = d_iter_ms; a->peak_mb = d_peak_mb; a->feasible = d_feasible; a->status = d_status; a->stage_out = d_stage_out;
    a->stage_ws = nullptr;
    return ACE_OK;
}

}  // extern "C"

template <bool BD, bool RANGED, bool WIN, bool DEFER>
static void launch_score_b(const ace_handle_t *h, const AceKernelArgs &a, hipStream_t s) {
    const size_t P = (size_t)a.g.P;
    if (a.g.flags & ACE_F_COLLECTIVE_MEM) {
        if (!DEFER)         // (ensure_stage_ws never hands such tables to the deferred kernel)
            hipLaunchKernelGGL((ace_score_kernel<BD, RANGED, WIN, false, kBlock, true>), dim3((unsigned)((P + kBlock - 1) / kBlock)),
                               dim3(kBlock), h->lds_bytes, s, a);
    } else if ((P + kBlock - 1) / kBlock < (size_t)kSmallBatchBlocks)
        hipLaunchKernelGGL((ace_score_kernel<BD, RANGED, WIN, DEFER, kSmallBlock>), dim3((unsigned)((P + kSmallBlock - 1) / kSmallBlock)),
                           dim3(kSmallBlock), h->lds_bytes, s, a);
    else
        hipLaunchKernelGGL((ace_score_kernel<BD, RANGED, WIN, DEFER, kBlock>), dim3((unsigned)((P + kBlock - 1) / kBlock)),
                           dim3(kBlock), h->lds_bytes, s, a);
}

template <bool BD, bool RANGED>
static void launch_score_w(const ace_handle_t *h, const AceKernelArgs &a, hipStream_t s) {
    if (h->n_windows > 1) launch_score_b<BD, RANGED, true, false>(h, a, s);
    else launch_score_b<BD, RANGED, false, false>(h, a, s);
}

template <bool BD, bool RANGED, bool COLL>
static void launch_spread_c(const AceKernelArgs &a, hipStream_t s) {
    SpreadShared sh;
    const uint32_t lds = ace_spread_layout(SpreadCols<BD, COLL>::kCols, a.g.G, nullptr, &sh);
    hipLaunchKernelGGL((ace_spread_kernel<BD, RANGED, COLL>), dim3((unsigned)a.g.P), dim3(kSpreadLanes), lds, s, a);
}
template <bool BD, bool RANGED>
static void launch_spread(const AceKernelArgs &a, hipStream_t s) {
    if (a.g.flags & ACE_F_COLLECTIVE_MEM) launch_spread_c<BD, RANGED, true>(a, s);
    else launch_spread_c<BD, RANGED, false>(a, s);
}

static void launch_many(const ace_handle_t *h, const AceKernelArgs &a, hipStream_t s) {
    const bool win = h->n_windows > 1;
    AceKernelArgs b = a;
    if (win) {                                          // (that loop lays LDS out its own way)
        b.g = h->geom_wa;
        b.g.P = a.g.P; b.g.mem_limit = a.g.mem_limit; b.g.strict = a.g.strict;
    }
    const AceShares w = ace_many_shares(a.g.P);
    hipLaunchKernelGGL(win ? ace_many_kernel<true> : ace_many_kernel<false>, dim3((unsigned)w.groups), dim3(1024), many_lds(h), s, b, w.slices);
}
static void launch_dense(const ace_handle_t *h, const AceKernelArgs &a, hipStream_t s) {
    const AceShares w = ace_dense_shares(h->route, a.g.P);
    const auto kernel = h->dense.events ? ace_dense_kernel<true, kDenseWinLanes> : h->dense_lanes == kDenseWinLanes ? ace_dense_kernel<false, kDenseWinLanes> : ace_dense_kernel<false, kDenseLanes>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)w.groups), dim3((unsigned)h->dense_lanes), h->dense_lds, s, a, h->dense, w.slices);
}
static void launch_duo(const ace_handle_t *h, const AceKernelArgs &a, hipStream_t s) {
    const int L = ace_duo_lanes(a.g.P);
    const dim3 groups((unsigned)((a.g.P + L - 1) / L));
    const uint32_t lds = h->dense.image16 * 16u + ace_duo_scratch(L);
    const auto kernel = L == 64 ? ace_duo_kernel<64> : L == 128 ? ace_duo_kernel<128> : ace_duo_kernel<256>;
    hipLaunchKernelGGL(kernel, groups, dim3(kDuoBlock), lds, s, a, h->dense);
}

// `workspace`: bytes behind a.stage_ws.
static void launch_score(const ace_handle_t *h, const AceKernelArgs &a, size_t workspace, hipStream_t s) {
    switch (ace_route(h->route, a.g.P, a.stage_out != nullptr, a.stage_ws ? workspace : 0)) {
    case ACE_K_SPREAD:
        if (a.range) launch_spread<true, true>(a, s);
        else if (a.stage_out) launch_spread<true, false>(a, s);
        else launch_spread<false, false>(a, s);
        return;
    case ACE_K_DUO: return launch_duo(h, a, s);
    case ACE_K_DENSE: return launch_dense(h, a, s);
    case ACE_K_MANY: return launch_many(h, a, s);
    case ACE_K_DEFERRED:
        if (h->n_windows > 1) launch_score_b<false, false, true, true>(h, a, s);
        else launch_score_b<false, false, false, true>(h, a, s);
        return;
    case ACE_K_IN_PLACE:
        if (a.range) launch_score_w<true, true>(h, a, s);
        else if (a.stage_out) launch_score_w<true, false>(h, a, s);
        else launch_score_w<false, false>(h, a, s);
    }
}

// Plain scoring defers its stage tails to a per-plan workspace; the handle keeps one and grows it on demand.
static int ensure_stage_ws(ace_handle_t *h, AceKernelArgs *a) {
    a->stage_ws = nullptr;
    const size_t need = a->range || a->stage_out ? 0 : ace_workspace(h->route, a->g.P), plans = ace_workspace_plans(a->g.P);
    if (need == 0) return ACE_OK;
    if (plans > h->stage_ws_plans) {
        if (h->stage_ws_fixed) return ACE_EFIXED;
        if (need > h->stage_ws_bytes) {
            if (h->d_stage_ws) ACE_HIP(hipFree(h->d_stage_ws));
            h->d_stage_ws = nullptr;
            h->stage_ws_plans = h->stage_ws_bytes = 0;
            ACE_HIP(hipMalloc((void **)&h->d_stage_ws, need));
            h->stage_ws_bytes = need;
        }
        h->stage_ws_plans = plans;
    }
    a->stage_ws = h->d_stage_ws;
    return ACE_OK;
}

extern "C" {

int ace_reserve(ace_handle_t *h, size_t max_plans, int fixed) {
    if (!h || max_plans > 0x7fffffffull) return ACE_EINVAL;
    std::lock_guard<std::mutex> lock(h->workspace);
    if (max_plans) {
        AceKernelArgs a;
        memset(&a, 0, sizeof(a));
        a.g.P = (int32_t)max_plans;
        const int was_fixed = h->stage_ws_fixed;
        h->stage_ws_fixed = 0;
        const int rc = ensure_stage_ws(h, &a);
        h->stage_ws_fixed = was_fixed;
        if (rc) return rc;
    }
    h->stage_ws_fixed = fixed ? 1 : 0;
    return ACE_OK;
}

int ace_score_batch(ace_handle_t *h, const ace_batch_t *batch, double memory_limit, int strict, double *d_iter_ms,
                    double *d_peak_mb, uint8_t *d_feasible, uint8_t *d_status, double *d_stage_out, void *stream) {
    AceKernelArgs a;
    int rc = fill_args(h, batch, memory_limit, strict, d_iter_ms, d_peak_mb, d_feasible, d_status, d_stage_out, &a);
    if (rc) return rc;
    std::lock_guard<std::mutex> lock(h->workspace);
    if ((rc = ensure_stage_ws(h, &a))) return rc;
    launch_score(h, a, h->stage_ws_bytes, (hipStream_t)stream);
    ACE_HIP(hipGetLastError());
    return ACE_OK;
}

size_t ace_pack_host(const uint8_t *codes, const uint32_t *hdr, const uint32_t *range, size_t n_plans, int num_ops, uint8_t *out) {
    const size_t P = n_plans, N = num_ops > 0 ? (size_t)num_ops : 0, G = (N + 15) / 16, off_hdr = G * P * 16, off_rng = off_hdr + P * 16;
    if (out) {
        for (size_t p = 0; p < P && G; ++p) {
            const uint8_t *row = codes + p * N;
            for (size_t g = 0; g + 1 < G; ++g) memcpy(out + (g * P + p) * 16, row + g * 16, 16);
            unsigned char last[16] = {0};
            memcpy(last, row + (G - 1) * 16, N - (G - 1) * 16);
            memcpy(out + ((G - 1) * P + p) * 16, last, 16);
        }
        memcpy(out + off_hdr, hdr, P * 16);
        if (range) memcpy(out + off_rng, range, P * 8);
    }
    return off_rng + (range ? P * 8 : 0);
}

int ace_score_host(ace_handle_t *h, const uint8_t *codes, const uint32_t *hdr, const uint32_t *range, size_t n_plans,
                   double memory_limit, int strict, double *times, uint8_t *flags, double *stage_out, void *stream) {
    if (!h || !codes || !hdr || !times || !flags || n_plans == 0 || (range && !stage_out)) return ACE_EINVAL;
    const size_t P = n_plans, N = (size_t)h->geom.N, G = (size_t)h->geom.G;
    const size_t rec_bytes = stage_out ? P * (range ? 1 : ACE_MAX_STAGES) * ACE_STAGE_REC * sizeof(double) : 0;
    // in: codes [G][P][16] | headers | ranges; out: times | records | flags
    const size_t off_hdr = G * P * 16, off_rng = off_hdr + P * 16, n_in = ace_pack_host(nullptr, nullptr, range, P, (int)N, nullptr);
    const size_t off_rec = 16 * P, off_flags = off_rec + rec_bytes, n_out = off_flags + 2 * P;
    if (P > kHostIoBytes || n_in > kHostIoBytes || n_out > kHostIoBytes) return ACE_ETOOBIG;
    std::lock_guard<std::mutex> lock(h->host_calls);
    int dev = -1;
    ACE_HIP(hipGetDevice(&dev));
    if (dev != h->device) ACE_HIP(hipSetDevice(h->device));
    int rc = ACE_OK;
    if (!h->host_in && (hipHostMalloc((void **)&h->host_in, kHostIoBytes, hipHostMallocDefault) != hipSuccess ||
                        hipHostMalloc((void **)&h->host_out, kHostIoBytes, hipHostMallocDefault) != hipSuccess)) {
        if (h->host_in) (void)hipHostFree(h->host_in);
        h->host_in = nullptr;
        h->host_out = nullptr;
        rc = ACE_ENOMEM;
    }
    if (rc == ACE_OK) {
        unsigned char *in = h->host_in, *out = h->host_out;
        ace_pack_host(codes, hdr, range, P, (int)N, in);
        if (rec_bytes) memset(out + off_rec, 0, rec_bytes);      // (a plan has records for its stages only)
        const ace_batch_t b{in, reinterpret_cast<const uint32_t *>(in + off_hdr), range ? reinterpret_cast<const uint32_t *>(in + off_rng) : nullptr,
                            P, nullptr};
        double *t = reinterpret_cast<double *>(out);
        rc = ace_score_batch(h, &b, memory_limit, strict, t, t + P, out + off_flags, out + off_flags + P,
                             rec_bytes ? reinterpret_cast<double *>(out + off_rec) : nullptr, stream);
        if (rc == ACE_OK && hipStreamSynchronize((hipStream_t)stream) != hipSuccess) {
            snprintf(g_hip_err, sizeof(g_hip_err), "hipStreamSynchronize failed");
            rc = ACE_EHIP;
        }
        if (rc == ACE_OK) {
            memcpy(times, t, 16 * P);
            memcpy(flags, out + off_flags, 2 * P);
            if (rec_bytes) memcpy(stage_out, out + off_rec, rec_bytes);
        }
    }
    if (dev != h->device) ACE_HIP(hipSetDevice(dev));
    return rc;
}

int ace_score_batch_static(ace_handle_t *h, const ace_batch_t *batch, double memory_limit, int strict, double *d_iter_ms,
                           double *d_peak_mb, uint8_t *d_feasible, uint8_t *d_status, void *stream) {
    if (batch && (batch->d_range || batch->n_plans > (size_t)ACE_STATIC_MAX_PLANS)) return batch->d_range ? ACE_EINVAL : ACE_ETOOBIG;
    AceKernelArgs a;
    int rc = fill_args(h, batch, memory_limit, strict, d_iter_ms, d_peak_mb, d_feasible, d_status, nullptr, &a);
    if (rc) return rc;
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev != h->device || dev < 0 || dev >= kMaxDevices) return ACE_EINVAL;
    // (tables that take the kernels without deferred stage tails need no scratch; it was looked up by ace_create on this device)
    const bool deferred = h->route.dense || h->route.deferred;
    a.stage_ws = deferred ? g_static_ptr[dev] : nullptr;
    if (deferred && !a.stage_ws) return ACE_EINVAL;
    launch_score(h, a, kStaticBytes, (hipStream_t)stream);
    ACE_HIP(hipGetLastError());
    return ACE_OK;
}

int ace_time_score_kernel(ace_handle_t *h, const ace_batch_t *batch, double memory_limit, int strict, double *d_iter_ms,
                          double *d_peak_mb, uint8_t *d_feasible, int reps, void *stream, double *avg_ms) {
    if (reps <= 0 || !avg_ms) return ACE_EINVAL;
    AceKernelArgs a;
    int rc = fill_args(h, batch, memory_limit, strict, d_iter_ms, d_peak_mb, d_feasible, nullptr, nullptr, &a);
    if (rc) return rc;
    std::lock_guard<std::mutex> lock(h->workspace);
    if ((rc = ensure_stage_ws(h, &a))) return rc;
    hipStream_t s = (hipStream_t)stream;
    hipEvent_t e0, e1;
    ACE_HIP(hipEventCreate(&e0));
    ACE_HIP(hipEventCreate(&e1));
    ACE_HIP(hipEventRecord(e0, s));
    for (int r = 0; r < reps; ++r) launch_score(h, a, h->stage_ws_bytes, s);
    ACE_HIP(hipEventRecord(e1, s));
    ACE_HIP(hipEventSynchronize(e1));
    float ms = 0.f;
    ACE_HIP(hipEventElapsedTime(&ms, e0, e1));
    ACE_HIP(hipEventDestroy(e0));
    ACE_HIP(hipEventDestroy(e1));
    ACE_HIP(hipGetLastError());
    *avg_ms = (double)ms / reps;
    return ACE_OK;
}

// workspace layout: TopkState | hist[kRadix] | less[cap] | ties[cap] | buf[pow2(2*cap)]
static unsigned int topk_cap(int k) { return (unsigned)k; }

size_t ace_topk_workspace_bytes(size_t n, int k) {
    (void)n;
    if (k <= 0) return 0;
    const unsigned cap = topk_cap(k);
    const unsigned p2 = next_pow2(2 * cap);
    // (the last part: what the short form's first launch leaves)
    return 256 + sizeof(unsigned int) * kRadix + sizeof(Cand) * ((size_t)cap * 2 + p2) + sizeof(Cand) * kShortMaxEntries;
}

int ace_topk(ace_handle_t *h, const double *d_iter_ms, const uint8_t *d_feasible, size_t n, int k, int64_t *d_idx,
             double *d_val, int32_t *d_count, void *d_workspace, size_t workspace_bytes, void *stream) {
    if (!h || !d_iter_ms || !d_feasible || !d_idx || !d_val || !d_workspace || n == 0 || k <= 0 || k > (1 << 20)) return ACE_EINVAL;
    if (workspace_bytes < ace_topk_workspace_bytes(n, k) || ((uintptr_t)d_workspace & 15u)) return ACE_EINVAL;
    hipStream_t s = (hipStream_t)stream;
    unsigned char *ws = (unsigned char *)d_workspace;
    TopkState *st = (TopkState *)ws;
    unsigned int *hist = (unsigned int *)(ws + 256);
    const unsigned cap = topk_cap(k);
    const unsigned p2 = next_pow2(2 * cap);
    Cand *less = (Cand *)(ws + 256 + sizeof(unsigned int) * kRadix);
    Cand *ties = less + cap;
    Cand *buf = ties + cap;
    unsigned blocks = (unsigned)((n + kTopBlock * 8 - 1) / (kTopBlock * 8));
    if (blocks < 1) blocks = 1;
    if (blocks > 2048) blocks = 2048;
    const unsigned int per = short_stretch(n, k);
    if (per != ~0u) {
        Cand *cand = per ? buf + p2 : nullptr;
        const unsigned int groups = per ? (unsigned int)((n + per - 1) / per) : 0u, m = per ? groups * (unsigned int)k : (unsigned int)n;
        const int spread = m <= 4096 ? 2 : m <= 8192 ? 3 : 4;
        if (per == 4096) hipLaunchKernelGGL(topk_local<4>, dim3(groups), dim3(1024), 0, s, d_iter_ms, d_feasible, n, k, spread, cand);
        else if (per == 8192) hipLaunchKernelGGL(topk_local<8>, dim3(groups), dim3(1024), 0, s, d_iter_ms, d_feasible, n, k, spread, cand);
        else if (per) hipLaunchKernelGGL(topk_local<16>, dim3(groups), dim3(1024), 0, s, d_iter_ms, d_feasible, n, k, spread, cand);
        const auto last = m <= 4096 ? topk_final<4> : m <= 8192 ? topk_final<8> : topk_final<16>;
        hipLaunchKernelGGL(last, dim3(1), dim3(1024), 0, s, d_iter_ms, d_feasible, cand, m, k, (long long *)d_idx, d_val, d_count);
        ACE_HIP(hipGetLastError());
        return ACE_OK;
    }
    hipLaunchKernelGGL(topk_init, dim3(1), dim3(256), 0, s, st, hist, k);
    for (int pass = 0; pass < kPasses; ++pass) {
        hipLaunchKernelGGL(topk_hist, dim3(blocks), dim3(kTopBlock), 0, s, d_iter_ms, d_feasible, n, pass, st, hist);
        hipLaunchKernelGGL(topk_pick, dim3(1), dim3(kTopBlock), 0, s, st, hist, pass);
    }
    hipLaunchKernelGGL(topk_gather, dim3(blocks), dim3(kTopBlock), 0, s, d_iter_ms, d_feasible, n, st, less, ties, cap, cap);
    // ties: the gather keeps an arbitrary subset when more than `cap` plans share the k-th time;
    // redo them exactly (lowest indices first): a single-workgroup scan that stops early.
    hipLaunchKernelGGL(topk_ties_exact, dim3(1), dim3(kTieBlock), 0, s, d_iter_ms, d_feasible, n, st, ties, cap);
    hipLaunchKernelGGL(topk_finish, dim3(1), dim3(1024), 0, s, st, less, ties, cap, k, buf, p2, (long long *)d_idx, d_val, d_count);
    ACE_HIP(hipGetLastError());
    return ACE_OK;
}

int ace_apply_moves(const uint8_t *d_template_codes, const uint32_t *d_template_hdr, int n_templates,
                    const uint32_t *d_moves, size_t n_moves, int num_ops, int n_algo, uint8_t *d_codes_out,
                    uint32_t *d_hdr_out, uint64_t *d_keys_out, void *stream) {
    if (!d_template_codes || !d_template_hdr || !d_moves || !d_codes_out || !d_hdr_out || n_templates <= 0 ||
        n_templates > 65536 || n_moves == 0 || n_moves > 0x7fffffffull || num_ops <= 0 || num_ops >= 65536 ||
        (n_algo != 1 && n_algo != 2))
        return ACE_EINVAL;
    if (((uintptr_t)d_template_codes & 15u) || ((uintptr_t)d_template_hdr & 15u) || ((uintptr_t)d_moves & 15u) ||
        ((uintptr_t)d_codes_out & 15u) || ((uintptr_t)d_hdr_out & 15u) || ((uintptr_t)d_keys_out & 7u))
        return ACE_EINVAL;
    const int G = (num_ops + 15) / 16;
    const unsigned long long total = (unsigned long long)n_moves * (unsigned long long)G;
    const unsigned long long blocks = (total + 255) / 256;
    if (blocks > 0x7fffffffull) return ACE_ETOOBIG;
    ace_grid_parts(blocks, 256, [&](uint64_t first, uint32_t groups) {
        hipLaunchKernelGGL(apply_moves_kernel, dim3(groups), dim3(256), 0, (hipStream_t)stream,
                           reinterpret_cast<const ace_u4 *>(d_template_codes), reinterpret_cast<const ace_u4 *>(d_template_hdr),
                           n_templates, reinterpret_cast<const ace_u4 *>(d_moves), (unsigned long long)n_moves, G,
                           n_algo == 2 ? 1 : 0, reinterpret_cast<ace_u4 *>(d_codes_out), reinterpret_cast<ace_u4 *>(d_hdr_out),
                           reinterpret_cast<unsigned long long *>(d_keys_out), (unsigned long long)first);
    });
    ACE_HIP(hipGetLastError());
    return ACE_OK;
}

int ace_group_keys(const uint8_t *d_codes, const uint32_t *d_hdr, size_t n_plans, int num_ops, uint64_t *d_keys, void *stream) {
    if (!d_codes || !d_hdr || !d_keys || n_plans == 0 || n_plans > 0x7fffffffull || num_ops <= 0 || num_ops >= (1 << 20)) return ACE_EINVAL;
    if (((uintptr_t)d_codes & 15u) || ((uintptr_t)d_hdr & 15u) || ((uintptr_t)d_keys & 7u)) return ACE_EINVAL;
    const int G = (num_ops + 15) / 16;
    hipLaunchKernelGGL(group_keys_kernel, dim3((unsigned)((n_plans + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       reinterpret_cast<const ace_u4 *>(d_codes), reinterpret_cast<const ace_u4 *>(d_hdr),
                       (unsigned long long)n_plans, G, num_ops, reinterpret_cast<unsigned long long *>(d_keys));
    ACE_HIP(hipGetLastError());
    return ACE_OK;
}

int ace_gather_plans(const uint8_t *d_codes_in, const uint32_t *d_hdr_in, const uint32_t *d_perm, size_t n_plans, int num_ops,
                     uint8_t *d_codes_out, uint32_t *d_hdr_out, void *stream) {
    if (!d_codes_in || !d_hdr_in || !d_perm || !d_codes_out || !d_hdr_out || n_plans == 0 || n_plans > 0x7fffffffull ||
        num_ops <= 0 || num_ops >= (1 << 20) || d_codes_in == d_codes_out || d_hdr_in == d_hdr_out)
        return ACE_EINVAL;
    if (((uintptr_t)d_codes_in & 15u) || ((uintptr_t)d_hdr_in & 15u) || ((uintptr_t)d_codes_out & 15u) ||
        ((uintptr_t)d_hdr_out & 15u) || ((uintptr_t)d_perm & 3u))
        return ACE_EINVAL;
    const int G = (num_ops + 15) / 16;
    const unsigned long long blocks = ((unsigned long long)n_plans * G + 255) / 256;
    if (blocks > 0x7fffffffull) return ACE_ETOOBIG;
    ace_grid_parts(blocks, 256, [&](uint64_t first, uint32_t groups) {
        hipLaunchKernelGGL(gather_plans_kernel, dim3(groups), dim3(256), 0, (hipStream_t)stream,
                           reinterpret_cast<const ace_u4 *>(d_codes_in), reinterpret_cast<const ace_u4 *>(d_hdr_in), d_perm,
                           (unsigned long long)n_plans, G, reinterpret_cast<ace_u4 *>(d_codes_out), reinterpret_cast<ace_u4 *>(d_hdr_out),
                           (unsigned long long)first);
    });
    ACE_HIP(hipGetLastError());
    return ACE_OK;
}

int ace_pack_plans(const uint8_t *d_rows, size_t n_plans, int num_ops, const uint32_t *d_hdr, int n_mbs, int n_codes,
                   uint8_t *d_codes_out, int32_t *d_flags, void *stream) {
    if (!d_rows || !d_codes_out || n_plans == 0 || n_plans > 0x7fffffffull || num_ops <= 0 || num_ops >= (1 << 20) || (d_hdr && !d_flags) ||
        n_codes < 1 || n_codes > 8 || ((uintptr_t)d_rows & 15u) || ((uintptr_t)d_codes_out & 15u) || ((uintptr_t)d_hdr & 15u))
        return ACE_EINVAL;
    PackArgs a{d_rows, nullptr, nullptr, reinterpret_cast<ace_u4 *>(d_codes_out), reinterpret_cast<const ace_u4 *>(d_hdr), d_flags,
               (long long)n_plans, num_ops, (num_ops + 15) / 16, n_mbs, n_codes};
    ace_grid_parts((n_plans + kPackPlans - 1) / kPackPlans, kPackLanes, [&](uint64_t first, uint32_t groups) {
        hipLaunchKernelGGL(pack_plans_kernel, dim3(groups), dim3(kPackLanes), 0, (hipStream_t)stream, a, (long long)first);
    });
    ACE_HIP(hipGetLastError());
    return ACE_OK;
}

int ace_unpack_plans(const uint8_t *d_codes, size_t n_plans, int num_ops, uint8_t *d_rows_out, void *stream) {
    if (!d_codes || !d_rows_out || n_plans == 0 || n_plans > 0x7fffffffull || num_ops <= 0 || num_ops >= (1 << 20) ||
        ((uintptr_t)d_codes & 15u) || ((uintptr_t)d_rows_out & 15u))
        return ACE_EINVAL;
    PackArgs a{nullptr, d_rows_out, reinterpret_cast<const ace_u4 *>(d_codes), nullptr, nullptr, nullptr, (long long)n_plans, num_ops,
               (num_ops + 15) / 16, 0, 8};
    ace_grid_parts((n_plans + kPackPlans - 1) / kPackPlans, kPackLanes, [&](uint64_t first, uint32_t groups) {
        hipLaunchKernelGGL(unpack_plans_kernel, dim3(groups), dim3(kPackLanes), 0, (hipStream_t)stream, a, (long long)first);
    });
    ACE_HIP(hipGetLastError());
    return ACE_OK;
}

int ace_check_plans(const uint8_t *codes, const uint32_t *hdr, size_t n_plans, int num_ops, int n_mbs, int n_codes) {
    if (!codes || !hdr || num_ops <= 0 || n_codes < 1 || n_codes > 8) return ACE_EINVAL;
    return ace_check_plans_host(codes, hdr, n_plans, num_ops, n_mbs, n_codes);
}

int ace_recompute_groups(const ace_rc_tables_t *t, int n_stages, const int32_t *d_plan, const int32_t *d_lo,
                         const int32_t *d_hi, const int32_t *d_nsb, const uint32_t *d_mrow, double *d_sum_size,
                         int32_t *d_first_pos, int32_t *d_bad, void *stream) {
    if (!t || n_stages <= 0 || !d_plan || !d_lo || !d_hi || !d_nsb || !d_mrow || !d_sum_size || !d_first_pos || !d_bad ||
        !t->d_codes || !t->d_type_of_pos || !t->d_activations || !t->d_no_recompute || t->num_ops <= 0 || t->num_types <= 0 ||
        t->n_tp <= 0 || t->n_tp > 4 || (t->n_algo != 1 && t->n_algo != 2) || t->n_mbs <= 0 || t->n_mbs > 15 || t->n_plans == 0)
        return ACE_EINVAL;
    RcTables k{t->d_codes, (unsigned long long)t->n_plans, t->d_type_of_pos, t->d_activations, t->d_no_recompute,
               t->num_ops, t->num_types, t->n_mbs, t->n_tp, t->n_algo, t->n_algo == 2 ? 1 : 0};
    hipLaunchKernelGGL(rc_groups_kernel, dim3((n_stages + 127) / 128), dim3(128), 0, (hipStream_t)stream, k, n_stages,
                       d_plan, d_lo, d_hi, d_nsb, d_mrow, d_sum_size, d_first_pos, d_bad);
    ACE_HIP(hipGetLastError());
    return ACE_OK;
}

int ace_recompute_select(const ace_rc_tables_t *t, uint8_t *d_codes_rw, int n_stages, const int32_t *d_plan,
                         const int32_t *d_lo, const int32_t *d_hi, const int32_t *d_nsb, const uint32_t *d_mrow,
                         const double *d_sum_size, const int32_t *d_first_pos, uint8_t *d_recomputed, const double *d_mem,
                         double memory_limit, uint8_t *d_alive, void *stream) {
    if (!t || !d_codes_rw || n_stages <= 0 || !d_plan || !d_lo || !d_hi || !d_nsb || !d_mrow || !d_sum_size ||
        !d_first_pos || !d_recomputed || !d_mem || !d_alive || !t->d_codes || !t->d_type_of_pos || !t->d_activations ||
        !t->d_no_recompute || t->num_ops <= 0 || t->num_types <= 0 || t->n_tp <= 0 || t->n_tp > 4 ||
        (t->n_algo != 1 && t->n_algo != 2) || t->n_mbs <= 0 || t->n_mbs > 15 || t->n_plans == 0)
        return ACE_EINVAL;
    RcTables k{t->d_codes, (unsigned long long)t->n_plans, t->d_type_of_pos, t->d_activations, t->d_no_recompute,
               t->num_ops, t->num_types, t->n_mbs, t->n_tp, t->n_algo, t->n_algo == 2 ? 1 : 0};
    hipLaunchKernelGGL(rc_select_kernel, dim3((n_stages + 127) / 128), dim3(128), 0, (hipStream_t)stream, k, d_codes_rw,
                       n_stages, d_plan, d_lo, d_hi, d_nsb, d_mrow, d_sum_size, d_first_pos, d_recomputed, d_mem,
                       memory_limit, d_alive);
    ACE_HIP(hipGetLastError());
    return ACE_OK;
}

int ace_recompute_prepare(ace_handle_t *h, const int32_t *type_of_pos, const double *activations, const uint8_t *no_recompute) {
    if (!h || !type_of_pos || !activations || !no_recompute) return ACE_EINVAL;
    const int N = h->geom.N;
    if (N > kRcMaxOps || !h->d_pos_spread || h->num_types > 0xffff) return ACE_ETOOBIG;
    for (int i = 0; i < N; ++i)
        if (type_of_pos[i] < 0 || type_of_pos[i] >= h->num_types) return ACE_EINVAL;
    ACE_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&ace_rc_kernel<false>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxLds));
    ACE_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&ace_rc_kernel<true>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxLds));
    std::vector<ace_u2> pos;
    if (or_enomem([&] { return pos.resize((size_t)N), ACE_OK; })) return ACE_ENOMEM;
    const int groups = ace_rc_positions(type_of_pos, no_recompute, N, h->num_types, pos.data()), waves = ace_rc_waves(N, h->geom.G, groups, kMaxLds);
    RcShared s;
    if (ace_rc_layout(N, h->geom.G, groups, waves, nullptr, &s) > kMaxLds) return ACE_ETOOBIG;
    if (h->d_rc_pos) (void)hipFree(h->d_rc_pos);
    if (h->d_rc_act) (void)hipFree(h->d_rc_act);
    h->d_rc_pos = nullptr;
    h->d_rc_act = nullptr;
    const size_t n_act = (size_t)h->num_types * h->geom.n_mbs * h->geom.n_tp * h->geom.n_algo;
    int rc = upload((void **)&h->d_rc_pos, pos.data(), pos.size() * sizeof(ace_u2));
    if (rc == ACE_OK) rc = upload((void **)&h->d_rc_act, activations, n_act * sizeof(double));
    h->rc_groups = groups;
    h->rc_waves = waves;
    return rc;
}

int ace_recompute_batch(ace_handle_t *h, const ace_batch_t *batch, double memory_limit, double peak_backward, const uint8_t *d_status,
                        uint8_t *d_codes_out, int32_t *d_flags, void *stream) {
    if (!h || !batch || batch->d_range || batch->d_order || !d_status || !d_codes_out || !d_flags || ((uintptr_t)d_codes_out & 15u))
        return ACE_EINVAL;
    if (!h->d_rc_pos || !h->d_rc_act) return ACE_EINVAL;
    RcArgs a;
    // (the scoring outputs are not written: any pointer will do)
    double *unused = h->d_rc_act;
    int rc = fill_args(h, batch, memory_limit, 0, unused, unused, d_codes_out, nullptr, nullptr, &a.k);
    if (rc) return rc;
    a.pos = h->d_rc_pos;
    a.act = h->d_rc_act;
    a.status = d_status;
    a.codes_out = reinterpret_cast<ace_u4 *>(d_codes_out);
    a.flags = d_flags;
    a.limit = memory_limit;
    a.peak_backward = peak_backward;
    RcShared s;
    a.groups = h->rc_groups;
    a.waves = h->rc_waves;
    const uint32_t lds = ace_rc_layout(a, nullptr, &s);
    const auto kernel = a.k.g.flags & ACE_F_COLLECTIVE_MEM ? ace_rc_kernel<true> : ace_rc_kernel<false>;
    ace_grid_parts((uint64_t)a.k.g.P, 64u * (uint32_t)a.waves, [&](uint64_t first, uint32_t groups) {
        hipLaunchKernelGGL(kernel, dim3(groups), dim3(64u * (uint32_t)a.waves), lds, (hipStream_t)stream, a, (long long)first);
    });
    ACE_HIP(hipGetLastError());
    return ACE_OK;
}

int ace_keyset_create(ace_keyset_t **out) {
    if (!out) return ACE_EINVAL;
    try {
        *out = reinterpret_cast<ace_keyset_t *>(new AceKeySet);
    } catch (const std::bad_alloc &) {
        *out = nullptr;
        return ACE_ENOMEM;
    }
    return ACE_OK;
}

static AceKeySet *key_set(ace_keyset_t *s) { return reinterpret_cast<AceKeySet *>(s); }
static const AceKeySet *key_set(const ace_keyset_t *s) { return reinterpret_cast<const AceKeySet *>(s); }

void ace_keyset_destroy(ace_keyset_t *s) { delete key_set(s); }

size_t ace_keyset_size(const ace_keyset_t *s) { return s ? key_set(s)->size() : 0; }

int ace_keyset_add(ace_keyset_t *s, const uint64_t *keys, size_t n) {
    if (!s || (n && !keys)) return ACE_EINVAL;
    try {
        AceKeySet *set = key_set(s);
        ace_each_key(keys, n, &set, 1, [&](size_t, const AceKey &k) { set->add(k); });
    } catch (const std::bad_alloc &) {
        return ACE_ENOMEM;
    }
    return ACE_OK;
}

// the sets behind the handles (at most four), or 0
static int key_sets(const ace_keyset_t *const *sets, int n_sets, const AceKeySet **out) {
    if (n_sets < 0 || n_sets > 4 || (n_sets && !sets)) return 0;
    for (int i = 0; i < n_sets; ++i) {
        if (!sets[i]) return 0;
        out[i] = key_set(sets[i]);
    }
    return 1;
}

int ace_keyset_unseen(const ace_keyset_t *const *sets, int n_sets, const uint64_t *keys, size_t n, uint8_t *mask) {
    const AceKeySet *in[5];
    if (!key_sets(sets, n_sets, in) || (n && (!keys || !mask))) return ACE_EINVAL;
    try {
        AceKeySet here;
        here.reserve(n);
        in[n_sets] = &here;
        ace_each_key(keys, n, in, n_sets + 1, [&](size_t i, const AceKey &k) {
            bool fresh = true;
            for (int j = 0; j < n_sets && fresh; ++j) fresh = !in[j]->has(k);
            mask[i] = (uint8_t)(fresh && here.add(k));
        });
    } catch (const std::bad_alloc &) {
        return ACE_ENOMEM;
    }
    return ACE_OK;
}

int ace_keyset_claim(ace_keyset_t *const *sets, int n_sets, const uint64_t *keys, size_t n, uint8_t *mask) {
    const AceKeySet *in[4];
    if (n_sets < 1 || !key_sets(sets, n_sets, in) || (n && (!keys || !mask))) return ACE_EINVAL;
    try {
        AceKeySet *set = key_set(sets[0]);
        ace_each_key(keys, n, in, n_sets, [&](size_t i, const AceKey &k) {
            bool fresh = true;
            for (int j = 1; j < n_sets && fresh; ++j) fresh = !in[j]->has(k);
            mask[i] = (uint8_t)(fresh && set->add(k));
        });
    } catch (const std::bad_alloc &) {
        return ACE_ENOMEM;
    }
    return ACE_OK;
}

int ace_keyset_move(ace_keyset_t *to, ace_keyset_t *from) {
    if (!to || !from || to == from) return ACE_EINVAL;
    try {
        AceKeySet *t = key_set(to);
        std::vector<uint64_t> keys;
        keys.reserve(2 * key_set(from)->size());
        key_set(from)->each([&](const AceKey &k) { keys.push_back(k.a); keys.push_back(k.b); });
        t->reserve(t->size() + keys.size() / 2);
        ace_each_key(keys.data(), keys.size() / 2, &t, 1, [&](size_t, const AceKey &k) { t->add(k); });
        key_set(from)->clear();
    } catch (const std::bad_alloc &) {
        return ACE_ENOMEM;
    }
    return ACE_OK;
}

int ace_keyset_keys(const ace_keyset_t *s, uint64_t *keys_out) {
    if (!s || !keys_out) return ACE_EINVAL;
    key_set(s)->each([&](const AceKey &k) { *keys_out++ = k.a; *keys_out++ = k.b; });
    return ACE_OK;
}

static bool moves_args(const uint8_t *codes, const uint32_t *hdr, int num_ops, int n_algo, int n_tp, int n_mbs, const uint32_t *stage_lut,
                       int gpus_per_node, const ace_move_draws_t *draws, uint32_t *moves_out, uint8_t *t_codes_out, uint32_t *t_hdr_out,
                       int *n_templates_out) {
    return codes && hdr && stage_lut && draws && moves_out && t_codes_out && t_hdr_out && n_templates_out && num_ops > 0 &&
           num_ops < 65536 && (n_algo == 1 || n_algo == 2) && n_tp > 0 && n_tp <= 4 && n_mbs > 0 && gpus_per_node > 0;
}

int ace_build_moves(const uint8_t *codes, const uint32_t *hdr, int num_ops, int n_algo, int n_tp, int n_mbs, const uint32_t *stage_lut,
                    int gpus_per_node, const ace_move_draws_t *draws, uint32_t *moves_out, uint8_t *t_codes_out, uint32_t *t_hdr_out,
                    int max_templates, int *n_templates_out) {
    if (!moves_args(codes, hdr, num_ops, n_algo, n_tp, n_mbs, stage_lut, gpus_per_node, draws, moves_out, t_codes_out, t_hdr_out, n_templates_out))
        return ACE_EINVAL;
    return or_enomem([&] {
        return ace_build_moves_body(codes, hdr, num_ops, n_algo, n_tp, n_mbs, stage_lut, gpus_per_node, *draws, moves_out, t_codes_out,
                                    t_hdr_out, max_templates, n_templates_out);
    });
}

int ace_new_moves(const uint8_t *codes, const uint32_t *hdr, int num_ops, int n_algo, int n_tp, int n_mbs, const uint32_t *stage_lut,
                  int gpus_per_node, const ace_move_draws_t *draws, ace_keyset_t *const *sets, int n_sets, uint32_t *moves_out,
                  size_t *n_moves_out, uint8_t *t_codes_out, uint32_t *t_hdr_out, int max_templates, int *n_templates_out) {
    const AceKeySet *in[4];
    if (!moves_args(codes, hdr, num_ops, n_algo, n_tp, n_mbs, stage_lut, gpus_per_node, draws, moves_out, t_codes_out, t_hdr_out, n_templates_out) ||
        !n_moves_out || !key_sets(sets, n_sets, in))
        return ACE_EINVAL;
    try {
        AceKeySet *s[4];
        for (int i = 0; i < n_sets; ++i) s[i] = key_set(sets[i]);
        return ace_new_moves_body(codes, hdr, num_ops, n_algo, n_tp, n_mbs, stage_lut, gpus_per_node, *draws, s, n_sets, moves_out, n_moves_out,
                                  t_codes_out, t_hdr_out, max_templates, n_templates_out);
    } catch (const std::bad_alloc &) {
        return ACE_ENOMEM;
    }
}

static int search_step(ace_handle_t *h, const uint8_t *codes, const uint32_t *hdr, const uint32_t *stage_lut, int gpus_per_node,
                       const ace_move_draws_t *draws, ace_keyset_t *const *sets, int n_sets, double memory_limit, int strict,
                       uint8_t *codes_out, uint32_t *hdr_out, ace_step_result_t *res, hipStream_t s) {
    const AceGeom &g = h->geom;
    const size_t N = (size_t)g.N, G = (size_t)g.G, n = draws->n;
    const int S = (int)(hdr[0] & 0xffu), cap = 3 + S * (S > 0 ? S - 1 : 0);
    if (!h->step) h->step = new StepBuffers();
    StepBuffers &b = *h->step;
    b.t_codes.resize((size_t)cap * N);
    b.t_hdr.resize((size_t)cap * 4);
    // page-locked: [StepOut][moves][template headers][template code rows, padded]
    const size_t host_need = 64 + 16 * n + (size_t)cap * 16 * (1 + G);
    if (b.host_bytes < host_need) {
        if (b.host) ACE_HIP(hipHostFree(b.host));
        b.host = nullptr;
        b.host_bytes = 0;
        ACE_HIP(hipHostMalloc((void **)&b.host, host_need, hipHostMallocDefault));
        b.host_bytes = host_need;
    }
    unsigned char *up = b.host + 64;
    uint32_t *moves = reinterpret_cast<uint32_t *>(up);
    int T = 0;
    size_t m = 0;
    int rc = ace_new_moves(codes, hdr, g.N, g.n_algo, g.n_tp, g.n_mbs, stage_lut, gpus_per_node, draws, sets, n_sets, moves, &m,
                           b.t_codes.data(), b.t_hdr.data(), cap, &T);
    if (rc) return rc;
    res->n_moves = m;
    if (!m) return ACE_OK;
    const size_t off_hdr = 16 * m, off_codes = off_hdr + 16 * (size_t)T, up_bytes = off_codes + (size_t)T * G * 16;
    memcpy(up + off_hdr, b.t_hdr.data(), 16 * (size_t)T);
    memset(up + off_codes, 0, (size_t)T * G * 16);
    for (int t = 0; t < T; ++t) memcpy(up + off_codes + (size_t)t * G * 16, b.t_codes.data() + (size_t)t * N, N);
    // device: what went up, the plans, their scores, the pick
    size_t at = 0;
    auto take = [&](size_t bytes) { const size_t o = at; at += (bytes + 255) & ~(size_t)255; return o; };
    const size_t ws = ace_topk_workspace_bytes(m, 1);
    const size_t o_up = take(up_bytes), o_codes = take(G * m * 16), o_hdr = take(16 * m), o_it = take(8 * m), o_pk = take(8 * m),
                 o_fe = take(m), o_top = take(24), o_ws = take(ws);
    if (b.dev_bytes < at) {
        if (b.dev) ACE_HIP(hipFree(b.dev));
        b.dev = nullptr;
        b.dev_bytes = 0;
        ACE_HIP(hipMalloc((void **)&b.dev, at + at / 4));
        b.dev_bytes = at + at / 4;
    }
    unsigned char *d = b.dev;
    ACE_HIP(hipMemcpyAsync(d + o_up, up, up_bytes, hipMemcpyHostToDevice, s));
    double *it = reinterpret_cast<double *>(d + o_it), *pk = reinterpret_cast<double *>(d + o_pk), *val = reinterpret_cast<double *>(d + o_top + 8);
    int64_t *idx = reinterpret_cast<int64_t *>(d + o_top);
    int32_t *count = reinterpret_cast<int32_t *>(d + o_top + 16);
    const ace_batch_t batch{d + o_codes, reinterpret_cast<const uint32_t *>(d + o_hdr), nullptr, m, nullptr};
    if ((rc = ace_apply_moves(d + o_up + off_codes, reinterpret_cast<const uint32_t *>(d + o_up + off_hdr), T,
                              reinterpret_cast<const uint32_t *>(d + o_up), m, g.N, g.n_algo, d + o_codes,
                              reinterpret_cast<uint32_t *>(d + o_hdr), nullptr, s)) ||
        (rc = ace_score_batch(h, &batch, memory_limit, strict, it, pk, d + o_fe, nullptr, nullptr, s)) ||
        (rc = ace_topk(h, it, d + o_fe, m, 1, idx, val, count, d + o_ws, ws, s)))
        return rc;
    StepOut *out = reinterpret_cast<StepOut *>(b.host);
    hipLaunchKernelGGL(step_out_kernel, dim3(1), dim3(1), 0, s, (const long long *)idx, val, count, pk, out);
    ACE_HIP(hipGetLastError());
    ACE_HIP(hipStreamSynchronize(s));
    if (out->count > 0 && out->idx >= 0 && (size_t)out->idx < m) {
        const uint32_t *mv = moves + 4 * out->idx;
        const size_t t = mv[0] & 0xffffu;
        memcpy(codes_out, b.t_codes.data() + t * N, N);
        memcpy(hdr_out, b.t_hdr.data() + 4 * t, 16);
        ace_apply_move(mv, g.N, g.n_algo, codes_out);
        res->found = 1;
        res->iter_ms = out->iter_ms;
        res->peak_mb = out->peak_mb;
    }
    return ACE_OK;
}

int ace_search_step(ace_handle_t *h, const uint8_t *codes, const uint32_t *hdr, const uint32_t *stage_lut, int gpus_per_node,
                    const ace_move_draws_t *draws, ace_keyset_t *const *sets, int n_sets, double memory_limit, int strict,
                    uint8_t *codes_out, uint32_t *hdr_out, ace_step_result_t *result, void *stream) {
    if (!h || !codes || !hdr || !stage_lut || !draws || !codes_out || !hdr_out || !result || draws->n == 0 || draws->n > 0x7fffffffull ||
        h->geom.N >= 65536)
        return ACE_EINVAL;
    *result = ace_step_result_t{0, 0, 0.0, 0.0};
    std::lock_guard<std::mutex> lock(h->host_calls);
    int dev = -1;
    ACE_HIP(hipGetDevice(&dev));
    if (dev != h->device) ACE_HIP(hipSetDevice(h->device));
    int rc;
    try {
        rc = search_step(h, codes, hdr, stage_lut, gpus_per_node, draws, sets, n_sets, memory_limit, strict, codes_out, hdr_out, result,
                         (hipStream_t)stream);
    } catch (const std::bad_alloc &) {
        rc = ACE_ENOMEM;
    }
    if (dev != h->device) ACE_HIP(hipSetDevice(dev));
    return rc;
}

}  // extern "C"
