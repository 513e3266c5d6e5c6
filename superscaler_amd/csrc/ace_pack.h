// Plans between the host's layout (one row of N code bytes per plan) and the kernels' ([16-op group][plan][16 bytes]), and
// the structural check of a batch, which rides along: it reads every byte once and so does this.
//
// A workgroup moves 32 plans, 64 groups at a time, through LDS: rows come in as 16-byte pieces along a row, go out as 512
// consecutive bytes per group (and the other way round).  16,384 plans of 523 ops (8.6 MB, read once and written once) take 10 to
// 11 us, the phases' latencies; 1,048,576 plans 199 us, 5.6 TB/s read and written.  Padding and permuting the small batch as two tensor operations
// took 2 x 13 us and the check on the host 3.3 ms.
#pragma once
#include "ace_plan_state.h"

constexpr int kPackPlans = 32, kPackGroups = 64, kPackLanes = 256;
constexpr int kPackPitch = kPackGroups * 16 + 20;      // bytes from row to row: room for a misaligned start; an odd number of words

struct PackArgs {
    const uint8_t *rows_in;     // [P][N] (pack)
    uint8_t *rows_out;          // [P][N] (unpack)
    const ace_u4 *codes_in;     // [G][P] (unpack)
    ace_u4 *codes_out;          // [G][P] (pack)
    const ace_u4 *hdr;          // [P], for the check (else null)
    int32_t *flags;             // the check's findings, bits PACK_*
    long long P;
    int N, G, n_mbs, C;
};
// in the order in which plan.validate_batch names them
enum { PACK_STAGES = 1, PACK_BITS = 2, PACK_FIRST = 4, PACK_MBS = 8, PACK_CODE = 16 };

struct PackShared { uint32_t rows[kPackPlans * kPackPitch / 4]; uint32_t count[kPackPlans]; uint32_t bad; };
static_assert(kPackPitch % 8 == 4, "an odd number of words");

#ifdef ACE_HOST_EMU
#define PACK_PHASE(...) for (int tid = 0; tid < kPackLanes; ++tid) { __VA_ARGS__; }
#define PACK_ADD(p, v) (*(p) += (v))
#define PACK_OR(p, v) (*(p) |= (v))
#else
#define PACK_PHASE(...) { __VA_ARGS__; } __syncthreads()
#define PACK_ADD(p, v) atomicAdd((p), (v))
#define PACK_OR(p, v) atomicOr((p), (v))
#endif

// the 32-bit word at byte offset `at` of a row in LDS
ACE_HD uint32_t pack_word(const uint32_t *row, uint32_t at) {
    const uint32_t w = at >> 2, s = (at & 3u) * 8u;
    return (uint32_t)((((uint64_t)row[w + 1] << 32) | row[w]) >> s);
}

ACE_HD void pack_rows_in(const PackArgs &a, PackShared &s, long long p0, int n_p, int g0, int n_g, int tid) {
    constexpr int kStep = kPackLanes / 64, kRows = kPackPlans / kStep;
    const long long total = a.P * (long long)a.N;
    const int q = tid & 63;
    auto place = [&](int r, int at_q) { return (((p0 + r) * a.N + g0 * 16) & ~15ll) + at_q * 16; };
    auto piece = [&](int r, int at_q) { return *reinterpret_cast<const ace_u4 *>(a.rows_in + place(r, at_q)); };
    auto has = [&](int r, int at_q) {
        const int bytes = (a.N - g0 * 16 < n_g * 16 ? a.N - g0 * 16 : n_g * 16) + (int)(((p0 + r) * a.N + g0 * 16) & 15ll);
        return r < n_p && at_q * 16 < bytes && place(r, at_q) + 16 <= total;
    };
    auto put = [&](int r, int at_q, const ace_u4 &x) {
        uint32_t *row = s.rows + r * (kPackPitch / 4) + 4 * at_q;
        row[0] = x.x; row[1] = x.y; row[2] = x.z; row[3] = x.w;
    };
    ace_u4 v[kRows];
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
        v[i] = ace_u4{0u, 0u, 0u, 0u};
        if (has((tid >> 6) + i * kStep, q)) v[i] = piece((tid >> 6) + i * kStep, q);
    }
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
        const int r = (tid >> 6) + i * kStep;
        if (has(r, q)) put(r, q, v[i]);
        if (q == 0 && has(r, 64)) put(r, 64, piece(r, 64));
    }
    // the batch's last bytes, where less than a piece is left
    if (p0 + n_p < a.P || tid != 0) return;
    const long long at = total & ~15ll;
    uint32_t w[4] = {0u, 0u, 0u, 0u};
    for (int k = 0; at + k < total; ++k) w[k >> 2] |= (uint32_t)a.rows_in[at + k] << (8 * (k & 3));
#pragma unroll 1
    for (int r = 0; r < n_p; ++r) {
        const long long base = place(r, 0);
        if (at < total && at >= base && at - base <= 64 * 16) put(r, (int)((at - base) >> 4), ace_u4{w[0], w[1], w[2], w[3]});
    }
}

ACE_HD void pack_groups_in(const PackArgs &a, PackShared &s, long long p0, int n_p, int g0, int n_g, int tid) {
    for (int k0 = tid; k0 < kPackPlans * n_g; k0 += 8 * kPackLanes) {
        ace_u4 v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int k = k0 + i * kPackLanes, r = k & (kPackPlans - 1), g = k / kPackPlans;
            v[i] = ace_u4{0u, 0u, 0u, 0u};
            if (g < n_g && r < n_p) v[i] = a.codes_in[(size_t)(g0 + g) * a.P + p0 + r];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int k = k0 + i * kPackLanes, r = k & (kPackPlans - 1), g = k / kPackPlans;
            if (g >= n_g || r >= n_p) continue;
            uint32_t *row = s.rows + r * (kPackPitch / 4) + 4 * g;
            row[0] = v[i].x; row[1] = v[i].y; row[2] = v[i].z; row[3] = v[i].w;
        }
    }
}

ACE_HD void ace_pack_body(const PackArgs &a, PackShared &s, int tid_, long long block) {
#ifdef ACE_HOST_EMU
    (void)tid_;
#else
    const int tid = tid_;
#endif
    const long long p0 = block * kPackPlans;
    const int n_p = (int)(a.P - p0 < kPackPlans ? a.P - p0 : kPackPlans);
    PACK_PHASE(
        if (tid < kPackPlans) s.count[tid] = 0u;
        if (tid == 0) s.bad = 0u);
    for (int g0 = 0; g0 < a.G; g0 += kPackGroups) {
        const int n_g = a.G - g0 < kPackGroups ? a.G - g0 : kPackGroups;
        // a wavefront per row: aligned 16-byte pieces from the one that holds the segment's first byte on, a piece per lane (and one
        // more where a full segment starts misaligned).  All of a wavefront's rows are asked for before the first one is put in
        // LDS: one trip to memory instead of eight.  Plans of 523 ops, us: 3,001 8.9 -> 8.0, 16,384 12.5 -> 10.7, 1,048,576
        // 320 -> 199
        PACK_PHASE(pack_rows_in(a, s, p0, n_p, g0, n_g, tid));
        PACK_PHASE(
            for (int k = tid; k < kPackPlans * n_g; k += kPackLanes) {
                const int r = k & (kPackPlans - 1);
                const int g = k / kPackPlans;
                if (r >= n_p) continue;
                const long long from = (p0 + r) * a.N + g0 * 16;
                const uint32_t *row = s.rows + r * (kPackPitch / 4);
                uint32_t w[4];
                uint32_t bits = 0;
                uint32_t over = 0;
                for (int j = 0; j < 4; ++j) {
                    const int left = a.N - ((g0 + g) * 16 + 4 * j);
                    const uint32_t m = left >= 4 ? 0xffffffffu : (left <= 0 ? 0u : ((1u << (8 * left)) - 1u));
                    w[j] = m ? pack_word(row, (uint32_t)(from & 15) + (uint32_t)(g * 16 + 4 * j)) & m : 0u;
                    bits += (uint32_t)__builtin_popcount(w[j] & 0x10101010u);
                    over |= ((w[j] & 0x07070707u) + (uint32_t)(8 - a.C) * 0x01010101u) & 0x08080808u & m;
                }
                a.codes_out[(size_t)(g0 + g) * a.P + p0 + r] = ace_u4{w[0], w[1], w[2], w[3]};
                if (a.hdr) {
                    if (bits) PACK_ADD(&s.count[r], bits);
                    if (over) PACK_OR(&s.bad, (uint32_t)PACK_CODE);
                    if (g0 + g == 0 && !(w[0] & 0x10u)) PACK_OR(&s.bad, (uint32_t)PACK_FIRST);
                }
            });
    }
    if (!a.hdr) return;
    PACK_PHASE(
        if (tid < n_p) {
            const uint32_t h = a.hdr[p0 + tid].x;
            const uint32_t S = h & 0xffu;
            const uint32_t bad = (S < 1u || S > (uint32_t)ACE_MAX_STAGES ? PACK_STAGES : 0u) | (s.count[tid] != S ? PACK_BITS : 0u) |
                                 (((h >> 8) & 0xffu) >= (uint32_t)a.n_mbs ? PACK_MBS : 0u);
            if (bad) PACK_OR(&s.bad, bad);
        });
    PACK_PHASE(if (tid == 0 && s.bad) PACK_OR(a.flags, (int32_t)s.bad));
}

ACE_HD void ace_unpack_body(const PackArgs &a, PackShared &s, int tid_, long long block) {
#ifdef ACE_HOST_EMU
    (void)tid_;
#else
    const int tid = tid_;
#endif
    const long long p0 = block * kPackPlans;
    const int n_p = (int)(a.P - p0 < kPackPlans ? a.P - p0 : kPackPlans);
    for (int g0 = 0; g0 < a.G; g0 += kPackGroups) {
        const int n_g = a.G - g0 < kPackGroups ? a.G - g0 : kPackGroups;
        // (eight loads of a lane in flight, 16-byte stores below: 16,384 plans 10.9 -> 10.4 us)
        PACK_PHASE(pack_groups_in(a, s, p0, n_p, g0, n_g, tid));
        // a wavefront per row: the aligned 16-byte pieces that the segment covers, a lane each, its ends byte by byte
        PACK_PHASE(
            for (int r = tid >> 6; r < n_p; r += kPackLanes / 64) {
                const long long from = (p0 + r) * a.N + g0 * 16;
                const int bytes = a.N - g0 * 16 < n_g * 16 ? a.N - g0 * 16 : n_g * 16;
                const int lead = (int)(-from & 15) < bytes ? (int)(-from & 15) : bytes;
                const uint32_t *row = s.rows + r * (kPackPitch / 4);
                const int l = tid & 63;
                const int pieces = (bytes - lead) >> 4;
                const int tail = lead + 16 * pieces;
                if (l < pieces) {
                    const uint32_t at = (uint32_t)(lead + 16 * l);
                    *reinterpret_cast<ace_u4 *>(a.rows_out + from + at) = ace_u4{pack_word(row, at), pack_word(row, at + 4u), pack_word(row, at + 8u), pack_word(row, at + 12u)};
                }
                if (l < lead) a.rows_out[from + l] = (uint8_t)pack_word(row, (uint32_t)l);
                if (l >= 16 && tail + l - 16 < bytes) a.rows_out[from + tail + l - 16] = (uint8_t)pack_word(row, (uint32_t)(tail + l - 16));
            });
    }
}

// The same check of a batch in host memory: the findings as PACK_* bits.
inline int ace_check_plans_host(const uint8_t *codes, const uint32_t *hdr, size_t P, int N, int n_mbs, int C) {
    int bad = 0;
    const uint64_t ones = 0x0101010101010101ull, up = (uint64_t)(8 - C) * ones;
    for (size_t p = 0; p < P; ++p) {
        const uint8_t *c = codes + p * (size_t)N;
        uint32_t count = 0;
        uint64_t over = 0;
        int i = 0;
        while (i + 8 <= N) {
            uint64_t bits = 0;                                     // a count per byte: at most 255 rounds
            for (int k = 0; k < 255 && i + 8 <= N; ++k, i += 8) {
                uint64_t w;
                __builtin_memcpy(&w, c + i, 8);
                bits += (w >> 4) & ones;
                over |= ((w & 7 * ones) + up) & 8 * ones;
            }
            count += (uint32_t)(((bits & 0x00ff00ff00ff00ffull) * 0x0001000100010001ull) >> 48) +
                     (uint32_t)((((bits >> 8) & 0x00ff00ff00ff00ffull) * 0x0001000100010001ull) >> 48);
        }
        for (; i < N; ++i) {
            count += (c[i] >> 4) & 1u;
            over |= (c[i] & 7) >= C;
        }
        const uint32_t S = hdr[4 * p] & 0xffu;
        bad |= (S < 1u || S > (uint32_t)ACE_MAX_STAGES ? PACK_STAGES : 0) | (count != S ? PACK_BITS : 0) | (c[0] & 16 ? 0 : PACK_FIRST) |
               (((hdr[4 * p] >> 8) & 0xffu) >= (uint32_t)n_mbs ? PACK_MBS : 0) | (over ? PACK_CODE : 0);
    }
    return bad;
}
