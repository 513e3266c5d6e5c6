// Host side of the neighbour moves: descriptors and templates from drawn choices (neighbours._draw_moves).  One pass per
// kind over a few thousand rows, 40 us for 16,384 neighbours of a 16-stage plan, where the same selection in numpy took 0.7 ms.
#pragma once
#include <string.h>

#include <algorithm>
#include <vector>

#include "ace_eval.h"

// The header of a plan of S stages of 2^glog devices: sizes, and which stage boundaries fall on node boundaries.
inline void ace_set_header(uint32_t *h, int S, uint32_t bidx, const int *glogs, int gpus_per_node) {
    uint64_t sizes = 0;
    uint32_t cross = 0;
    int64_t till = 0;
    for (int s = 0; s < S; ++s) {
        sizes |= (uint64_t)glogs[s] << (4 * s);
        if (till % gpus_per_node == 0 && till > 0) cross |= 1u << s;
        till += (int64_t)1 << glogs[s];
        if (till % gpus_per_node == 0) cross |= 1u << (16 + s);
    }
    h[0] = (uint32_t)S | (bidx << 8);
    h[1] = (uint32_t)sizes;
    h[2] = (uint32_t)(sizes >> 32);
    h[3] = cross;
}

inline int ace_build_moves_body(const uint8_t *codes, const uint32_t *hdr, int N, int A, int n_tp, int n_mbs, const uint32_t *stage_lut,
                                int gpus_per_node, const ace_move_draws_t &d, uint32_t *moves, uint8_t *t_codes, uint32_t *t_hdr,
                                int max_templates, int *n_templates) {
    const int S = (int)(hdr[0] & 0xffu);
    const uint32_t bidx = (hdr[0] >> 8) & 0xffu;
    if (S < 1 || S > ACE_MAX_STAGES || bidx >= (uint32_t)n_mbs || max_templates < 3 + S * (S - 1)) return ACE_EINVAL;
    // the tp indices a stage of 2^g devices may use, a bit each, by [micro-batch index * 16 + g]
    std::vector<uint8_t> allowed((size_t)n_mbs * 16);
    for (size_t j = 0; j < allowed.size(); ++j)
        for (int t = 0; t < n_tp; ++t)
            if (((stage_lut[j] >> (16 + 4 * t)) & 15u) != 15u) allowed[j] |= (uint8_t)(1u << t);
    const uint64_t sizes = (uint64_t)hdr[1] | ((uint64_t)hdr[2] << 32);
    const int a_shift = A == 2 ? 1 : 0;
    int glogs[ACE_MAX_STAGES], lo[ACE_MAX_STAGES + 1];
    uint32_t present[ACE_MAX_STAGES] = {0};               // tp indices in use, a bit each
    int found = 0;
    for (int s = 0; s < S; ++s) glogs[s] = (int)(sizes >> (4 * s)) & 15;
    for (int i = 0; i < N; ++i) {
        if (codes[i] & 16) {
            if (found == S) return ACE_EINVAL;
            lo[found++] = i;
        }
        if (!found) return ACE_EINVAL;
        present[found - 1] |= 1u << ((codes[i] & 7) >> a_shift);
    }
    if (found != S) return ACE_EINVAL;
    lo[S] = N;
    for (int k = 0; k < 6; ++k)
        for (size_t r = 0; r < d.count[k]; ++r)
            if ((uint64_t)d.rows[k][r] >= d.n) return ACE_EINVAL;
    memset(moves, 0, d.n * 16);
    memcpy(t_codes, codes, (size_t)N);
    memcpy(t_hdr, hdr, 16);
    int T = 1;
    auto edit = [&](int64_t row, uint32_t op, uint32_t p0, uint32_t p1) {
        uint32_t *m = moves + 4 * row;
        m[0] = op << 16;
        m[1] = p0;
        m[2] = p1;
    };
    // op migration: the ops that change stage take the tp of the op they now follow / precede in the receiving stage
    for (size_t r = 0; r < d.count[0]; ++r) {
        const int64_t j = d.x[0][r], by = d.y[0][r];
        if (j < 1 || j >= S) return ACE_EINVAL;
        const int64_t cut = lo[j], to = cut + by;
        if (to > lo[j - 1] && to < lo[j + 1])
            edit(d.rows[0][r], 1, (uint32_t)cut | ((uint32_t)to << 16), (uint32_t)(codes[by > 0 ? cut - 1 : cut] & 7) >> a_shift);
    }
    // tp <-> dp: legal if every tp in use has a legal target
    for (size_t r = 0; r < d.count[1]; ++r) {
        const int64_t s = d.x[1][r];
        if (s < 0 || s >= S) return ACE_EINVAL;
        const bool up = d.y[1][r] > 0;
        const uint32_t want = up ? present[s] << 1 : present[s] >> 1;
        if (!(want & ~(uint32_t)allowed[bidx * 16 + glogs[s]]) && (up || !(present[s] & 1u)))
            edit(d.rows[1][r], 2, (uint32_t)lo[s] | ((uint32_t)lo[s + 1] << 16), up ? 1u : 0u);
    }
    // micro-batch size: a template of its own, if every op stays on the profiled grid
    for (int up = 1; up >= 0; --up) {
        const int b2 = (int)bidx + (up ? 1 : -1);
        bool any = false;
        for (size_t r = 0; r < d.count[2]; ++r) any = any || (d.x[2][r] > 0) == (up == 1);
        bool fits = any && b2 >= 0 && b2 < n_mbs;
        for (int s = 0; s < S && fits; ++s) fits = !(present[s] & ~(uint32_t)allowed[b2 * 16 + glogs[s]]);
        if (!fits) continue;
        memcpy(t_codes + (size_t)T * N, codes, (size_t)N);
        memcpy(t_hdr + 4 * T, hdr, 16);
        t_hdr[4 * T] = (uint32_t)S | ((uint32_t)b2 << 8);
        for (size_t r = 0; r < d.count[2]; ++r)
            if ((d.x[2][r] > 0) == (up == 1)) moves[4 * d.rows[2][r]] = (uint32_t)T;
        ++T;
    }
    for (size_t r = 0; r < d.count[3]; ++r) {
        const int64_t first = d.x[3][r], end = std::min<int64_t>(N, first + d.y[3][r]);
        if (first < 0 || first >= N) return ACE_EINVAL;
        edit(d.rows[3][r], 3, (uint32_t)first | ((uint32_t)end << 16), 0);
    }
    for (size_t r = 0; r < d.count[4]; ++r) edit(d.rows[4][r], 4, (uint32_t)d.x[4][r], 0);
    // devices: half of stage a's go to a stage b that has exactly that many; a template per (a, b), in order
    int of_pair[ACE_MAX_STAGES * ACE_MAX_STAGES];
    std::fill(of_pair, of_pair + ACE_MAX_STAGES * ACE_MAX_STAGES, 0);
    for (size_t r = 0; r < d.count[5]; ++r) {
        if (d.x[5][r] < 0 || d.x[5][r] >= S || d.y[5][r] < 0 || d.y[5][r] >= S) return ACE_EINVAL;
        of_pair[d.x[5][r] * ACE_MAX_STAGES + d.y[5][r]] = -1;
    }
    for (int a = 0; a < S; ++a)
        for (int b = 0; b < S; ++b) {
            int &t = of_pair[a * ACE_MAX_STAGES + b];
            if (t == 0) continue;
            t = 0;
            if (a == b || glogs[a] - 1 != glogs[b]) continue;
            int g2[ACE_MAX_STAGES];
            std::copy(glogs, glogs + S, g2);
            --g2[a];
            ++g2[b];
            uint8_t *row = t_codes + (size_t)T * N;
            memcpy(row, codes, (size_t)N);
            bool good = true;
            for (int st : {a, b}) {
                const uint32_t ok = allowed[bidx * 16 + g2[st]];
                if (!ok) { good = false; break; }
                const int least = __builtin_ctz(ok), most = 31 - __builtin_clz(ok);
                for (int i = lo[st]; i < lo[st + 1] && good; ++i) {
                    int tp = (codes[i] & 7) >> a_shift;
                    tp = tp < least ? least : (tp > most ? most : tp);
                    good = (ok >> tp) & 1u;
                    row[i] = (uint8_t)((codes[i] & 0xF8) | (tp * A + (codes[i] & (A - 1))));
                }
                if (!good) break;
            }
            if (!good) continue;
            ace_set_header(t_hdr + 4 * T, S, bidx, g2, gpus_per_node);
            t = T++;
        }
    for (size_t r = 0; r < d.count[5]; ++r) moves[4 * d.rows[5][r]] = (uint32_t)of_pair[d.x[5][r] * ACE_MAX_STAGES + d.y[5][r]];
    *n_templates = T;
    return ACE_OK;
}
