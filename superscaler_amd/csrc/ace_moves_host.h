// Host side of the neighbour moves: descriptors and templates from drawn choices (neighbours._draw_moves).  One pass per
// kind over a few thousand rows, 40 us for 16,384 neighbours of a 16-stage plan, where the same selection in numpy took 0.7 ms.
#pragma once
#include <string.h>

#include <algorithm>
#include <vector>

#include "ace_edit_kernels.h"
#include "ace_eval.h"
#include "ace_keyset.h"

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

// `first` (may be null; else zeros): per row 1 if no earlier row has the same descriptor -- of recompute runs, as far as a bit
// per possible run tells.
inline int ace_build_moves_body(const uint8_t *codes, const uint32_t *hdr, int N, int A, int n_tp, int n_mbs, const uint32_t *stage_lut,
                                int gpus_per_node, const ace_move_draws_t &d, uint32_t *moves, uint8_t *t_codes, uint32_t *t_hdr,
                                int max_templates, int *n_templates, uint8_t *first = nullptr) {
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
    constexpr int kRuns = 16;                             // recompute runs below this length have a bit each
    std::vector<uint64_t> bits(first ? ((size_t)N * (S + kRuns + 1) >> 6) + 2 : 0);
    auto fresh = [&](size_t i) {
        const uint64_t b = 1ull << (i & 63);
        const bool was = (bits[i >> 6] & b) != 0;
        bits[i >> 6] |= b;
        return (uint8_t)!was;
    };
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
        if (to > lo[j - 1] && to < lo[j + 1]) {
            edit(d.rows[0][r], 1, (uint32_t)cut | ((uint32_t)to << 16), (uint32_t)(codes[by > 0 ? cut - 1 : cut] & 7) >> a_shift);
            if (first) first[d.rows[0][r]] = fresh((size_t)j * N + (size_t)to);
        }
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
    if (first) {
        uint8_t seen[2 * ACE_MAX_STAGES] = {0};
        for (size_t r = 0; r < d.count[1]; ++r) {
            uint8_t &was = seen[2 * d.x[1][r] + (d.y[1][r] > 0)];
            first[d.rows[1][r]] = was ^ 1u;
            was = 1;
        }
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
        const int64_t at = d.x[3][r], end = std::min<int64_t>(N, at + d.y[3][r]);
        if (at < 0 || at >= N) return ACE_EINVAL;
        edit(d.rows[3][r], 3, (uint32_t)at | ((uint32_t)end << 16), 0);
        if (first) first[d.rows[3][r]] = end > at && end - at < kRuns ? fresh((size_t)N * S + (size_t)at * kRuns + (size_t)(end - at)) : 1;
    }
    for (size_t r = 0; r < d.count[4]; ++r) {
        edit(d.rows[4][r], 4, (uint32_t)d.x[4][r], 0);
        if (first) first[d.rows[4][r]] = d.x[4][r] >= 0 && d.x[4][r] < N ? fresh((size_t)N * (S + kRuns) + (size_t)d.x[4][r]) : 1;
    }
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
    if (first) {
        // rows without an edit: the first of each template, and the first row that is the plan itself
        std::vector<uint8_t> seen((size_t)T);
        for (int k = 2; k <= 5; k += 3)
            for (size_t r = 0; r < d.count[k]; ++r) {
                uint8_t &was = seen[moves[4 * d.rows[k][r]]];
                first[d.rows[k][r]] = was ^ 1u;
                was = 1;
            }
        for (int k : {0, 1, 2, 5})
            for (size_t r = 0; r < d.count[k]; ++r) first[d.rows[k][r]] &= (uint8_t)(moves[4 * d.rows[k][r]] != 0u);
        for (size_t i = 0; i < d.n; ++i)
            if (!moves[4 * i]) {
                first[i] = 1;
                break;
            }
    }
    *n_templates = T;
    return ACE_OK;
}

// One move applied to its template (whose code bytes are `row`), in place.
inline void ace_apply_move(const uint32_t *mv, int N, int n_algo, uint8_t *row) {
    const int a_shift = n_algo == 2 ? 1 : 0, amask = n_algo - 1;
    const uint32_t op = mv[0] >> 16;
    const int p = (int)(mv[1] & 0xffffu), q = (int)(mv[1] >> 16);
    int lo = op == 1u ? std::min(p, q) : p, hi = op == 1u ? std::max(p, q) : op == 4u ? p + 1 : q;
    hi = std::min(hi, N);
    if (op == 1u && p < N) row[p] &= 0xEF;
    for (int i = lo; i < hi; ++i) {
        if (op == 1u) row[i] = (uint8_t)((row[i] & 0xF8) | ((mv[2] << a_shift) + (uint32_t)(row[i] & amask)));
        else if (op == 2u) {
            const int x = ((row[i] & 7) >> a_shift) + (mv[2] == 1u ? 1 : -1);
            row[i] = (uint8_t)((row[i] & 0xF8) | (((x < 0 ? 0 : x > 7 ? 7 : x) << a_shift) + (row[i] & amask)));
        } else if (op == 3u) row[i] ^= 8;
        else if (op == 4u) row[i] ^= 1;
    }
    if (op == 1u && q < N) row[q] |= 16;
}

// The 128-bit keys of moves' plans (what ace_apply_moves computes for the expanded plans) without expanding them: a key is the
// XOR of a value per 16-byte word, so a move's is its template's with the words it edits exchanged.
class AceMoveKeys {
  public:
    AceMoveKeys(const uint8_t *t_codes, const uint32_t *t_hdr, int T, int N, int n_algo)
        : G_((N + 15) / 16), T_(T), a_shift_(n_algo == 2 ? 1 : 0), rows_((size_t)T * G_ * 16), words_((size_t)T * G_), keys_(T) {
        for (int t = 0; t < T; ++t) {
            memcpy(&rows_[(size_t)t * G_ * 16], t_codes + (size_t)t * N, (size_t)N);
            const uint32_t *h = t_hdr + 4 * t;
            AceKey k{plan_key_word(h[0], h[1], h[2], 0u, 0u), plan_key_word2(h[0], h[1], h[2], 0u, 0u)};
            for (int g = 0; g < G_; ++g) {
                const AceKey w = word(&rows_[((size_t)t * G_ + g) * 16], g);
                words_[(size_t)t * G_ + g] = w;
                k.a ^= w.a;
                k.b ^= w.b;
            }
            keys_[t] = k;
        }
    }
    const std::vector<AceKey> &templates() const { return keys_; }
    AceKey key(const uint32_t *mv) const {
        switch (mv[0] >> 16) {
            case 0: return keys_[of_template(mv)];
            case 1: return edited<1>(mv);
            case 2: return edited<2>(mv);
            case 3: return edited<3>(mv);
            default: return edited<4>(mv);
        }
    }

  private:
    size_t of_template(const uint32_t *mv) const {
        const size_t t = mv[0] & 0xffffu;
        return t < (size_t)T_ ? t : 0;
    }
    // 0xff in the bytes [from, to) of eight
    static uint64_t bytes(int from, int to) {
        from = from < 0 ? 0 : from;
        to = to > 8 ? 8 : to;
        return from >= to ? 0 : (~0ull << (8 * from)) & (~0ull >> (8 * (8 - to)));
    }
    template <int OP> AceKey edited(const uint32_t *mv) const {
        constexpr uint64_t kEach = 0x0101010101010101ull;
        const size_t t = of_template(mv);
        const int p = (int)(mv[1] & 0xffffu), q = (int)(mv[1] >> 16);
        const int lo = OP == 1 ? std::min(p, q) : p, hi = OP == 1 ? std::max(p, q) : OP == 4 ? p + 1 : q;    // the bytes [lo, hi) change ...
        const int end = std::min(OP == 1 ? hi + 1 : hi, G_ * 16);                                            // ... (a migration also sets the bit at hi)
        const uint64_t amask = (1ull << a_shift_) - 1ull, keep = kEach * (0xF8u | amask), tp = kEach * (uint8_t)(mv[2] << a_shift_);
        AceKey k = keys_[t];
        for (int g = lo >> 4; g * 16 < end; ++g) {
            uint64_t w[2];
            memcpy(w, &rows_[(t * G_ + g) * 16], 16);
            for (int h = 0; h < 2; ++h) {
                const int base = g * 16 + 8 * h;
                const uint64_t in = bytes(lo - base, hi - base);
                if (OP == 1) {
                    w[h] &= ~(bytes(p - base, p + 1 - base) & (kEach * 0x10u));
                    w[h] = (w[h] & ~in) | (in & ((w[h] & keep) | tp));
                    w[h] |= bytes(q - base, q + 1 - base) & (kEach * 0x10u);
                } else if (OP == 2) {
                    for (int j = 0; j < 8; ++j) {
                        if (!((in >> (8 * j)) & 1u)) continue;
                        const int b = (int)(w[h] >> (8 * j)) & 0xff;
                        int x = ((b & 7) >> a_shift_) + (mv[2] == 1u ? 1 : -1);
                        x = x < 0 ? 0 : (x > 7 ? 7 : x);
                        w[h] = (w[h] & ~(0xffull << (8 * j))) | ((uint64_t)(uint8_t)((b & 0xF8) | ((x << a_shift_) + (b & (int)amask))) << (8 * j));
                    }
                } else
                    w[h] ^= in & (kEach * (OP == 3 ? 8u : 1u));
            }
            const AceKey was = words_[t * G_ + g], now = word(w, g);
            k.a ^= was.a ^ now.a;
            k.b ^= was.b ^ now.b;
        }
        return k;
    }
    static AceKey word(const void *bytes16, int g) {
        uint32_t w[4];
        memcpy(w, bytes16, 16);
        return AceKey{plan_key_word(w[0], w[1], w[2], w[3], (uint32_t)g + 1u), plan_key_word2(w[0], w[1], w[2], w[3], (uint32_t)g + 1u)};
    }
    int G_, T_, a_shift_;
    std::vector<uint8_t> rows_;
    std::vector<AceKey> words_, keys_;
};

// ace_build_moves, and of its moves (in order) those whose plan is in none of the sets and not an earlier move's; their keys
// go to sets[0].  Without sets: the first of each descriptor.  A few thousand of 16,384 moves on one plan are different ones,
// and most of those edit one or two words of it: 150 us, where expanding all of them on the device, fetching their keys and
// selecting among them took 400 us and two waits for the device.
inline int ace_new_moves_body(const uint8_t *codes, const uint32_t *hdr, int N, int A, int n_tp, int n_mbs, const uint32_t *stage_lut,
                              int gpus_per_node, const ace_move_draws_t &d, AceKeySet *const *sets, int n_sets, uint32_t *moves,
                              size_t *n_moves, uint8_t *t_codes, uint32_t *t_hdr, int max_templates, int *n_templates) {
    std::vector<uint8_t> first(d.n);
    const int rc = ace_build_moves_body(codes, hdr, N, A, n_tp, n_mbs, stage_lut, gpus_per_node, d, moves, t_codes, t_hdr, max_templates,
                                        n_templates, first.data());
    if (rc) return rc;
    // (nothing below branches on a row's kind or on whether it is kept: both are random)
    std::vector<uint32_t> at(n_sets ? d.n : 0);               // where a kept row goes
    size_t m = 0;
    if (n_sets)
        for (size_t i = 0; i < d.n; m += first[i++]) {
            at[i] = (uint32_t)m;
            memmove(moves + 4 * m, moves + 4 * i, 16);
        }
    else
        for (size_t i = 0; i < d.n; m += first[i++]) memmove(moves + 4 * m, moves + 4 * i, 16);
    std::vector<AceKey> keys(m);
    if (n_sets) {
        const AceMoveKeys of(t_codes, t_hdr, *n_templates, N, A);
        std::vector<uint32_t> kept(d.n);
        size_t listed = 0;
        for (int k = 0; k < 6; ++k) {
            size_t c = 0;
            for (size_t r = 0; r < d.count[k]; ++r) {
                kept[c] = at[d.rows[k][r]];
                c += first[d.rows[k][r]];
            }
            for (size_t r = 0; r < c; ++r) keys[kept[r]] = of.key(moves + 4 * kept[r]);
            listed += c;
        }
        // (a row of no kind is the plan itself: the one that is kept, if it is one of these, is the first plain move)
        if (listed < m)
            for (size_t i = 0; i < m; ++i)
                if (!moves[4 * i]) {
                    keys[i] = of.key(moves + 4 * i);
                    break;
                }
    } else if (m)
        memcpy(keys.data(), moves, m * 16);
    AceKeySet here;
    if (!n_sets) here.reserve(m);
    AceKeySet *own = &here;
    AceKeySet *const *in = n_sets ? sets : &own;
    const int n_in = n_sets ? n_sets : 1;
    size_t kept = 0;
    ace_each_key(reinterpret_cast<const uint64_t *>(keys.data()), m, in, n_in, [&](size_t i, const AceKey &k) {
        bool fresh = true;
        for (int j = 1; j < n_in && fresh; ++j) fresh = !in[j]->has(k);
        if (fresh && in[0]->add(k)) {
            memmove(moves + 4 * kept, moves + 4 * i, 16);
            ++kept;
        }
    });
    *n_moves = kept;
    return ACE_OK;
}
