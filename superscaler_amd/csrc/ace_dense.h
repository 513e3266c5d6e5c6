// Scoring of LARGE batches over dense tables: a plan per lane, like ace_many.h, but what an op costs a lane beside the
// reference's own additions is as little as could be found: two v_dot4_u32_u8 for all addresses, one 8-byte LDS read per value,
// one 16-byte read for both collectives' costs, and records that are stored in whole cache lines (gen_dense_loop_asm.py).  Where the
// tables take less than half of a CU's LDS in the form below, two workgroups of eight wavefronts share a CU, and one evaluates
// its stage tails or stages its tables while the other walks; else one of sixteen has it to itself.
// Rows resident: from 65,537 plans on.  Rows in windows: from what the kernel of small batches leaves.
// Measured, us per launch, ace_many.h -> here:
//   plans      315 ops           523 ops           821 ops, no resharding   1,251 ops, 16 stages
//   65,537     64.2 ->  58.9     130.1 -> 117.5    134.7 -> 113.9           285.1 -> 235.2
//   100,000    65.5 ->  60.1     131.4 -> 120.9    135.8 -> 116.2           287.8 -> 238.8
//   262,144   102.4 ->  88.6     176.9 -> 149.5    167.0 -> 148.7           461.0 -> 398.3
//   1,048,576                    694.0 -> 555.9
//   (523 ops, 1,048,576 plans, all of one stage: 447 -> 357, all of sixteen: 1,456 -> 981)
//   windowed rows: 134 ops, 7,681 plans 45.7 -> 32.6, 65,536 55.4 -> 41.1, 131,072 63.7 -> 48.0, 262,144 92.6 -> 72.9, 300,000 132.7 -> 99.9;
//   230 ops, 262,144 plans 121.7 -> 88.0; 270 ops in 270 types (the C++ loop before), 100,000 plans 455.8 -> 66.0, 500,000 475.8 -> 196.6
//   tables of more than 80 KB (all of a CU for one workgroup), in windows or as the table compiler's rows before: 523 ops with 80 entries per
//   row 100,000 plans 123.1 -> 106.8, 262,144 195.2 -> 164.4; 1,251 ops, all sizes of the database different, 262,144 461.8 -> 388.7; 821 ops with
//   44 entries 181.6 -> 163.3 (ace_duo.h: 8,192 plans 89.5 -> 52.6, 235.7 -> 87.8, 85.0 -> 68.5; 65,536 115.8 -> 84.1, 255.4 -> 172.3, 111.0 -> 93.6)
// What bounds it is the issue of vector instructions: about 30 per op and wavefront of the mix of depths (35 before), and the issue
// of everything else beside them; with fewer than four wavefronts per SIMD the latency of a step.  One workgroup of 1,024 lanes per
// CU instead: 594 us where two of 512 took 567.
//
// The dense tables, one block that is copied to LDS address 0 on:
//   pairs   16 bytes {forward, backward} ms of resharding, every distinct pair once, {0, 0} first
//   rows    per op type used, 40 bytes per entry: forward, backward, weights, activations, and the ranks of the two reserved sizes
//           (16 bits each) among all that occur; entry diag * C + code as in the table compiler's rows, as many as there are
//   slabs   per distinct (pair kind, next op's type): blocks of [code][next code] 16-bit addresses into `pairs`, one block per
//           distinct (diag, stage size)
//   lut     per (micro-batch size, stage size): LDS address of the diag's entries in the first row, of its block in the first slab
//   stages  the stage LUT as it is
// and what the evaluation of the stage tails looks up (from global memory those were six gathers per stage, 1 ns per lane and CU
// each: 115 of 760 us per 1,048,576 plans of 523 ops):
//   reserved sizes by rank; per (op type, diag * C + code) and per (op type, output entry) a 16-bit LDS address of the distinct
//   {input MB, intra-node ms, inter-node ms} and {output intra, inter}; types that agree in all of them share one list
// An entry's stride of 40 bytes is ten banks of 64: like at a stride of eight bytes, the 8-byte reads of any 32 entries in a row meet no
// bank twice.  The values' offsets within an entry are constants of the loops, whatever the tables.  (An array per value instead, of 40, 64,
// 72 or 120 entries as a template's parameter: the same times within 1 % where a row filled its array -- 1,048,576 plans of 523 ops 547.4 and
// 547.4 us, 65,536 of 821 93.5 and 93.1 --, and rows of 41 entries took the room of 64.)
// With two algorithms and four tp sizes most codes in use are even, and diags four apart lie 32 entries apart: from the fourth on
// they lie one entry further, so that their even codes read different banks.  Blocks of a slab are 132 bytes apart for the same reason.
// Rows that do not all fit go through windows (as many ops as the rows of half the space behind the rest serve, a multiple of four),
// consecutive windows in alternate halves, fetched by the loop itself; everything else stays resident.
// What a code byte reads that names no profiled entry (codes past the last tp size) is what it reads in the table compiler's
// rows: the tables are filled by those addresses.
#pragma once
#include <algorithm>
#include <cstring>
#include <map>
#include <utility>
#include <vector>

#include "ace_score_loop.h"

constexpr uint32_t kDenseLds = 80u * 1024u;    // LDS of a workgroup: two per CU
constexpr int kDenseLanes = 512;
// ... one per CU: tables of more than that, up to all of a CU's LDS, and windowed rows, so that a window holds more ops (134 ops, two
// workgroups of 512 lanes per CU with windows of 8 ops against one of 1,024 with 20: 65,536 plans 44.9 / 41.1 us, 262,144 69.4 / 72.9,
// 300,000 104.6 / 99.9)
constexpr uint32_t kDenseWinLds = 160u * 1024u;
constexpr int kDenseWinLanes = 1024;
constexpr uint32_t kDenseEntry = 40u, kDenseValue = 8u;          // bytes of an entry; from one of its values to the next

struct AceDenseArgs {
    const ace_u4 *image;        // the tables
    const ace_u4 *pos;          // [16 * G + 16] per position: dot4 scalars of the row and of the slab, record word, flags (as pos4)
    const ace_u2 *pos_duo;      // ... as the roles of ace_duo.h have it: the two scalars; then the row's and the record word with the flags at bit 12
    const unsigned char *events;        // windowed rows: fetch records, 48 bytes per event and wavefront (see dense_events)
    uint32_t n_events;
    uint32_t image16;           // size of the image in 16-byte pieces
    uint32_t lut_off, stg_off, rf_off, rb_off, in_off, out_off;   // LDS offsets
    uint32_t in_entries, out_entries;   // 16-bit addresses per list
    uint32_t half, lut_half;    // windowed rows: from the first half of the rows, of the offsets' table, to the second
    uint32_t kv;                // constant byte(s) of the code words
    uint32_t first_in;          // list of the first op
};

// What the library keeps of it (built on the host).
struct AceDenseTables {
    std::vector<unsigned char> image;
    std::vector<ace_u4> pos;
    std::vector<ace_u2> pos_duo;
    std::vector<unsigned char> rows;            // windowed: every row, `row_pitch` bytes each ...
    std::vector<std::vector<uint32_t>> windows; // ... the rows of each window in the order of their slots
    std::vector<int> window_start;
    uint32_t row_pitch = 0, rows_off = 0;
    AceDenseArgs args{};        // (offsets)
    uint32_t array = kDenseValue, lds = 0;
    int lanes = 0;              // of a workgroup of large batches
    bool ok = false;
};

// LDS behind the image: the deal's bins and permutation, and the arrival counters; windowed, the rows lie there afterwards.
inline uint32_t ace_dense_scratch(int lanes) { return 128u + 2u * (uint32_t)lanes + 128u; }
// ... that of the kernel of mid-sized batches (ace_duo.h), whose workgroup of L plans has a CU to itself: bins, permutation, the parts'
// stage counts.
constexpr int kDuoBlock = 1024;     // its lanes: eight wavefronts per role
inline uint32_t ace_duo_scratch(int L) { return 128u + 2u * (uint32_t)L + 2u * (uint32_t)kDuoBlock; }

// Fills `d` (d.ok false: the tables do not fit this form).  `lds`: how much of it a workgroup may take, `scratch`: what of that is for
// the kernel's own use (windowed: before the first rows arrive); `lanes`: of a workgroup that fetches windows.
inline void dense_build(const ace_tables_t *t, size_t pos_entries, bool windowed, uint32_t lds, uint32_t scratch, int lanes, AceDenseTables &d) {
    d = AceDenseTables();
    const int N = t->num_ops, C = t->n_tp * t->n_algo, ND = t->n_diag;
    if ((t->flags & ACE_F_COLLECTIVE_MEM) || N >= 32768) return;
    const bool rsh = (t->flags & ACE_F_RESHARDING) != 0;
    const uint32_t entries = (uint32_t)(ND * C + 8), further = C == 8 && t->n_algo == 2 && ND > 4 ? 1u : 0u, row_bytes = (entries + further) * kDenseEntry;
    auto diag_entry = [&](uint32_t dg) { return dg * (uint32_t)C + (dg >= 4u ? further : 0u); };
    const size_t n_rows_all = (size_t)t->num_types * (size_t)t->row_doubles;
    auto at = [&](size_t type, size_t off) {                       // a double of a row, or of what follows it in memory
        const size_t i = type * (size_t)t->row_doubles + off;
        return i < n_rows_all ? t->rows[i] : 0.0;
    };
    // the op type of each position; those in use, in the order of their numbers
    std::vector<uint32_t> types(N), used;
    for (int i = 0, w = 0; i < N; ++i) {
        while (w + 1 < t->n_windows && t->win_pos[w + 1] <= i) ++w;
        const uint32_t slot_off = (t->pos_info[i] & 0xffu) * (uint32_t)t->row_doubles * 8u;
        for (int r = t->win_row_begin[w]; r < t->win_row_begin[w + 1]; ++r)
            if (t->win_rows[2 * r + 1] == slot_off) types[i] = t->win_rows[2 * r];
    }
    std::vector<int> row_of(t->num_types, -1);
    for (int i = 0; i < N; ++i) row_of[types[i]] = 0;
    for (int ty = 0; ty < t->num_types; ++ty)
        if (row_of[ty] == 0) { row_of[ty] = (int)used.size(); used.push_back((uint32_t)ty); }
    if (!windowed && used.size() * row_bytes > lds) return;         // (before anything that takes time: 134 rows of 72 entries 5 ms)
    // ranks of the reserved sizes: what a running maximum from 0.0 can become (0.0: rank 0)
    std::vector<double> reserved_fwd, reserved_bwd, *const values[2] = {&reserved_fwd, &reserved_bwd};
    for (int w = 0; w < 2; ++w) {
        std::vector<double> &v = *values[w];
        for (uint32_t ty : used)
            for (uint32_t e = 0; e < entries; ++e) {
                const double x = at(ty, (size_t)t->hot_off + e * 6u + 4u + (size_t)w);
                if (x > 0.0) v.push_back(x);
            }
        v.push_back(0.0);
        std::sort(v.begin(), v.end());
        v.erase(std::unique(v.begin(), v.end()), v.end());
        if (v.size() > 65536u) return;
    }
    auto rank = [&](int w, double x) {
        return x > 0.0 ? (uint32_t)(std::lower_bound(values[w]->begin(), values[w]->end(), x) - values[w]->begin()) : 0u;
    };
    // pairs, slabs, blocks
    std::vector<std::pair<uint64_t, uint64_t>> pairs{{0u, 0u}};
    std::map<std::pair<uint64_t, uint64_t>, uint32_t> pair_at{{{0u, 0u}, 0u}};
    std::vector<uint32_t> slab_of(pos_entries, 0u);                // per position, of the (this op, next op) pair
    std::vector<uint32_t> block_of((size_t)t->n_mbs * 16u, 0u);
    std::vector<std::vector<uint16_t>> slabs;                      // [slab][block * 64 + code * 8 + next code]
    size_t n_blocks = 1;
    constexpr uint32_t kBlock = 132u;
    if (rsh) {
        std::vector<std::pair<uint32_t, uint32_t>> kinds, stages;   // (pair kind, next type); (diag, stage size as the pair kinds index it)
        std::vector<uint32_t> kind_of(N, 0u), stage_of((size_t)t->n_mbs * 16u);
        auto index = [](std::vector<std::pair<uint32_t, uint32_t>> &v, std::pair<uint32_t, uint32_t> x) {
            const auto it = std::find(v.begin(), v.end(), x);
            if (it != v.end()) return (uint32_t)(it - v.begin());
            v.push_back(x);
            return (uint32_t)v.size() - 1u;
        };
        for (int i = 0; i + 1 < N; ++i) kind_of[i] = index(kinds, {(t->pos_info[i] >> 16) & 0xffu, types[i + 1]});
        if (kinds.empty()) kinds.push_back({0u, types[0]});
        for (uint32_t j = 0; j < (uint32_t)t->n_mbs * 16u; ++j)
            stage_of[j] = index(stages, {t->stage_lut[j] & 15u, (j & 15u) < (uint32_t)t->n_glog ? j & 15u : 0u});
        // a stage's block over all kinds at once: equal ones are kept once
        std::vector<std::vector<uint16_t>> columns;
        std::vector<uint32_t> column_of;
        for (const auto &st : stages) {
            std::vector<uint16_t> col;
            for (const auto &k : kinds)
                for (uint32_t cc = 0; cc < 64u; ++cc) {
                    const uint32_t id = t->pair_kinds[((size_t)k.first * t->n_glog + st.second) * 64u + cc];
                    const size_t e = (size_t)t->z_off + st.first * (uint32_t)C + (cc & 7u);
                    std::pair<uint64_t, uint64_t> p;
                    const double f = at(k.second, e + (size_t)(id & 15u) * t->z_table_doubles), b = at(k.second, e + (size_t)(id >> 4) * t->z_table_doubles);
                    memcpy(&p.first, &f, 8);
                    memcpy(&p.second, &b, 8);
                    const auto ins = pair_at.insert({p, (uint32_t)pairs.size()});
                    if (ins.second) pairs.push_back(p);
                    if (pairs.size() > 4096u) return;               // (16-bit LDS addresses)
                    col.push_back((uint16_t)(ins.first->second * 16u));
                }
            uint32_t c = (uint32_t)(std::find(columns.begin(), columns.end(), col) - columns.begin());
            if (c == columns.size()) columns.push_back(col);
            column_of.push_back(c);
        }
        n_blocks = columns.size();
        for (size_t j = 0; j < block_of.size(); ++j) block_of[j] = column_of[stage_of[j]];
        // ... and equal slabs
        std::vector<uint32_t> slab_of_kind;
        for (size_t k = 0; k < kinds.size(); ++k) {
            std::vector<uint16_t> s;
            for (const auto &col : columns) s.insert(s.end(), col.begin() + k * 64u, col.begin() + (k + 1u) * 64u);
            uint32_t at_slab = (uint32_t)(std::find(slabs.begin(), slabs.end(), s) - slabs.begin());
            if (at_slab == slabs.size()) slabs.push_back(s);
            slab_of_kind.push_back(at_slab);
        }
        for (int i = 0; i + 1 < N; ++i) slab_of[i] = slab_of_kind[kind_of[i]];
    }
    // what the evaluation looks up comes first (it decides how much room the rows have)
    AceDenseArgs &g = d.args;
    // what the evaluation looks up: distinct {input MB, intra, inter} and {output intra, inter}, their place per row and entry
    // (numbered as they come.  Tables that turn out not to fit are left as soon as that is known: with every size of a database of its
    // own, 566 types of 72 entries, a search from the front each time and a look at the end took 530 ms, this 24)
    typedef std::vector<uint64_t> Bits;
    std::vector<Bits> values_in, values_out;
    std::map<Bits, uint32_t> in_at, out_at;
    auto place_of = [&](std::vector<Bits> &v, std::map<Bits, uint32_t> &known, uint32_t ty, size_t off, size_t n) {
        Bits b(n);
        for (size_t k = 0; k < n; ++k) {
            const double x = at(ty, off + k);
            memcpy(&b[k], &x, 8);
        }
        const auto ins = known.insert({b, (uint32_t)v.size()});
        if (ins.second) v.push_back(b);
        return ins.first->second;
    };
    g.in_entries = entries;
    g.out_entries = (uint32_t)(t->n_mbs * t->n_tp + 8) * (uint32_t)t->n_algo;    // (a code past the last tp size: up to index 7)
    std::vector<std::vector<uint32_t>> in_lists, out_lists;
    std::vector<uint32_t> in_of, out_of;                            // per row: its list
    auto list_of = [](std::vector<std::vector<uint32_t>> &v, const std::vector<uint32_t> &x) {
        const size_t i = (size_t)(std::find(v.begin(), v.end(), x) - v.begin());
        if (i == v.size()) v.push_back(x);
        return (uint32_t)i;
    };
    for (uint32_t ty : used) {
        std::vector<uint32_t> in, out;
        for (uint32_t e = 0; e < g.in_entries; ++e) in.push_back(place_of(values_in, in_at, ty, (size_t)t->start_off + e * 3u, 3));
        for (uint32_t e = 0; e < g.out_entries; ++e) out.push_back(place_of(values_out, out_at, ty, (size_t)t->out_off + e * 2u, 2));
        in_of.push_back(list_of(in_lists, in));
        out_of.push_back(list_of(out_lists, out));
        if (in_lists.size() > 256u || out_lists.size() > 256u) return;   // (eight bits each in a record word)
        if (pairs.size() * 16u + values_out.size() * 16u + values_in.size() * 24u > 65536u) return;   // (16-bit LDS addresses)
    }
    // How far apart rows and slabs lie, and the constant bytes whose multiples (at most 255 of each) name their places; rows: as many as
    // `slots` (windowed: in each half, and fetched in pieces of 16 bytes, 1 KB at a time).  With resharding one constant K for both;
    // else two of the rows alone: 248 and 8, which name any place below 63 KB, or for more rows than those reach K twice.
    const uint32_t n_slabs = (uint32_t)slabs.size(), slab_bytes = (uint32_t)n_blocks * kBlock, row_least = windowed ? std::max(row_bytes, 1024u) : row_bytes;
    const size_t lists = (in_lists.size() * g.in_entries + out_lists.size() * g.out_entries) * 2u;
    uint32_t K = 0, K2 = 0, row_pitch = 0, slab_pitch = 0, slots = windowed ? 31u : (uint32_t)used.size();
    auto fits = [&](uint32_t n) {                                   // n rows: K and the pitches, the smallest in all
        K = 0;
        uint64_t best = ~0ull;
        const uint32_t whole = (row_least + 15u) & ~15u;
        if (!rsh && (n - 1u) * whole <= 248u * 255u + 247u) {
            row_pitch = whole;
            K = 248u;
            K2 = 8u;
            best = (uint64_t)n * row_pitch * (windowed ? 2u : 1u);
        } else
            for (uint32_t k = 8; k <= 248u; k += 8u) {
                uint32_t u = (row_least + k - 1u) / k;
                const uint32_t v = (slab_bytes + k - 1u) / k;
                u += windowed && ((u * k) & 15u) ? 1u : 0u;
                if ((n - 1u) * u > (rsh ? 255u : 510u) || (rsh && (n_slabs - 1u) * v > 255u)) continue;
                const uint64_t size = (uint64_t)n * u * k * (windowed ? 2u : 1u) + (uint64_t)n_slabs * v * k;
                if (size < best) { best = size; K = K2 = k; row_pitch = u * k; slab_pitch = v * k; }
            }
        const uint64_t rest = pairs.size() * 16u + values_out.size() * 16u + values_in.size() * 24u + (size_t)t->n_mbs * (windowed ? 320u : 192u) +
                              (reserved_fwd.size() + reserved_bwd.size()) * 8u + lists + 256u;
        return K != 0u && best + rest + (windowed ? 0u : scratch) <= lds;
    };
    if (windowed)
        while (slots >= 4u && (!fits(slots) || slots * ((row_pitch + 1023u) / 1024u) > 4u * (uint32_t)lanes / 64u)) --slots;   // (four loads per event and wavefront)
    if (slots < 4u && windowed) return;
    if (!fits(slots)) return;
    g.kv = (K << 24) | (rsh ? 0u : K2 << 16);
    // the image (what 16-bit addresses name lies in front)
    uint32_t end = 0;
    auto take = [&](size_t bytes, uint32_t align) {
        const uint32_t off = (end + align - 1u) / align * align;
        end = off + (uint32_t)bytes;
        return off;
    };
    take(pairs.size() * 16u, 16u);
    const uint32_t vout_off = take(values_out.size() * 16u, 16u), vin_off = take(values_in.size() * 24u, 8u);
    if (end > 65536u) return;
    const uint32_t slabs_off = take((size_t)n_slabs * slab_pitch, 16u);
    g.lut_half = (uint32_t)t->n_mbs * 128u;
    g.lut_off = take((size_t)g.lut_half * (windowed ? 2u : 1u), 128u);
    g.stg_off = take((size_t)t->n_mbs * 64u, 4u);
    g.rf_off = take(reserved_fwd.size() * 8u, 8u);
    g.rb_off = take(reserved_bwd.size() * 8u, 8u);
    g.in_off = take(in_lists.size() * g.in_entries * 2u, 2u);
    g.out_off = take(out_lists.size() * g.out_entries * 2u, 2u);
    const uint32_t n_rows = (uint32_t)used.size(), rows_off = take(windowed ? 0u : (size_t)n_rows * row_pitch, 16u), bytes = take(0, 16u);
    g.half = slots * row_pitch;
    d.lds = bytes + (windowed ? std::max(2u * g.half, scratch) : scratch);
    if (d.lds > lds) return;
    d.row_pitch = row_pitch;
    d.lanes = lanes;
    d.rows_off = rows_off;
    g.image16 = bytes / 16u;
    // windows: a multiple of four ops each (or up to the last op), of at most `slots` different rows
    std::vector<uint32_t> place(N, 0u);                             // of each position's row, from the first one (of its half) on
    if (windowed) {
        for (int i = 0; i < N;) {
            std::vector<uint32_t> seen;
            size_t good_n = 0;
            int good = -1;
            for (int j = i; j < N;) {
                const uint32_t r = (uint32_t)row_of[types[j]];
                if (std::find(seen.begin(), seen.end(), r) == seen.end()) {
                    if (seen.size() >= slots) break;
                    seen.push_back(r);
                }
                ++j;
                if (j == N || (j & 3) == 0) { good = j; good_n = seen.size(); }
            }
            if (good < 0) return;
            seen.resize(good_n);
            for (int j = i; j < good; ++j) place[j] = (uint32_t)(std::find(seen.begin(), seen.end(), (uint32_t)row_of[types[j]]) - seen.begin()) * row_pitch;
            d.window_start.push_back(i);
            d.windows.push_back(seen);
            i = good;
        }
        if (d.windows.size() < 2u) return;
    } else
        for (int i = 0; i < N; ++i) place[i] = (uint32_t)row_of[types[i]] * row_pitch;
    d.image.assign(bytes, 0);
    auto put = [&](uint32_t off, const void *p, size_t n) { if (n) memcpy(d.image.data() + off, p, n); };
    for (size_t i = 0; i < pairs.size(); ++i) {
        put((uint32_t)i * 16u, &pairs[i].first, 8);
        put((uint32_t)i * 16u + 8u, &pairs[i].second, 8);
    }
    for (size_t i = 0; i < values_out.size(); ++i) put(vout_off + (uint32_t)i * 16u, values_out[i].data(), 16);
    for (size_t i = 0; i < values_in.size(); ++i) put(vin_off + (uint32_t)i * 24u, values_in[i].data(), 24);
    auto put_lists = [&](uint32_t off, const std::vector<std::vector<uint32_t>> &v, uint32_t base, uint32_t size) {
        for (const auto &list : v)
            for (uint32_t x : list) {
                const uint16_t a16 = (uint16_t)(base + x * size);
                put(off, &a16, 2);
                off += 2u;
            }
    };
    put_lists(g.in_off, in_lists, vin_off, 24u);
    put_lists(g.out_off, out_lists, vout_off, 16u);
    put(g.rf_off, reserved_fwd.data(), reserved_fwd.size() * 8u);
    put(g.rb_off, reserved_bwd.data(), reserved_bwd.size() * 8u);
    if (windowed) d.rows.assign((size_t)n_rows * row_pitch, 0);
    unsigned char *rows = windowed ? d.rows.data() : d.image.data() + rows_off;
    for (size_t r = 0; r < n_rows; ++r)
        for (uint32_t dg = 0; dg <= (uint32_t)ND; ++dg)
            for (uint32_t c = 0; c < 8u; ++c) {
                // (a code past the last one reads what follows its diag's entries)
                const uint32_t e = dg * (uint32_t)C + c;
                unsigned char *to = rows + r * row_pitch + (diag_entry(dg) + c) * kDenseEntry;
                if (c >= (uint32_t)C && dg < (uint32_t)ND) continue;
                double v[6];
                for (uint32_t k = 0; k < 6u; ++k) v[k] = at(used[r], (size_t)t->hot_off + e * 6u + k);
                for (uint32_t k = 0; k < 4u; ++k) memcpy(to + k * kDenseValue, &v[k], 8);
                const uint32_t both = rank(0, v[4]) | (rank(1, v[5]) << 16);
                memcpy(to + 4u * kDenseValue, &both, 4);
            }
    for (uint32_t s = 0; s < n_slabs; ++s)
        for (uint32_t b = 0; b < (uint32_t)n_blocks; ++b) put(slabs_off + s * slab_pitch + b * kBlock, slabs[s].data() + b * 64u, 128);
    for (uint32_t j = 0; j < (uint32_t)t->n_mbs * 16u; ++j) {
        const ace_u2 z{rows_off + diag_entry(t->stage_lut[j] & 15u) * kDenseEntry, slabs_off + block_of[j] * kBlock};
        put(g.lut_off + j * 8u, &z, 8);
        const ace_u2 other{z.x + g.half, z.y};
        if (windowed) put(g.lut_off + g.lut_half + j * 8u, &other, 8);
        put(g.stg_off + j * 4u, &t->stage_lut[j], 4);
    }
    // positions
    d.pos.assign(pos_entries, ace_u4{0u, 0u, 0u, 0u});
    d.pos_duo.assign(2u * pos_entries, ace_u2{0u, 0u});
    for (size_t i = 0; i < pos_entries; ++i) {
        const bool odd = (i & 1u) != 0u, in = i < (size_t)N;
        const uint32_t info = in ? t->pos_info[i] : 0u, at_row = in ? place[i] : 0u, slab = in ? slab_of[i] : 0u;
        const uint32_t last = in ? out_of[row_of[types[i]]] : 0u, next = in && i + 1 < (size_t)N ? in_of[row_of[types[i + 1]]] : 0u;
        ace_u4 &p = d.pos[i];
        const uint32_t units = std::min(at_row / K, 255u);
        p.x = (odd ? kDenseEntry << 8 : kDenseEntry) | (units << 24) | (rsh ? 0u : ((at_row - units * K) / K2) << 16);
        p.y = rsh ? (odd ? (16u << 8) | (2u << 16) : 16u | (2u << 8)) | ((slab * (slab_pitch / K)) << 24) : 0u;
        // record word: codes of the stage's last op and of the next one in bytes 0 and 1 (odd positions with resharding: 1
        // and 2, bit 11 set), the last op's list of outputs and the next one's of inputs in the other two
        p.z = rsh && odd ? last | (next << 24) | (1u << 11) : (last << 16) | (next << 24);
        p.w = (((info >> 24) & 1u) ^ 1u) | (((info >> 25) & 1u) << 1);
        d.pos_duo[i] = ace_u2{p.x, p.y};
        d.pos_duo[pos_entries + i] = ace_u2{p.x, p.z | (p.w << 12)};
    }
    g.first_in = in_of[row_of[types[0]]];
    d.ok = true;
}

// Every row resident where they fit: beside a second workgroup on the CU, else in all of its LDS; windows for more than that.
inline void ace_dense_build(const ace_tables_t *t, size_t pos_entries, AceDenseTables &d) {
    dense_build(t, pos_entries, false, kDenseLds, ace_dense_scratch(kDenseLanes), kDenseLanes, d);
    if (!d.ok) dense_build(t, pos_entries, false, kDenseWinLds, std::max(ace_dense_scratch(kDenseWinLanes), ace_duo_scratch(256)), kDenseWinLanes, d);
    if (!d.ok) dense_build(t, pos_entries, true, kDenseWinLds, ace_dense_scratch(kDenseWinLanes), kDenseWinLanes, d);
}

// Windowed rows: the fetch records, per event and wavefront 48 bytes = {first position of the window after the one being entered,
// bit 0: wait for the fetch (else it completes before the next event) | number of loads << 8, address of the rows} and four
// LDS-direct loads {byte offset in the rows, LDS address} of 1 KB each.  Events: 0 fetches window 0 and waits, 1 fetches window 1,
// and entering window w >= 1 fetches window w + 1 (the last one fetches window w - 1 again, into the half nobody reads).
inline std::vector<uint32_t> dense_events(const AceDenseTables &d, uint64_t rows_at) {
    const int n_w = (int)d.windows.size();
    const uint32_t waves = (uint32_t)kDenseWinLanes / 64u;
    std::vector<uint32_t> out((size_t)(n_w + 1) * waves * 12u, 0u);
    for (int e = 0; e <= n_w; ++e) {
        const int entering = e < 2 ? 0 : e - 1;                        // the window walked after this event
        int fetch = e == 0 ? 0 : entering + 1;
        if (fetch >= n_w) fetch = entering - 1;
        std::vector<ace_u2> loads;
        for (size_t s = 0; s < d.windows[fetch].size(); ++s)
            for (uint32_t off = 0; off < d.row_pitch; off += 1024u) {
                // (the last load of a row ends with it: it may overlap the one before it)
                const uint32_t o = off + 1024u <= d.row_pitch ? off : d.row_pitch - 1024u;
                loads.push_back(ace_u2{d.windows[fetch][s] * d.row_pitch + o, d.rows_off + (fetch & 1 ? d.args.half : 0u) + (uint32_t)s * d.row_pitch + o});
            }
        for (uint32_t v = 0; v < waves; ++v) {
            uint32_t *rec = &out[((size_t)e * waves + v) * 12u], n = 0;
            for (size_t c = v; c < loads.size(); c += waves, ++n) { rec[4 + 2 * n] = loads[c].x; rec[5 + 2 * n] = loads[c].y; }
            rec[0] = entering + 1 < n_w ? (uint32_t)d.window_start[entering + 1] : 0x7fffffffu;
            rec[1] = (e == 0 ? 1u : 0u) | (n << 8);
            rec[2] = (uint32_t)rows_at;
            rec[3] = (uint32_t)(rows_at >> 32);
        }
    }
    return out;
}

// What a record word says.
struct DenseMeta { uint32_t c_last, c_next, out_list, in_list; };
ACE_HD DenseMeta dense_meta(uint32_t m) {
    const bool odd = (m >> 11) & 1u;
    const uint32_t w = odd ? m >> 8 : m;
    return DenseMeta{w & 7u, (w >> 8) & 7u, (odd ? m : m >> 16) & 0xffu, m >> 24};
}

// Slices of 64 plans per workgroup (`most`: as many as it has wavefronts), so that the rounds of `places` workgroups that the batch
// needs are all full.
inline uint32_t ace_dense_slices(long long plans, long long most, long long places) {
    const long long fullest = ((plans + 63) / 64 + places - 1) / places;
    const long long rounds = (fullest + most - 1) / most;
    return (uint32_t)((fullest + rounds - 1) / rounds);
}

// A wavefront's part of the workspace: the records of its plans' stages in the order in which they were stored, as five pieces of up
// to 1,024 times 16 bytes -- {fwd + bwd, recompute}, {resharding forward, backward}, {weights, activations}, {saved, peak},
// {ranks, record word, record word of the stage before, place} --, and behind them what each came to: {ms, MB} at [stage][lane].
// A place is stage * 128 + lane * 2.
constexpr uint32_t kDensePiece = 64u * ACE_MAX_STAGES * 16u, kDenseResults = 5u * kDensePiece, kDenseWave = 6u * kDensePiece;
static_assert(kDensePiece == 16384u, "as the loop has it");
constexpr uint32_t kDensePlan = kDenseWave / 64u;                // workspace bytes per plan

typedef PlanState<false, false, true> DenseState;
struct DenseRecord { ace_d2 r[4]; ace_u4 tail; };
ACE_HD void dense_load(const unsigned char *ws, uint32_t i, DenseRecord &rec) {
#pragma unroll
    for (uint32_t j = 0; j < 4u; ++j) rec.r[j] = *reinterpret_cast<const ace_d2 *>(ws + j * kDensePiece + i * 16u);
    rec.tail = *reinterpret_cast<const ace_u4 *>(ws + 4u * kDensePiece + i * 16u);
}

#ifdef ACE_HOST_EMU
ACE_HD uint32_t dense_shfl(uint32_t x, uint32_t) { return x; }   // (wavefronts of one lane)
constexpr uint32_t kDenseWidth = 1;
#else
ACE_HD uint32_t dense_shfl(uint32_t x, uint32_t lane) { return (uint32_t)__shfl((int)x, (int)lane, 64); }
constexpr uint32_t kDenseWidth = 64;
#endif

// One record: time and memory of its stage (number `s`, 2^glog GPUs), in st.sum_t and st.max_mem.
ACE_HD void dense_tail(const AceDenseArgs &d, const AceGeom &g, const AceLds &lds, uint32_t bidx, uint32_t glog, uint32_t s, const DenseRecord &rec, DenseState &st) {
    st.s = (int)s;
    const DenseMeta m = dense_meta(rec.tail.y), before = dense_meta(rec.tail.z);
    const uint32_t lut = lds.ld<uint32_t>(d.stg_off + (bidx * 16u + glog) * 4u);
    st.mrow = lut >> 16;
    st.t_first = before.c_next >> g.A_shift;
    const uint32_t e = ace_mul24(lut & 15u, (uint32_t)g.C) + before.c_next, o = DenseState::out_entry_addr(g, 0u, m.c_last, st.t_first, st.mrow) >> 4;
    const uint32_t in = lds.ld<uint16_t>(d.in_off + (ace_mul24(before.in_list, d.in_entries) + e) * 2u);
    const uint32_t out = lds.ld<uint16_t>(d.out_off + (ace_mul24(m.out_list, d.out_entries) + o) * 2u);
    st.rfm = lds.ld<double>(d.rf_off + (rec.tail.x & 0xffffu) * 8u);
    st.rbm = lds.ld<double>(d.rb_off + (rec.tail.x >> 16) * 8u);
    st.inputs = lds.ld<double>(in);
    st.in_comm = lds.ld<double>(in + (((st.cross >> s) & 1u) ? 16u : 8u));
    const ace_d2 oe = lds.ld<ace_d2>(out);
    st.out_cross = (st.cross >> (16u + s)) & 1u;
    // (fwd + bwd is added up already, and the peak closed)
    st.fwd = rec.r[0].x; st.bwd = 0.0; st.rcs = rec.r[0].y; st.rs_f = rec.r[1].x; st.rs_b = rec.r[1].y; st.W = rec.r[2].x; st.A = rec.r[2].y;
    st.saved = rec.r[3].x; st.peak = rec.r[3].y; st.run = 0.0; st.lastclose = false;
    st.sum_t = 0.0; st.max_t = 0.0; st.max_mem = 0.0;
    st.finish_tail(g, lds, 0u, m.c_last, oe, nullptr);
}

// ... of the loop here.  `own`: the lane's own plan (its header's words reach the lanes that evaluate its stages through dense_shfl).
ACE_HD void dense_stage(const AceDenseArgs &d, const AceGeom &g, const AceLds &lds, const DenseState &own, const DenseRecord &rec, DenseState &st) {
    const uint32_t lane = (rec.tail.w >> 1) & 63u, s = rec.tail.w >> 7;
    const uint32_t sb = dense_shfl((uint32_t)own.S | (own.bidx << 8), lane);
    const uint32_t glogs = dense_shfl((uint32_t)own.glogs, lane), glogs_hi = dense_shfl((uint32_t)(own.glogs >> 32), lane);
    st.cross = dense_shfl(own.cross, lane);
    st.S = (int)(sb & 0xffu);
    dense_tail(d, g, lds, sb >> 8, ((s & 8u ? glogs_hi : glogs) >> (4u * (s & 7u))) & 15u, s, rec, st);
}

// The tails of all stages of a wavefront's plans, a record per lane whoever's it is (all lanes are busy whatever the depths of the
// plans), the next two rounds' records on their way; then each lane puts its own plan together, stage times in order.
ACE_HD void dense_replay(const AceDenseArgs &d, const AceGeom &g, const AceLds &lds, DenseState &own, unsigned char *ws, uint32_t lane,
                         uint32_t stored, int n_st) {
    DenseRecord r[3];
    auto fetch = [&](uint32_t round, DenseRecord &rec) {
        const uint32_t i = round * kDenseWidth + lane;
        dense_load(ws, i < stored ? i : stored - 1u, rec);
    };
    if (stored == 0u) return;                                      // (plans of more stages than there may be)
    const uint32_t rounds = (stored + kDenseWidth - 1u) / kDenseWidth;
    fetch(0, r[0]);
    fetch(1, r[1]);
    fetch(2, r[2]);
    for (uint32_t base = 0; base < rounds; base += 3u) {
#pragma unroll
        for (uint32_t k = 0; k < 3u; ++k) {
            const uint32_t round = base + k;
            if (round >= rounds) break;
            DenseState st;
            dense_stage(d, g, lds, own, r[k], st);
            const uint32_t place = r[k].tail.w;
            if (round + 3u < rounds) fetch(round + 3u, r[k]);
            if (round * kDenseWidth + lane < stored)
                *reinterpret_cast<ace_d2 *>(ws + kDenseResults + (place >> 7) * 1024u + ((place >> 1) & 63u) * 16u) = ace_d2{st.sum_t, st.max_mem};
        }
    }
#ifndef ACE_HOST_EMU
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#endif
    const int n = n_st < ACE_MAX_STAGES ? n_st : ACE_MAX_STAGES;
    for (int base = 0; base < ACE_MAX_STAGES; base += 4) {
        if (!ACE_ANY(base < n)) return;
        ace_d2 v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = base + k < n ? *reinterpret_cast<const ace_d2 *>(ws + kDenseResults + (uint32_t)(base + k) * 1024u + lane * 16u) : ace_d2{0.0, 0.0};
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (base + k < n) {
                own.sum_t += v[k].x;
                own.max_t = ace_max(own.max_t, v[k].x);
                own.max_mem = ace_max(own.max_mem, v[k].y);
            }
    }
}

#ifndef ACE_HOST_EMU
#include "ace_dense_loop_asm.inc"

// The op loop: returns the number of stages of the lane's plan, and in `stored` that of the wavefront's records; `ws`: the
// wavefront's part of the workspace.
template <bool WIN, int LANES>
__device__ __forceinline__ uint32_t dense_loop(const AceKernelArgs &a, const AceDenseArgs &d, uint64_t glogs, uint32_t lut2, uint64_t zvrk, uint32_t code_off,
                                               const unsigned char *ws, uint32_t lane, uint32_t meta0, uint32_t pace, uint32_t prio, uint32_t wave, uint32_t &stored) {
    uint32_t placed;
    const uint64_t gstride = (uint64_t)(uint32_t)a.g.P * 16u;
    const uint32_t gs_lo = (uint32_t)gstride, gs_hi = (uint32_t)(gstride >> 32);
#define ACE_DENSE_RUN(TEXT, ...)                                                                                                  \
    asm volatile(TEXT : [placed] "=&v"(placed), [stored] "=&v"(stored)                                                           \
                 : [glogs] "v"(glogs), [lut2] "v"(lut2), [zvrk] "v"(zvrk), [codeoff] "v"(code_off), [place] "v"(lane * 2u),      \
                   [meta0] "v"(meta0), [codes] "s"(a.codes), [pos] "s"(d.pos), [n_ops] "s"(a.g.N), [recbase] "s"(ws),            \
                   [gstride_lo] "s"(gs_lo), [gstride_hi] "s"(gs_hi), [kv] "s"(d.kv), __VA_ARGS__ \
                 : ACE_DENSE_ASM_CLOBBERS)
#define ACE_DENSE_RESIDENT [pace] "s"(pace), [pacemask] "s"((uint32_t)LANES / 512u)
#define ACE_DENSE_WINDOWED [prio] "s"(prio), [dma] "s"(d.events), [eventsize] "s"((uint32_t)(kDenseWinLanes / 64) * 48u), \
                           [waveoff] "s"(wave * 48u), [half] "s"(d.half), [luthalf] "s"(d.lut_half)
    if (WIN) {
        if (a.g.flags & ACE_F_RESHARDING) ACE_DENSE_RUN(ACE_DENSE_ASM_WIN_RSH1, ACE_DENSE_WINDOWED);
        else ACE_DENSE_RUN(ACE_DENSE_ASM_WIN_RSH0, ACE_DENSE_WINDOWED);
    } else {
        if (a.g.flags & ACE_F_RESHARDING) ACE_DENSE_RUN(ACE_DENSE_ASM_RSH1, ACE_DENSE_RESIDENT);
        else ACE_DENSE_RUN(ACE_DENSE_ASM_RSH0, ACE_DENSE_RESIDENT);
    }
#undef ACE_DENSE_RUN
#undef ACE_DENSE_RESIDENT
#undef ACE_DENSE_WINDOWED
    return placed >> 7;
}

// Windowed rows: the fetches of a wavefront without plans, in step with the loops of the others (fetch_event of
// gen_dense_loop_asm.py).  As many events as they have: every barrier is met.
__device__ __forceinline__ void dense_fetch(const AceDenseArgs &d, unsigned char *lds_raw, uint32_t wave, uint32_t lane) {
    typedef const void __attribute__((address_space(1))) *gptr;
    typedef void __attribute__((address_space(3))) *lptr;
    for (uint32_t e = 0; e < d.n_events; ++e) {
        const uint32_t *rec = reinterpret_cast<const uint32_t *>(d.events + (e * (uint32_t)(kDenseWinLanes / 64) + wave) * 48u);
        const unsigned char *rows = reinterpret_cast<const unsigned char *>(((uint64_t)rec[3] << 32) | rec[2]);
        const uint32_t n = (rec[1] >> 8) & 15u, wait = rec[1] & 1u;
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n s_barrier" ::: "memory");
        for (uint32_t k = 0; k < n; ++k) {
            const uint32_t from = (uint32_t)__builtin_amdgcn_readfirstlane((int)rec[4 + 2 * k]), to = (uint32_t)__builtin_amdgcn_readfirstlane((int)rec[5 + 2 * k]);
            __builtin_amdgcn_global_load_lds((gptr)(rows + from + lane * 16u), (lptr)(lds_raw + to), 16, 0, 0);
        }
        if (wait) asm volatile("s_waitcnt vmcnt(0)\n s_barrier" ::: "memory");
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// The tables, to LDS address 0 on, by the LANES lanes of the workgroup: 1 KB per wavefront and load, all in flight at once.
template <int LANES> __device__ __forceinline__ void dense_stage_image(const AceDenseArgs &d, unsigned char *lds_raw, uint32_t wave, uint32_t lane) {
    typedef const void __attribute__((address_space(1))) *gptr;
    typedef void __attribute__((address_space(3))) *lptr;
    for (uint32_t at = wave * 64u; at < d.image16; at += LANES)
        if (at + lane < d.image16) __builtin_amdgcn_global_load_lds((gptr)(d.image + at + lane), (lptr)(lds_raw + at * 16u), 16, 0, 0);
}

// One workgroup; its LDS array starts at address 0 (the kernel has no other LDS variables).
template <bool WIN, int LANES> __device__ __forceinline__ void ace_dense_body(const AceKernelArgs &a, const AceDenseArgs &d, uint32_t slices, unsigned char *lds_raw,
                                                                int tid, long long block) {
    constexpr int kLanes = LANES;
    static_assert(!WIN || LANES == kDenseWinLanes, "as many wavefronts as the fetch records say");
    const AceGeom &g0 = a.g;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(tid >> 6), lane = (uint32_t)tid & 63u;
    const uint32_t lanes = 64u * slices;
    dense_stage_image<kLanes>(d, lds_raw, wave, lane);
    // Deal: counting sort of the plans by pipeline depth, the deepest first (see ace_score_body); sorted slice q goes to
    // wavefront q in rows of four, every second row reversed: each SIMD gets the same mix.
    unsigned int *cnt = reinterpret_cast<unsigned int *>(lds_raw + d.image16 * 16u);
    unsigned short *plan_of = reinterpret_cast<unsigned short *>(cnt + 32);
    uint32_t *pace = reinterpret_cast<uint32_t *>(plan_of + kLanes);
    const uint32_t q = (wave & 4u) ? wave ^ 3u : wave;
    if (tid < 32) { cnt[tid] = 0u; if (!WIN) pace[tid] = 0u; }
    const long long slot = block * lanes + tid;
    uint32_t depth = 0, rank = 0;                                   // (slots past the batch: last)
    if ((uint32_t)tid < lanes && slot < g0.P) {
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
    const bool in_batch = plan < g0.P;
    const long long pl = in_batch ? plan : (long long)g0.P - 1;     // plan this lane reads
    const long long out = a.order ? (long long)a.order[pl] : plan;
    const bool active = in_batch && out < g0.P;
    const ace_u4 h = a.hdr[pl];
    const uint32_t first = a.codes[pl].x & 0x1fu;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                 // the tables
    __syncthreads();
    if (q >= slices) {
        if (WIN) dense_fetch(d, lds_raw, wave, lane);
        return;
    }

    AceGeom g = g0;
    g.out_off = 0u;                                                 // (what the evaluation indexes the outputs' addresses by)
    const AceLds lds = ace_make_lds(lds_raw, 0u);
    DenseState st;
    st.init(g, lds, h, ace_u2{0u, 0u});
    if (!(first & 0x10u)) st.status = ACE_PLAN_MALFORMED;            // the first op must open a stage
    const uint32_t lut = d.lut_off + st.bidx * 128u;
    unsigned char *ws = reinterpret_cast<unsigned char *>(a.stage_ws) + ((size_t)block * slices + q) * kDenseWave;
    const uint64_t zvrk = lds.ld<uint64_t>(lut + ((uint32_t)st.glogs & 15u) * 8u);
    uint32_t stored;
    // (windowed rows: the deeper its plans, the higher a wavefront's issue priority)
    const uint32_t prio = (uint32_t)__builtin_amdgcn_readfirstlane((int)(3u - q * 4u / (uint32_t)(kLanes / 64)));
    const int n_st = (int)dense_loop<WIN, LANES>(a, d, st.glogs >> 1, lut, zvrk, (uint32_t)pl * 16u, ws, lane, ((first & 7u) << 8) | (d.first_in << 24),
                                             d.image16 * 16u + 128u + 2u * kLanes + (wave & 3u) * 32u, prio, wave, stored);
    dense_replay(d, g, lds, st, ws, lane, (uint32_t)__builtin_amdgcn_readfirstlane((int)stored), n_st);
    st.s = n_st;                                                    // (result() checks the count of the op loop)
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
