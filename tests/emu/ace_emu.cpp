// Bounds-checked CPU build of the per-plan state machine (superscaler_amd/csrc/ace_plan_state.h)
// -- TEST INFRASTRUCTURE ONLY.  It lets the CPU test-suite run the exact source the GPU kernel
// is made of (same header, compiled with ACE_HOST_EMU) against the oracle, with every "LDS"
// access checked for range and alignment, before anything is launched on a GPU.  The product
// library never links or loads this file.
#define ACE_HOST_EMU 1
#include "ace_edit_kernels.h"
#include "ace_grid.h"
#include "ace_score_loop.h"
#include "ace_dense.h"
#include "ace_route.h"
#include "ace_spread.h"
#include "ace_recompute.h"
#include "ace_pack.h"

#include <sys/mman.h>

#include <vector>

namespace {

template <bool BD, bool RANGED, bool DEFER = false, bool COLL = false>
void score_one(const ace_tables_t *t, const AceGeom &g, std::vector<unsigned char> &lds, uint32_t lds_bytes,
               const uint8_t *codes, ace_u4 h, ace_u2 range, double *rec, double &iter, double &peak, uint8_t &feas,
               uint8_t &st) {
    const size_t row_bytes = (size_t)t->row_doubles * 8;
    const uint32_t *pos = t->pos_info;
    AceLds view{lds.data(), lds_bytes};
    PlanState<BD, RANGED, DEFER, COLL> s;
    std::vector<double> ws(ACE_MAX_STAGES * ACE_WS_REC, __builtin_nan(""));
    if (DEFER) rec = ws.data();
    s.init(g, view, h, range);
    int w = 0, next_win = t->win_pos[0];
    for (int i = 0; i < g.N; ++i) {
        if (i == next_win) {
            // poison, then stage exactly the rows the window lists: a read of any other row yields NaN
            memset(lds.data(), 0xff, t->lds_row_bytes);
            for (int r = t->win_row_begin[w]; r < t->win_row_begin[w + 1]; ++r)
                memcpy(lds.data() + t->win_rows[2 * r + 1], t->rows + (size_t)t->win_rows[2 * r] * t->row_doubles, row_bytes);
            next_win = t->win_pos[++w];
        }
        if (!RANGED && i == 0) s.begin(g, view, 0, codes[0], pos[0]);
        const uint32_t nbyte = i + 1 < g.N ? codes[i + 1] : 0u;
        s.step(g, view, i, codes[i], nbyte, pair_bit(codes[i], nbyte), pos[i], i > 0 ? pos[i - 1] : 0u, i + 1 == g.N, rec);
    }
    if (DEFER) {
        s.replay_all(g, view, rec, s.s, codes[0] & 7u, pos[0] & 0xffu);
    }
    s.result(g, t->nb_minus_1[s.bidx], iter, peak, feas, st);
}

}  // namespace

extern "C" int ace_emu_score(const ace_tables_t *t, const uint8_t *codes /* [P][N] plan-major */,
                             const uint32_t *hdr /* [P][4] */, const uint32_t *range /* nullable [P][2] */,
                             long long P, double memory_limit, int strict, int defer, double *iter_ms, double *peak_mb,
                             uint8_t *feasible, uint8_t *status, double *stage_out /* nullable [P][16][18]; with ranges [P][18] */) {
    const int C = t->n_tp * t->n_algo;
    AceGeom g;
    memset(&g, 0, sizeof(g));
    g.N = t->num_ops; g.P = (int32_t)P; g.G = (t->num_ops + 15) / 16;
    g.C = C; g.A_shift = t->n_algo == 2 ? 1 : 0;
    g.n_mbs = t->n_mbs; g.n_tp = t->n_tp; g.n_algo = t->n_algo; g.n_glog = t->n_glog; g.n_pair_kinds = t->n_pair_kinds;
    g.hot_off = t->hot_off * 8u; g.start_off = t->start_off * 8u; g.out_off = t->out_off * 8u; g.z_off = t->z_off * 8u;
    g.z_shift = 3;
    while ((1 << (g.z_shift - 3)) < t->z_table_doubles) ++g.z_shift;
    g.zm_delta = (uint32_t)t->n_z << g.z_shift;
    const int32_t rk_bytes = t->n_pair_kinds * t->n_glog * 64;
    g.rk_lds_off = (uint32_t)t->lds_row_bytes;
    const uint32_t lds_bytes = ace_lds_layout(g.rk_lds_off, (uint32_t)rk_bytes, (uint32_t)t->n_mbs * 16u, &g.stg_lds_off, &g.lut2_lds_off);
    g.rk_kind_stride = (uint32_t)(t->n_glog * 64);
    g.row_bytes = (uint32_t)t->row_doubles * 8u;
    g.flags = t->flags; g.main_params = t->main_params; g.optimizer = t->optimizer;
    g.mem_limit = memory_limit; g.strict = strict ? 1 : 0;
    if (range && !stage_out) return -1;

    std::vector<unsigned char> lds(lds_bytes);
    for (long long p = 0; p < P; ++p) {
        memset(lds.data(), 0xff, lds.size());
        memcpy(lds.data() + g.rk_lds_off, t->pair_kinds, rk_bytes);
        memcpy(lds.data() + g.stg_lds_off, t->stage_lut, (size_t)t->n_mbs * 16 * 4);
        for (int j = 0; j < t->n_mbs * 16; ++j) {       // (as the kernel's staging loop fills this region)
            const uint32_t glog = (uint32_t)j & 15u, z_v = (t->stage_lut[j] & 15u) * (uint32_t)C * 8u;
            const ace_u2 e{z_v, ((glog < (uint32_t)t->n_glog ? glog : 0u) << 6) - z_v};
            memcpy(lds.data() + g.lut2_lds_off + 8 * j, &e, 8);
        }
        ace_u4 h;
        memcpy(&h, hdr + 4 * p, 16);
        ace_u2 rg{0u, 0u};
        if (range) memcpy(&rg, range + 2 * p, 8);
        double *rec = stage_out ? stage_out + (size_t)p * (range ? 1 : ACE_MAX_STAGES) * ACE_STAGE_REC : nullptr;
        const uint8_t *c = codes + (size_t)p * g.N;
        double iter, peak;
        uint8_t feas, st;
        const bool coll = (t->flags & ACE_F_COLLECTIVE_MEM) != 0;
        if (coll) {
            if (range) score_one<true, true, false, true>(t, g, lds, lds_bytes, c, h, rg, rec, iter, peak, feas, st);
            else if (stage_out) score_one<true, false, false, true>(t, g, lds, lds_bytes, c, h, rg, rec, iter, peak, feas, st);
            else score_one<false, false, false, true>(t, g, lds, lds_bytes, c, h, rg, rec, iter, peak, feas, st);
        }
        else if (range) score_one<true, true>(t, g, lds, lds_bytes, c, h, rg, rec, iter, peak, feas, st);
        else if (stage_out) score_one<true, false>(t, g, lds, lds_bytes, c, h, rg, rec, iter, peak, feas, st);
        else if (defer && t->n_windows == 1) score_one<false, false, true>(t, g, lds, lds_bytes, c, h, rg, rec, iter, peak, feas, st);
        else score_one<false, false>(t, g, lds, lds_bytes, c, h, rg, rec, iter, peak, feas, st);
        iter_ms[p] = iter; peak_mb[p] = peak; feasible[p] = feas;
        if (status) status[p] = st;
    }
    return 0;
}


// ------------------------------------------------------------------------------------------
// The dense tables (ace_dense.h): built as the library builds them and walked as the assembly loop walks them -- one dot product per
// address, ranks, parked records -- with every read checked against the image.  Returns 1 if the tables do not fit that form.
// ------------------------------------------------------------------------------------------
extern "C" int ace_emu_dense(const ace_tables_t *t, const uint8_t *codes /* [P][N] */, const uint32_t *hdr, long long P, double memory_limit,
                             int strict, double *iter_ms, double *peak_mb, uint8_t *feasible, uint8_t *status, int32_t *shape /* [4] */) {
    const int N = t->num_ops;
    const size_t pos_entries = (size_t)((N + 15) / 16) * 16 + 16;
    AceDenseTables d;
    ace_dense_build(t, pos_entries, d);
    if (!d.ok) return 1;
    shape[0] = (int32_t)d.image.size(); shape[1] = (int32_t)d.array; shape[2] = (int32_t)(d.args.rb_off - d.args.rf_off) / 8; shape[3] = (int32_t)d.args.kv;
    const bool rsh = (t->flags & ACE_F_RESHARDING) != 0;
    AceGeom g;
    memset(&g, 0, sizeof(g));
    g.N = N; g.P = (int32_t)P; g.C = t->n_tp * t->n_algo; g.A_shift = t->n_algo == 2 ? 1 : 0;
    g.n_mbs = t->n_mbs; g.n_tp = t->n_tp; g.n_algo = t->n_algo; g.n_glog = t->n_glog;
    g.hot_off = t->hot_off * 8u; g.start_off = t->start_off * 8u; g.out_off = t->out_off * 8u; g.z_off = t->z_off * 8u;
    g.row_bytes = (uint32_t)t->row_doubles * 8u;
    g.flags = t->flags; g.main_params = t->main_params; g.optimizer = t->optimizer;
    g.mem_limit = memory_limit; g.strict = strict ? 1 : 0;
    const AceDenseArgs &da = d.args;
    // (windowed rows: both halves behind the image; a window's rows are put there before its first op, everything else is poisoned)
    std::vector<unsigned char> mem(std::max<size_t>(d.lds, d.image.size()), 0xff);
    memcpy(mem.data(), d.image.data(), d.image.size());
    const AceLds lds{mem.data(), (uint32_t)(d.windows.empty() ? d.image.size() : d.rows_off + 2u * da.half)};
    g.out_off = 0u;
    auto dot = [](uint32_t a, uint32_t b, uint32_t c) {
        for (int k = 0; k < 4; ++k) c += ((a >> (8 * k)) & 255u) * ((b >> (8 * k)) & 255u);
        return c;
    };
    for (long long p = 0; p < P; ++p) {
        auto code = [&](int i) { return i < N ? (uint32_t)(codes[(size_t)p * N + i] & 0x1fu) : i == N ? 0x10u : 0u; };
        ace_u4 h;
        memcpy(&h, hdr + 4 * p, 16);
        DenseState st;
        st.init(g, lds, h, ace_u2{0u, 0u});
        if (!(code(0) & 0x10u)) st.status = ACE_PLAN_MALFORMED;
        std::vector<unsigned char> ws(kDenseWave, 0xff);                // (a wavefront of one lane)
        uint64_t glogs = st.glogs;
        auto stage = [&]() {
            const ace_u2 z = lds.ld<ace_u2>(da.lut_off + st.bidx * 128u + ((uint32_t)glogs & 15u) * 8u);
            glogs >>= 4;
            return z;
        };
        ace_u2 z = stage();
        double fwd = 0, bwd = 0, rcs = 0, rsf = 0, rsb = 0, w = 0, act = 0, saved = 0, peak = 0, run = 0;
        uint32_t rf = 0, rb = 0, cost = 0, before = (code(0) & 7u) << 8 | da.first_in << 24;
        int n_st = 0;
        size_t win = 0;
        uint32_t half = 0;
        for (int i = 0; i < N; ++i) {
            if (win < d.windows.size() && d.window_start[win] == i) {
                half = win & 1 ? da.half : 0u;
                memset(mem.data() + d.rows_off, 0xff, 2u * da.half);
                for (size_t s = 0; s < d.windows[win].size(); ++s)
                    memcpy(mem.data() + d.rows_off + half + s * d.row_pitch, d.rows.data() + (size_t)d.windows[win][s] * d.row_pitch, d.row_pitch);
                ++win;
            }
            const uint32_t b = code(i), nb = code(i + 1);
            const ace_u4 &pos = d.pos[i];
            uint32_t word = 0;                                          // codes from the even position on, behind them the constant(s)
            for (int k = 0; k < (rsh ? 3 : 2); ++k) word |= (code((i & ~1) + k) & 7u) << (8 * k);
            word |= da.kv;
            const uint32_t e = dot(word, pos.x, z.x) + half;
            const double v[4] = {lds.ld<double>(e), lds.ld<double>(e + d.array), lds.ld<double>(e + 2 * d.array), lds.ld<double>(e + 3 * d.array)};
            const uint32_t ranks = lds.ld<uint32_t>(e + 4 * d.array);
            fwd += v[0]; bwd += v[1]; w += v[2]; act += v[3];
            if (rsh) {
                const ace_d2 c = lds.ld<ace_d2>(cost);
                rsf += c.x; rsb += c.y;
                cost = lds.ld<uint16_t>(dot(word, pos.y, z.y));
            }
            const bool last = (nb >> 4) & 1u, rc = (b >> 3) & 1u, pair = rc && ((nb >> 3) & 1u) && !last, keep = pair && (pos.w & 1u);
            if (last && !(i > 0 && (d.pos[i - 1].w & 2u))) run = 0.0;
            if (!last) {
                rf = (ranks & 0xffffu) > rf ? ranks & 0xffffu : rf;
                rb = (ranks >> 16) > rb ? ranks >> 16 : rb;
            }
            if (rc) rcs += v[0];
            if (pair) run += v[3];
            if (keep) saved += v[3];
            else { peak = ace_max(peak, run); run = 0.0; }
            if (!last) continue;
            if (n_st < ACE_MAX_STAGES) {
                const double vals[8] = {fwd + bwd, rcs, rsf, rsb, w, act, saved, peak};
                for (uint32_t j = 0; j < 4u; ++j) memcpy(ws.data() + j * kDensePiece + (uint32_t)n_st * 16u, vals + 2 * j, 16);
                const uint32_t even = (b & 7u) | (nb & 7u) << 8, odd = (b & 7u) << 8 | (nb & 7u) << 16;
                const uint32_t word = (rsh && (i & 1) ? odd : even) | pos.z;
                const ace_u4 tail{rf | rb << 16, word, before, (uint32_t)n_st * 128u};
                memcpy(ws.data() + 4u * kDensePiece + (uint32_t)n_st * 16u, &tail, 16);
                before = word;
            }
            ++n_st;
            fwd = bwd = rcs = rsf = rsb = w = act = saved = peak = run = 0.0;
            rf = rb = cost = 0;
            z = stage();
        }
        dense_replay(da, g, lds, st, ws.data(), 0u, (uint32_t)(n_st < ACE_MAX_STAGES ? n_st : ACE_MAX_STAGES), n_st);
        st.s = n_st;
        uint8_t feas, stat;
        st.result(g, t->nb_minus_1[st.bidx], iter_ms[p], peak_mb[p], feas, stat);
        feasible[p] = feas;
        status[p] = stat;
    }
    return 0;
}

// What the tables of that form are like: fits, windows, bytes of LDS per workgroup, of the image, of a row (with what follows it to the
// next one), most rows of a window.
extern "C" void ace_emu_dense_shape(const ace_tables_t *t, int32_t *out /* [6] */) {
    AceDenseTables d;
    ace_dense_build(t, (size_t)((t->num_ops + 15) / 16) * 16 + 16, d);
    size_t most = 0;
    for (const auto &w : d.windows) most = std::max(most, w.size());
    const int32_t v[6] = {d.ok, (int32_t)d.windows.size(), (int32_t)d.lds, (int32_t)d.image.size(), (int32_t)d.row_pitch, (int32_t)most};
    memcpy(out, v, sizeof(v));
}

// Which kernel a batch takes (AceKernelId).  `other`: what the table compiler's rows allow beside the dense tables (1: the assembly loop, 2: the
// C++ loop with deferred stage tails, 3: both), which the library finds out as it lays its own tables out.
static AceRouteTables emu_route_tables(const ace_tables_t *t, int other) {
    AceDenseTables d;
    ace_dense_build(t, (size_t)((t->num_ops + 15) / 16) * 16 + 16, d);
    AceRouteTables r{};
    r.ops = t->num_ops;
    r.spread = true;
    r.dense = d.ok;
    r.dense_windows = (int32_t)d.windows.size();
    r.dense_lanes = d.lanes;
    r.many = other & 1;
    r.windows = t->n_windows;
    r.deferred = other & 2;
    return r;
}
extern "C" int ace_emu_route(const ace_tables_t *t, long long plans, int records, int other, size_t workspace) {
    return ace_route(emu_route_tables(t, other), plans, records != 0, workspace);
}
// ... and the bytes of workspace that the library gets for it.
extern "C" size_t ace_emu_workspace(const ace_tables_t *t, long long plans, int other) { return ace_workspace(emu_route_tables(t, other), plans); }

// ------------------------------------------------------------------------------------------
// The kernel's own op loop (ace_score_loop.h) on the CPU, one lane per "workgroup", with every
// array the kernel reads or writes placed flush against an inaccessible page: an index past an
// array's end (or a page or more before its start) ends the process with SIGSEGV instead of
// going unnoticed.  Callers run this in a child process.
// ------------------------------------------------------------------------------------------
namespace {

struct GuardedPool {
    struct Map { void *base; size_t len; };
    std::vector<Map> maps;
    // a writable copy of `bytes` bytes of `src` (zeros if null) whose end (rounded up to `align` bytes, the
    // alignment the kernel's loads of that array need) touches a PROT_NONE page
    void *place(const void *src, size_t bytes, size_t align = 16) {
        const size_t pg = 4096, body = (bytes + pg - 1) / pg * pg + pg;
        unsigned char *m = (unsigned char *)mmap(nullptr, body + 2 * pg, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
        if (m == MAP_FAILED) { perror("mmap"); abort(); }
        mprotect(m, pg, PROT_NONE);
        mprotect(m + pg + body, pg, PROT_NONE);
        maps.push_back({m, body + 2 * pg});
        unsigned char *p = m + pg + body - ((bytes + align - 1) / align * align);
        if (src) memcpy(p, src, bytes);
        return p;
    }
    ~GuardedPool() { for (auto &m : maps) munmap(m.base, m.len); }
};

template <bool BD, bool RANGED, bool WIN, bool DEFER, bool COLL = false>
void run_lanes(const AceKernelArgs &a, unsigned char *lds, uint32_t lds_bytes) {
    for (long long p = 0; p < a.g.P; ++p) {
        memset(lds, 0xff, lds_bytes);
        ace_score_body<BD, RANGED, WIN, DEFER, 1, COLL>(a, lds, lds_bytes, 0, p, (uint32_t)a.g.P);
    }
}

// The kernel of small batches: its workgroup's lanes one after the other within each phase, LDS behind guard pages.
template <bool BD, bool RANGED, bool COLL>
void run_spread(const AceKernelArgs &a, GuardedPool &pool) {
    SpreadShared sh;
    const uint32_t bytes = ace_spread_layout(SpreadCols<BD, COLL>::kCols, a.g.G, nullptr, &sh);
    unsigned char *lds = (unsigned char *)pool.place(nullptr, bytes);
    for (long long p = 0; p < a.g.P; ++p) {
        memset(lds, 0xff, bytes);
        ace_spread_body<BD, RANGED, COLL>(a, lds, 0, p);
    }
}
template <bool BD, bool RANGED> void run_spread_c(const AceKernelArgs &a, GuardedPool &pool) {
    if (a.g.flags & ACE_F_COLLECTIVE_MEM) run_spread<BD, RANGED, true>(a, pool);
    else run_spread<BD, RANGED, false>(a, pool);
}

struct RcJob {
    const int32_t *type_of_pos;
    const double *activations;
    const uint8_t *no_recompute, *status;
    double peak_backward;
    uint8_t *codes_out;
    int32_t *flags;
};
int emu_kernel(const ace_tables_t *t, const uint8_t *codes, const uint32_t *hdr, const uint32_t *range, const uint32_t *order, long long P,
               double memory_limit, int strict, double *iter_ms, double *peak_mb, uint8_t *feasible, uint8_t *status, double *stage_out,
               bool spread, const RcJob *rc = nullptr);

}  // namespace

// codes: uint8 [G][P][16] (the kernel's layout).  Chooses the kernel variant as the library's launcher does.
extern "C" int ace_emu_kernel(const ace_tables_t *t, const uint8_t *codes, const uint32_t *hdr, const uint32_t *range,
                              const uint32_t *order /* nullable [P] */, long long P, double memory_limit, int strict,
                              double *iter_ms, double *peak_mb, uint8_t *feasible, uint8_t *status, double *stage_out) {
    return emu_kernel(t, codes, hdr, range, order, P, memory_limit, strict, iter_ms, peak_mb, feasible, status, stage_out, false);
}
// ... and the kernel of small batches.
extern "C" int ace_emu_spread(const ace_tables_t *t, const uint8_t *codes, const uint32_t *hdr, const uint32_t *range,
                              const uint32_t *order /* nullable [P] */, long long P, double memory_limit, int strict,
                              double *iter_ms, double *peak_mb, uint8_t *feasible, uint8_t *status, double *stage_out) {
    return emu_kernel(t, codes, hdr, range, order, P, memory_limit, strict, iter_ms, peak_mb, feasible, status, stage_out, true);
}

// LDS that check_recompute's workgroup may take: decides about its wavefronts
extern "C" { uint32_t ace_emu_rc_lds = 160u * 1024u; }
// ... and whether the arguments of the launch say how many groups and wavefronts there are (0: they are left as they come)
extern "C" { int32_t ace_emu_rc_set = 1; }
// ... and how many wavefronts it has with that much
extern "C" int ace_emu_rc_waves(int N, int groups) { return ace_rc_waves(N, (N + 15) / 16, groups, ace_emu_rc_lds); }

// ace_recompute_batch: codes and codes_out uint8 [G][P][16], flags int32 [4] zeroed by the caller.
extern "C" int ace_emu_recompute(const ace_tables_t *t, const uint8_t *codes, const uint32_t *hdr, long long P, double memory_limit,
                                 double peak_backward, const int32_t *type_of_pos, const double *activations, const uint8_t *no_recompute,
                                 const uint8_t *status, uint8_t *codes_out, int32_t *flags) {
    const RcJob rc{type_of_pos, activations, no_recompute, status, peak_backward, codes_out, flags};
    std::vector<double> d((size_t)P);
    std::vector<uint8_t> b((size_t)P);
    return emu_kernel(t, codes, hdr, nullptr, nullptr, P, memory_limit, 0, d.data(), d.data(), b.data(), nullptr, nullptr, true, &rc);
}

namespace {
int emu_kernel(const ace_tables_t *t, const uint8_t *codes, const uint32_t *hdr, const uint32_t *range, const uint32_t *order, long long P,
               double memory_limit, int strict, double *iter_ms, double *peak_mb, uint8_t *feasible, uint8_t *status, double *stage_out,
               bool spread, const RcJob *rc) {
    if (range && !stage_out) return -1;
    AceKernelArgs a;
    memset(&a, 0, sizeof(a));
    AceGeom &g = a.g;
    const int C = t->n_tp * t->n_algo;
    g.N = t->num_ops; g.P = (int32_t)P; g.G = (t->num_ops + 15) / 16;
    g.C = C; g.A_shift = t->n_algo == 2 ? 1 : 0;
    g.n_mbs = t->n_mbs; g.n_tp = t->n_tp; g.n_algo = t->n_algo; g.n_glog = t->n_glog; g.n_pair_kinds = t->n_pair_kinds;
    g.hot_off = t->hot_off * 8u; g.start_off = t->start_off * 8u; g.out_off = t->out_off * 8u; g.z_off = t->z_off * 8u;
    g.z_shift = 3;
    while ((1 << (g.z_shift - 3)) < t->z_table_doubles) ++g.z_shift;
    g.zm_delta = (uint32_t)t->n_z << g.z_shift;
    a.rk_bytes = t->n_pair_kinds * t->n_glog * 64;
    g.rk_lds_off = (uint32_t)t->lds_row_bytes;
    a.stg_words = t->n_mbs * 16;
    const uint32_t lds_bytes = ace_lds_layout(g.rk_lds_off, (uint32_t)a.rk_bytes, (uint32_t)a.stg_words, &g.stg_lds_off, &g.lut2_lds_off);
    g.rk_kind_stride = (uint32_t)(t->n_glog * 64);
    g.row_bytes = (uint32_t)t->row_doubles * 8u;
    g.flags = t->flags; g.main_params = t->main_params; g.optimizer = t->optimizer;
    g.mem_limit = memory_limit; g.strict = strict ? 1 : 0;
    a.n_windows = t->n_windows; a.row_doubles = t->row_doubles;

    GuardedPool pool;
    const size_t G = (size_t)g.G, n_win_rows = (size_t)t->win_row_begin[t->n_windows];
    a.codes = (const ace_u4 *)pool.place(codes, G * (size_t)P * 16);
    a.hdr = (const ace_u4 *)pool.place(hdr, (size_t)P * 16);
    a.range = range ? (const ace_u2 *)pool.place(range, (size_t)P * 8, 8) : nullptr;
    a.order = order ? (const uint32_t *)pool.place(order, (size_t)P * 4, 4) : nullptr;
    a.rows = (const double *)pool.place(t->rows, (size_t)t->num_types * t->row_doubles * 8);
    // (the library uploads the num_ops + 1 descriptors into a zeroed array of 16 * G + 16)
    uint32_t *pos = (uint32_t *)pool.place(nullptr, (G * 16 + 16) * 4);
    memcpy(pos, t->pos_info, (size_t)(t->num_ops + 1) * 4);
    a.pos_info = pos;
    if (t->n_windows > 1 && t->num_types <= 256) {
        uint32_t *pt = (uint32_t *)pool.place(nullptr, (G * 16 + 16) * 4);
        ace_pos_types(t, pt, G * 16 + 16);
        a.pos_types = pt;
    }
    a.pair_kinds = (const uint8_t *)pool.place(t->pair_kinds, (size_t)a.rk_bytes, 4);
    a.stage_lut = (const uint32_t *)pool.place(t->stage_lut, (size_t)a.stg_words * 4, 4);
    a.nbm1 = (const double *)pool.place(t->nb_minus_1, (size_t)t->n_mbs * 8, 8);
    a.win_pos = (const int32_t *)pool.place(t->win_pos, (size_t)(t->n_windows + 1) * 4, 4);
    a.win_row_begin = (const int32_t *)pool.place(t->win_row_begin, (size_t)(t->n_windows + 1) * 4, 4);
    a.win_rows = (const uint32_t *)pool.place(t->win_rows, n_win_rows * 8, 4);
    // (what the library works out at ace_create: resident rows that lie in LDS as in global memory are staged as one block)
    if (t->n_windows == 1 && (t->row_doubles & 1) == 0) {
        bool flat = true;
        for (int r = 0; r < t->win_row_begin[1]; ++r)
            flat = flat && t->win_rows[2 * r] == (uint32_t)r && t->win_rows[2 * r + 1] == (uint32_t)r * (uint32_t)t->row_doubles * 8u;
        if (flat) a.flat_rows16 = t->win_row_begin[1] * (t->row_doubles / 2);
    }
    a.iter_ms = (double *)pool.place(iter_ms, (size_t)P * 8, 8);
    a.peak_mb = (double *)pool.place(peak_mb, (size_t)P * 8, 8);
    a.feasible = (uint8_t *)pool.place(feasible, (size_t)P, 1);
    a.status = status ? (uint8_t *)pool.place(status, (size_t)P, 1) : nullptr;
    const size_t rec_bytes = (size_t)P * (range ? 1 : ACE_MAX_STAGES) * ACE_STAGE_REC * 8;
    a.stage_out = stage_out ? (double *)pool.place(stage_out, rec_bytes, 8) : nullptr;   // (records of unused stages stay as the caller left them)
    unsigned char *lds = (unsigned char *)pool.place(nullptr, lds_bytes);
    if (spread) {
        // (as the library uploads them: positions padded, zeros behind the last row)
        ace_u2 *ps = (ace_u2 *)pool.place(nullptr, (G * 16 + 16) * 8, 8);
        ace_pos_spread(t, ps, G * 16 + 16);
        a.pos_spread = ps;
        const size_t rows = (size_t)t->num_types * t->row_doubles * 8;
        double *padded = (double *)pool.place(nullptr, rows + 4096);
        memcpy(padded, t->rows, rows);
        a.rows = padded;
        if (rc) {
            const size_t N = (size_t)g.N, n_act = (size_t)t->num_types * t->n_mbs * t->n_tp * t->n_algo;
            RcArgs r;
            r.k = a;
            ace_u2 *pos = (ace_u2 *)pool.place(nullptr, N * 8, 8);
            const int groups = ace_rc_positions(rc->type_of_pos, rc->no_recompute, g.N, t->num_types, pos);
            if (ace_emu_rc_set) {
                r.groups = groups;
                r.waves = ace_rc_waves(g.N, (int)G, groups, ace_emu_rc_lds);
            }
            r.pos = pos;
            r.act = (const double *)pool.place(rc->activations, n_act * 8, 8);
            r.status = (const uint8_t *)pool.place(rc->status, (size_t)P, 1);
            r.codes_out = (ace_u4 *)pool.place(nullptr, G * (size_t)P * 16);
            r.flags = rc->flags;
            r.limit = memory_limit;
            r.peak_backward = rc->peak_backward;
            RcShared sh;
            const uint32_t bytes = ace_emu_rc_set ? ace_rc_layout(r, nullptr, &sh) : ace_rc_layout(g.N, g.G, nullptr, &sh);
            unsigned char *rlds = (unsigned char *)pool.place(nullptr, bytes);
            for (long long p = 0; p < P; ++p) {
                memset(rlds, 0xff, bytes);
                if (g.flags & ACE_F_COLLECTIVE_MEM) ace_rc_body<true>(r, rlds, 0, p);
                else ace_rc_body<false>(r, rlds, 0, p);
            }
            memcpy(rc->codes_out, r.codes_out, G * (size_t)P * 16);
            return 0;
        }
        if (range) run_spread_c<true, true>(a, pool);
        else if (stage_out) run_spread_c<true, false>(a, pool);
        else run_spread_c<false, false>(a, pool);
        memcpy(iter_ms, a.iter_ms, (size_t)P * 8);
        memcpy(peak_mb, a.peak_mb, (size_t)P * 8);
        memcpy(feasible, a.feasible, (size_t)P);
        if (status) memcpy(status, a.status, (size_t)P);
        if (stage_out) memcpy(stage_out, a.stage_out, rec_bytes);
        return 0;
    }
    const bool win = t->n_windows > 1;
    const bool coll = (t->flags & ACE_F_COLLECTIVE_MEM) != 0;
    const bool defer = !range && !stage_out && (!win || a.pos_types) && g.N < 32768 && !coll;
    if (defer) a.stage_ws = (double *)pool.place(nullptr, (size_t)P * ACE_MAX_STAGES * ACE_WS_REC * 8);

    if (coll) {
        if (range) { if (win) run_lanes<true, true, true, false, true>(a, lds, lds_bytes); else run_lanes<true, true, false, false, true>(a, lds, lds_bytes); }
        else if (stage_out) { if (win) run_lanes<true, false, true, false, true>(a, lds, lds_bytes); else run_lanes<true, false, false, false, true>(a, lds, lds_bytes); }
        else if (win) run_lanes<false, false, true, false, true>(a, lds, lds_bytes);
        else run_lanes<false, false, false, false, true>(a, lds, lds_bytes);
    }
    else if (range) { if (win) run_lanes<true, true, true, false>(a, lds, lds_bytes); else run_lanes<true, true, false, false>(a, lds, lds_bytes); }
    else if (stage_out) { if (win) run_lanes<true, false, true, false>(a, lds, lds_bytes); else run_lanes<true, false, false, false>(a, lds, lds_bytes); }
    else if (defer && win) run_lanes<false, false, true, true>(a, lds, lds_bytes);
    else if (defer) run_lanes<false, false, false, true>(a, lds, lds_bytes);
    else if (win) run_lanes<false, false, true, false>(a, lds, lds_bytes);
    else run_lanes<false, false, false, false>(a, lds, lds_bytes);

    memcpy(iter_ms, a.iter_ms, (size_t)P * 8);
    memcpy(peak_mb, a.peak_mb, (size_t)P * 8);
    memcpy(feasible, a.feasible, (size_t)P);
    if (status) memcpy(status, a.status, (size_t)P);
    if (stage_out) memcpy(stage_out, a.stage_out, rec_bytes);
    return 0;
}
}  // namespace

// ------------------------------------------------------------------------------------------
// The plan-editing kernels (ace_edit_kernels.h) on the CPU, one call per work item, arrays behind
// guard pages as above.  Sizes follow the C ABI's documentation of ace_apply_moves /
// ace_recompute_groups / ace_recompute_select.
// ------------------------------------------------------------------------------------------
extern "C" int ace_emu_apply_moves(const uint8_t *tmpl_codes, const uint32_t *tmpl_hdr, int n_templates, const uint32_t *moves,
                                   long long n, int num_ops, int n_algo, uint8_t *codes_out, uint32_t *hdr_out,
                                   unsigned long long *keys_out) {
    GuardedPool pool;
    const int G = (num_ops + 15) / 16;
    const size_t cb = (size_t)G * 16;
    const ace_u4 *tc = (const ace_u4 *)pool.place(tmpl_codes, (size_t)n_templates * cb);
    const ace_u4 *th = (const ace_u4 *)pool.place(tmpl_hdr, (size_t)n_templates * 16);
    const ace_u4 *mv = (const ace_u4 *)pool.place(moves, (size_t)n * 16);
    ace_u4 *co = (ace_u4 *)pool.place(nullptr, (size_t)n * cb);
    ace_u4 *ho = (ace_u4 *)pool.place(nullptr, (size_t)n * 16);
    unsigned long long *ko = keys_out ? (unsigned long long *)pool.place(keys_out, (size_t)n * 16, 8) : nullptr;
    // (the library launches whole workgroups of 256: ids past n * G must fall out at the first test)
    const unsigned long long total = ((unsigned long long)n * G + 255) / 256 * 256;
    for (unsigned long long id = 0; id < total; ++id)
        apply_moves_body(id, tc, th, n_templates, mv, (unsigned long long)n, G, n_algo == 2 ? 1 : 0, co, ho, ko);
    memcpy(codes_out, co, (size_t)n * cb);
    memcpy(hdr_out, ho, (size_t)n * 16);
    if (keys_out) memcpy(keys_out, ko, (size_t)n * 16);
    return 0;
}

namespace {
struct RcHost {
    GuardedPool pool;
    RcTables k;
    uint8_t *codes;
    size_t code_bytes;
    const int32_t *plan, *lo, *hi, *nsb;
    const uint32_t *mrow;
    RcHost(const ace_rc_tables_t *t, int n, const int32_t *q_plan, const int32_t *q_lo, const int32_t *q_hi, const int32_t *q_nsb,
           const uint32_t *q_mrow) {
        code_bytes = (size_t)((t->num_ops + 15) / 16) * t->n_plans * 16;
        codes = (uint8_t *)pool.place(t->d_codes, code_bytes);
        k = RcTables{codes, (unsigned long long)t->n_plans,
                     (const int32_t *)pool.place(t->d_type_of_pos, (size_t)t->num_ops * 4, 4),
                     (const double *)pool.place(t->d_activations, (size_t)t->num_types * t->n_mbs * t->n_tp * t->n_algo * 8, 8),
                     (const uint8_t *)pool.place(t->d_no_recompute, (size_t)t->num_types, 1),
                     t->num_ops, t->num_types, t->n_mbs, t->n_tp, t->n_algo, t->n_algo == 2 ? 1 : 0};
        plan = (const int32_t *)pool.place(q_plan, (size_t)n * 4, 4);
        lo = (const int32_t *)pool.place(q_lo, (size_t)n * 4, 4);
        hi = (const int32_t *)pool.place(q_hi, (size_t)n * 4, 4);
        nsb = (const int32_t *)pool.place(q_nsb, (size_t)n * 4, 4);
        mrow = (const uint32_t *)pool.place(q_mrow, (size_t)n * 4, 4);
    }
};
}  // namespace

// (same parameter lists as ace_recompute_groups / ace_recompute_select, so a test double can stand in for the library)
extern "C" int ace_emu_rc_groups(const ace_rc_tables_t *t, int n, const int32_t *q_plan, const int32_t *q_lo, const int32_t *q_hi,
                                 const int32_t *q_nsb, const uint32_t *q_mrow, double *sum_size, int32_t *first_pos, int32_t *bad,
                                 void * /*stream*/) {
    RcHost h(t, n, q_plan, q_lo, q_hi, q_nsb, q_mrow);
    const size_t nt = (size_t)n * t->num_types;
    double *sum = (double *)h.pool.place(sum_size, nt * 8, 8);
    int32_t *first = (int32_t *)h.pool.place(first_pos, nt * 4, 4);
    int32_t *b = (int32_t *)h.pool.place(bad, (size_t)n * 4, 4);
    for (int a = 0; a < (n + 127) / 128 * 128; ++a)
        rc_groups_body(a, h.k, n, h.plan, h.lo, h.hi, h.nsb, h.mrow, sum, first, b);
    memcpy(sum_size, sum, nt * 8);
    memcpy(first_pos, first, nt * 4);
    memcpy(bad, b, (size_t)n * 4);
    return 0;
}

// (codes_rw must be t->d_codes, the usual call: the batch is edited in place)
extern "C" int ace_emu_rc_select(const ace_rc_tables_t *t, uint8_t *codes_rw, int n, const int32_t *q_plan, const int32_t *q_lo,
                                 const int32_t *q_hi, const int32_t *q_nsb, const uint32_t *q_mrow, const double *sum_size,
                                 const int32_t *first_pos, uint8_t *recomputed, const double *mem, double memory_limit,
                                 uint8_t *alive, void * /*stream*/) {
    if (codes_rw != t->d_codes) return -1;
    RcHost h(t, n, q_plan, q_lo, q_hi, q_nsb, q_mrow);
    const size_t nt = (size_t)n * t->num_types;
    const double *sum = (const double *)h.pool.place(sum_size, nt * 8, 8);
    const int32_t *first = (const int32_t *)h.pool.place(first_pos, nt * 4, 4);
    uint8_t *done = (uint8_t *)h.pool.place(recomputed, nt, 1);
    const double *m = (const double *)h.pool.place(mem, (size_t)n * 8, 8);
    uint8_t *al = (uint8_t *)h.pool.place(alive, (size_t)n, 1);
    for (int a = 0; a < (n + 127) / 128 * 128; ++a)
        rc_select_body(a, h.k, h.codes, n, h.plan, h.lo, h.hi, h.nsb, h.mrow, sum, first, done, m, memory_limit, al);
    memcpy(codes_rw, h.codes, h.code_bytes);
    memcpy(recomputed, done, nt);
    memcpy(alive, al, (size_t)n);
    return 0;
}

extern "C" int ace_emu_group_keys(const uint8_t *codes /* [G][P][16] */, const uint32_t *hdr, long long n, int num_ops,
                                  unsigned long long *keys) {
    GuardedPool pool;
    const int G = (num_ops + 15) / 16;
    const ace_u4 *c = (const ace_u4 *)pool.place(codes, (size_t)G * n * 16);
    const ace_u4 *h = (const ace_u4 *)pool.place(hdr, (size_t)n * 16);
    unsigned long long *k = (unsigned long long *)pool.place(nullptr, (size_t)n * 8, 8);
    for (unsigned long long p = 0; p < ((unsigned long long)n + 255) / 256 * 256; ++p)
        group_keys_body(p, c, h, (unsigned long long)n, G, num_ops, k);
    memcpy(keys, k, (size_t)n * 8);
    return 0;
}

extern "C" int ace_emu_gather_plans(const uint8_t *codes_in, const uint32_t *hdr_in, const uint32_t *perm, long long n, int num_ops,
                                    uint8_t *codes_out, uint32_t *hdr_out) {
    GuardedPool pool;
    const int G = (num_ops + 15) / 16;
    const ace_u4 *ci = (const ace_u4 *)pool.place(codes_in, (size_t)G * n * 16);
    const ace_u4 *hi = (const ace_u4 *)pool.place(hdr_in, (size_t)n * 16);
    const uint32_t *pm = (const uint32_t *)pool.place(perm, (size_t)n * 4, 4);
    ace_u4 *co = (ace_u4 *)pool.place(nullptr, (size_t)G * n * 16);
    ace_u4 *ho = (ace_u4 *)pool.place(nullptr, (size_t)n * 16);
    const unsigned long long total = ((unsigned long long)n * G + 255) / 256 * 256;
    for (unsigned long long id = 0; id < total; ++id) gather_plans_body(id, ci, hi, pm, (unsigned long long)n, G, co, ho);
    memcpy(codes_out, co, (size_t)G * n * 16);
    memcpy(hdr_out, ho, (size_t)n * 16);
    return 0;
}

// ace_pack_plans (with the check) / ace_unpack_plans; returns the findings.
extern "C" int ace_emu_pack(const uint8_t *rows, const uint32_t *hdr, long long P, int N, int n_mbs, int C, uint8_t *codes_out) {
    GuardedPool pool;
    const int G = (N + 15) / 16;
    int32_t flags = 0;
    PackShared *s = (PackShared *)pool.place(nullptr, sizeof(PackShared));
    PackArgs a{(const uint8_t *)pool.place(rows, (size_t)P * N), nullptr, nullptr, (ace_u4 *)pool.place(nullptr, (size_t)G * P * 16),
               (const ace_u4 *)pool.place(hdr, (size_t)P * 16), &flags, P, N, G, n_mbs, C};
    for (long long b = 0; b < (P + kPackPlans - 1) / kPackPlans; ++b) {
        memset((void *)s, 0xff, sizeof(*s));
        ace_pack_body(a, *s, 0, b);
    }
    memcpy(codes_out, a.codes_out, (size_t)G * P * 16);
    return flags;
}
extern "C" int ace_emu_unpack(const uint8_t *codes, long long P, int N, uint8_t *rows_out) {
    GuardedPool pool;
    const int G = (N + 15) / 16;
    PackShared *s = (PackShared *)pool.place(nullptr, sizeof(PackShared));
    PackArgs a{nullptr, (uint8_t *)pool.place(nullptr, (size_t)P * N), (const ace_u4 *)pool.place(codes, (size_t)G * P * 16), nullptr, nullptr, nullptr,
               P, N, G, 0, 8};
    for (long long b = 0; b < (P + kPackPlans - 1) / kPackPlans; ++b) {
        memset((void *)s, 0xff, sizeof(*s));
        ace_unpack_body(a, *s, 0, b);
    }
    memcpy(rows_out, a.rows_out, (size_t)P * N);
    return 0;
}

// The parts of a grid (ace_grid.h): up to `room` pairs (first workgroup, workgroups) in `out`; returns their number.
extern "C" int ace_emu_grid_parts(unsigned long long groups, unsigned lanes, unsigned long long *out, int room) {
    int n = 0;
    ace_grid_parts(groups, lanes, [&](uint64_t first, uint32_t count) {
        if (n < room) { out[2 * n] = first; out[2 * n + 1] = count; }
        ++n;
    });
    return n;
}
