"""Writes ace_duo_loop_asm.inc: the op loop of the scoring kernel for mid-sized batches (ace_duo.h) as gfx950 assembly.

    python3 superscaler_amd/csrc/gen_duo_loop_asm.py

Same operations per plan, in the same order, as the loop of gen_score_loop_asm.py, split over two lanes of different
wavefronts:
  time     forward, backward, recompute and resharding sums; parks 32 bytes of a stage's record
  memory   weights, activations, saved activations, running segment and peak, reserved maxima; parks the other 48
and, along the sequence, over the wavefronts of several parts: a part's lane walks from the part's first group on, parks
the stages that start in the part, and stops behind the last of them (at or behind `cut`, the next part's first position).
What it adds up before the first stage that starts there belongs to the part before it and is not parked.

Written for one to four wavefronts per SIMD, where what counts is how long a wavefront takes per op (4 cycles per
instruction at best; measured besides: a taken branch 22, a scalar instruction on a vector compare's result right
behind it 16 more):
  * it never waits for what it has just asked for: at op k the collective ids of op k + 4 and the table entries of
    op k + 2 are asked for (rings of four register sets; LDS returns in order, so the waits are counts), the code words
    of group g + 2 while group g is walked, and a stage's two table offsets a stage ahead;
  * the per-position scalars come from the lanes of a vector register (sixteen ops x four words, one load per group,
    v_readlane) instead of scalar loads, which share the LDS counter and would drain the reads in flight every four ops;
  * the compares run ahead of their use, and ops at which no lane starts a stage are walked without a taken branch: the
    steps that start or end one lie behind the loop.
The loop ends with the plan's last op, behind which a stage start is planted, if not with its part.

One text per (time: resharding on / off; memory: reserved-memory rule).  v28-v127 and s24-s99 belong to the loop.
"""
import os

HERE = os.path.dirname(os.path.abspath(__file__))

GLOGS, GLOGS_LO, LUT2, WSOFF = "v[28:29]", "v28", "v30", "v31"
# time
FB, RCS, RSF, RSB, FWD, BWD = "v[32:33]", "v[34:35]", "v[36:37]", "v[38:39]", "v[40:41]", "v[42:43]"
# memory
W_, A_, SAVED, PEAK, RES, CNOUT, META = "v[32:33]", "v[34:35]", "v[36:37]", "v[38:39]", "v[40:41]", "v42", "v43"
RUN, RFM, RBM = "v[44:45]", "v[46:47]", "v[48:49]"


def pair(b):
    return f"v[{b}:{b + 1}]"


def quad(b):
    return f"v[{b}:{b + 3}]"


def T0(x):
    return f"v{88 + x}"


def R(x):
    return f"v{92 + x}"


WORD = [f"v{96 + j}" for j in range(4)]
NEXT = [f"v{100 + j}" for j in range(4)]
FAR = [f"v{104 + j}" for j in range(4)]


def D(y):
    b = 108 + 3 * y
    return dict(w8=f"v{b}", cn=f"v{b + 1}", r8=f"v{b + 2}")


POSV, POSN, POSF, ZEROPV = "v114", "v115", "v116", "v117"
WSNEXT = "v50"                               # where the lane's record after the current one goes (WSOFF: the current one's; BIG: nowhere)
ZVRK, ZV, RK, NZVRK = "v[118:119]", "v118", "v119", "v[120:121]"
T1, T2, T3, LANE4, T01 = "v122", "v123", "v124", "v125", "v[126:127]"

CPTR, CPTR_LO, CPTR_HI = "s[26:27]", "s26", "s27"
PPTR, PPTR_LO, PPTR_HI = "s[36:37]", "s36", "s37"


def SM(x):                                   # "op starts a stage", ring of eight ops
    b = (40, 42, 44, 46, 92, 94, 96, 98)[x & 7]
    return f"s[{b}:{b + 1}]"


MRC = ["s[48:49]", "s[50:51]"]
CUTA, CUTB = "s34", "s35"
M_E, M_P, M_KP, NKEEP, ORD, PREVORD = "s[24:25]", "s[52:53]", "s[54:55]", "s[56:57]", "s[58:59]", "s60"
SHOT, SZ, SPK, ZDELTA = "s61", "s62", "s63", "s64"
GRP, NGRP, POSBASE, LEFT, K07, K08, K1F, VMN, WSLIMIT = "s66", "s67", "s68", "s69", "s70", "s71", "s72", "s73", "s74"
S0, S1, S2, S23, MASK, PLANT = "s76", "s77", "s78", "s[78:79]", "s80", "s81"


def PIECE(i):                                # where piece i of the workgroup's records begins (the five 16-byte pieces of a record lie L lanes apart)
    return f"s[{82 + 2 * i}:{83 + 2 * i}]"


class Duo:
    def __init__(self, time, rsh=False, mode="max"):
        self.time, self.rsh, self.mode, self.lines = time, time and rsh, mode, []
        self.per_step = (4 if self.rsh else 1) if time else 2      # LDS reads of a step (beside a stage's offsets)

    def o(self, s):
        self.lines.append(s)

    def c(self, s):
        self.lines.append("; " + s)

    def prep(self, y, wa, wb):
        d = D(y)
        self.o(f"v_and_b32 {d['w8']}, {K07}, {wa}")
        self.o(f"v_lshlrev_b32 {d['w8']}, 3, {d['w8']}")
        if self.rsh or not self.time:
            self.o(f"v_alignbit_b32 {T1}, {wb}, {wa}, 8")
            self.o(f"v_and_or_b32 {d['cn']}, {T1}, {K07}, {d['w8']}")
        self.o(f"v_and_b32 {d['r8']}, {K08}, {wa}")

    def stage_fetch(self, dst):
        self.o(f"v_and_b32 {T1}, 15, {GLOGS_LO}")
        self.o(f"v_lshl_add_u32 {T1}, {T1}, 3, {LUT2}")
        self.o(f"v_lshrrev_b64 {GLOGS}, 4, {GLOGS}")
        self.o(f"ds_read_b64 {dst}, {T1}")

    def scalars(self, k):
        """Row address of op k + 2, pair table of ops k + 3 and k + 4 (k: -4 .. 15)."""
        if self.rsh and k + 3 >= 0:
            i = k + 3
            self.o(f"v_readlane_b32 {SPK}, {POSV if i < 16 else POSN}, {4 * (i & 15) + 2}")
        if k + 2 >= 0:
            i = k + 2
            self.o(f"v_readlane_b32 {SHOT}, {POSV if i < 16 else POSN}, {4 * (i & 15)}")

    def compare_stage(self, j):
        """Which lanes' op j starts a stage (j: 1 .. 20)."""
        w = j >> 2
        word = WORD[w] if w < 4 else NEXT[w - 4]
        self.o(f"v_cmp_gt_u32_sdwa {SM(j)}, {word}, 15 src0_sel:BYTE_{j & 3} src1_sel:DWORD")

    def ahead_a(self, k, event, L):
        """Op k + 4: its entry index; its collective ids.  `event`: some lane's op may start a stage."""
        j, b = k + 4, k & 3
        w = j >> 2
        d, before = D(w & 1), D((w + 1) & 1)
        self.c(f"op {j}: entry index, collective ids")
        if event:
            self.o(f"s_cmp_lg_u64 {SM(j)}, 0")
            self.o(f"s_cbranch_scc0 L_as_{L}")
            self.o(f"s_mov_b64 exec, {SM(j)}")
            self.o(f"s_waitcnt lgkmcnt({self.per_step})")
            self.o(f"v_mov_b64 {ZVRK}, {NZVRK}")
            self.stage_fetch(NZVRK)
            self.o("s_mov_b64 exec, -1")
            self.o(f"L_as_{L}:")
        sel = "dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_"
        self.o(f"v_add_u32_sdwa {T0(j & 3)}, {ZV}, {d['w8']} {sel}{b}")
        if not self.rsh:
            return
        if j > 0:
            self.o(f"v_add_u32_sdwa {T1}, {RK}, {(d if b else before)['cn']} {sel}{b - 1 if b else 3}")
            self.o(f"v_lshl_add_u32 {T1}, {T1}, 2, {SPK}")
            if event:
                self.o(f"v_cndmask_b32_e64 {T1}, {T1}, {ZEROPV}, {SM(j)}")
        else:
            self.o(f"v_mov_b32 {T1}, {ZEROPV}")
        self.o(f"ds_read_b32 {R(j & 3)}, {T1}")

    def ahead_b(self, k, drain=False):
        """Op k + 2: its table entries."""
        x = (k + 2) & 3
        self.c(f"op {k + 2}: table entries")
        self.o(f"v_mad_u32_u24 {T2}, {T0(x)}, 6, {SHOT}")
        if not self.time:
            self.o(f"ds_read_b128 {quad(56 + 8 * x)}, {T2} offset:16")
            self.o(f"ds_read_b128 {quad(60 + 8 * x)}, {T2} offset:32")
            return
        self.o(f"ds_read_b128 {quad(56 + 4 * x)}, {T2}")
        if not self.rsh:
            return
        self.o(f"s_add_u32 {SZ}, {SHOT}, {ZDELTA}")
        self.o(f"v_add_u32_e32 {T3}, {SZ}, {T0(x)}")
        self.o(f"s_waitcnt lgkmcnt({0 if drain else 9})")          # its ids, asked for two steps ago
        wsel = "dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_"
        self.o(f"v_add_u32_sdwa {T1}, {T3}, {R(x)} {wsel}0")
        self.o(f"v_add_u32_sdwa {T2}, {T3}, {R(x)} {wsel}1")
        self.o(f"ds_read_b64 {pair(72 + 4 * x)}, {T1}")
        self.o(f"ds_read_b64 {pair(74 + 4 * x)}, {T2}")

    def reserved(self):
        if self.mode == "max":          # max(rf + rb, W)
            self.o(f"v_add_f64 {RES}, {RFM}, {RBM}")
            self.o(f"v_max_f64 {RES}, {RES}, {W_}")
        elif self.mode == "min":        # max(max(rf, rb), max(W, 0))
            self.o(f"v_max_f64 {RES}, {RFM}, {RBM}")
            self.o(f"v_max_f64 {T01}, {W_}, 0")
            self.o(f"v_max_f64 {RES}, {RES}, {T01}")
        else:
            self.o(f"v_mov_b64 {RES}, 0")

    def park(self, k, sm, stores):
        """The stage's record (lanes with a place for one), the next one's place: none if the next op is the next part's."""
        self.o(f"v_cmp_gt_u32_e32 vcc, {WSLIMIT}, {WSOFF}")
        self.o("s_and_b64 exec, exec, vcc")
        self.o(f"s_cselect_b32 {S0}, {len(stores)}, 0")             # (no such lane: the stores may not be issued at all)
        self.o(f"s_add_u32 {VMN}, {VMN}, {S0}")
        for src, piece in stores:
            self.o(f"global_store_dwordx4 {WSOFF}, {src}, {PIECE(piece)}")
        self.o(f"s_mov_b64 exec, {sm}")
        self.o(f"v_max_u32_e32 {WSOFF}, {CUTA if k < 15 else CUTB}, {WSNEXT}")
        self.o(f"v_add_u32_e32 {WSNEXT}, %[wsstride], {WSNEXT}")

    def plan_end(self, k):
        self.o(f"s_add_u32 {S0}, {POSBASE}, {k + 1}")
        self.o(f"s_cmp_eq_u32 {S0}, %[n_ops]")
        self.o("s_cbranch_scc1 L_exit_%=")

    def step(self, k, event):
        """One op.  `event`: op k + 1 or op k + 4 starts a stage in some lane; these steps lie behind the loop, so that the
        others are walked without a taken branch."""
        L = f"{k}_%="
        b, x, k1 = k & 3, k & 3, k + 1
        d, d1 = D((k >> 2) & 1), D((k1 >> 2) & 1)
        sm = SM(k1)
        if event:
            self.o(f"L_ev_{L}:")
        else:
            self.c(f"================ op {k} of the group")
            self.o(f"L_op_{L}:")
            self.o(f"s_or_b64 {M_E}, {SM(k + 4)}, {sm}")
            self.o(f"s_cbranch_scc1 L_ev_{L}")
        self.scalars(k)
        self.compare_stage(k + 5)
        if self.time:
            self.o(f"v_cmp_ne_u32_sdwa {MRC[0]}, {d['r8']}, 0 src0_sel:BYTE_{b} src1_sel:DWORD")
        else:
            self.o(f"v_cmp_ne_u32_sdwa {MRC[k1 & 1]}, {d1['r8']}, 0 src0_sel:BYTE_{k1 & 3} src1_sel:DWORD")
        self.ahead_a(k, event, L)
        self.ahead_b(k)
        self.o(f"s_waitcnt lgkmcnt({2 * self.per_step})")           # the entries of op k, asked for two steps ago
        self.c(f"op {k}: sums")
        if self.time:
            e, z = 56 + 4 * x, 72 + 4 * x
            self.o(f"v_add_f64 {FWD}, {FWD}, {pair(e)}")
            self.o(f"v_add_f64 {BWD}, {BWD}, {pair(e + 2)}")
            if self.rsh:
                self.o(f"v_add_f64 {RSF}, {RSF}, {pair(z)}")
                self.o(f"v_add_f64 {RSB}, {RSB}, {pair(z + 2)}")
            self.o(f"s_mov_b64 exec, {MRC[0]}")
            self.o(f"v_add_f64 {RCS}, {RCS}, {pair(e)}")
            if event:
                self.o(f"s_cmp_lg_u64 {sm}, 0")
                self.o(f"s_cbranch_scc0 L_ne_{L}")
                self.o(f"s_mov_b64 exec, {sm}")
                self.o(f"v_add_f64 {FB}, {FWD}, {BWD}")
                self.park(k, sm, [("v[32:35]", 0), ("v[36:39]", 1)])
                for r in (FWD, BWD):
                    self.o(f"v_mov_b64 {r}, 0")
                self.o("s_nop 1")
                for r in (RCS,) + ((RSF, RSB) if self.rsh else ()):
                    self.o(f"v_mov_b64 {r}, 0")
                self.plan_end(k)
                self.o(f"L_ne_{L}:")
            self.o("s_mov_b64 exec, -1")
        else:
            e = 56 + 8 * x
            act = pair(e + 2)
            self.o(f"v_add_f64 {W_}, {W_}, {pair(e)}")
            self.o(f"v_add_f64 {A_}, {A_}, {act}")
            self.o(f"s_and_b64 {M_P}, {MRC[0]}, {MRC[1]}")
            if event:
                self.o(f"s_andn2_b64 {M_P}, {M_P}, {sm}")
                self.o(f"s_cmp_lg_u64 {sm}, 0")
                self.o(f"s_cbranch_scc0 L_ne_{L}")
                self.c("lanes whose stage ends with this op (the reserved maxima do not take it)")
                if k:
                    self.o(f"s_bitcmp1_b64 {ORD}, {4 * k - 1}")
                else:
                    self.o(f"s_bitcmp1_b32 {PREVORD}, 0")
                self.o(f"s_cselect_b64 exec, {sm}, 0")
                self.o(f"v_max_f64 {PEAK}, {PEAK}, {RUN}")
                self.o(f"s_mov_b64 exec, {sm}")
                self.reserved()
                self.o(f"v_readlane_b32 {S1}, {POSV}, {4 * k + 3}")
                self.o(f"v_mov_b32 {CNOUT}, {d['cn']}")
                self.o(f"s_add_u32 {S0}, {POSBASE}, {k}")
                self.o(f"s_andn2_b32 {S1}, {S1}, 0xff")
                self.o(f"s_lshl_b32 {S1}, {S1}, 8")
                self.o(f"s_or_b32 {S0}, {S0}, {S1}")
                self.o(f"v_mov_b32 {META}, {S0}")
                self.park(k, sm, [("v[32:35]", 2), ("v[36:39]", 3), ("v[40:43]", 4)])
                for r in (RUN, RFM, RBM):
                    self.o(f"v_mov_b64 {r}, 0")
                self.o("s_nop 1")
                for r in (W_, A_, SAVED, PEAK):
                    self.o(f"v_mov_b64 {r}, 0")
                self.plan_end(k)
                self.o(f"s_andn2_b64 exec, -1, {sm}")               # (the next stage's maxima start behind this op)
                self.o(f"L_ne_{L}:")
            self.o(f"v_max_f64 {RFM}, {RFM}, {pair(e + 4)}")
            self.o(f"v_max_f64 {RBM}, {RBM}, {pair(e + 6)}")
            self.c("recompute pair (this op, next op): saved activations, running segment, peak")
            self.o(f"s_bitcmp1_b64 {NKEEP}, {4 * k + 3}")
            self.o(f"s_cselect_b64 {M_KP}, {M_P}, 0")
            self.o(f"s_mov_b64 exec, {M_P}")
            self.o(f"v_add_f64 {RUN}, {RUN}, {act}")
            self.o(f"s_mov_b64 exec, {M_KP}")
            self.o(f"v_add_f64 {SAVED}, {SAVED}, {act}")
            self.o(f"s_andn2_b64 exec, -1, {M_KP}")
            self.o(f"v_max_f64 {PEAK}, {PEAK}, {RUN}")
            self.o(f"v_mov_b64 {RUN}, 0")
            self.o("s_mov_b64 exec, -1")
        if b == 3:
            n = (k >> 2) + 2
            self.c("the word two ahead")
            self.prep(n & 1, WORD[n] if n < 4 else NEXT[n - 4], WORD[n + 1] if n + 1 < 4 else NEXT[n - 3])
        if event:
            self.o(f"s_branch L_op_{k1}_%=")

    def apply_masks(self, regs, tag):
        """LEFT = N - (first position of the group): code bytes past the last op read as zero, the byte right behind it
        gets a stage start; five code bits used."""
        self.o(f"s_cmp_ge_i32 {LEFT}, 16")
        self.o(f"s_cbranch_scc1 L_full_{tag}_%=")
        for j in range(4):
            self.o(f"s_sub_i32 {S0}, {LEFT}, {4 * j}")
            self.o(f"s_min_i32 {S1}, {S0}, 4")
            self.o(f"s_max_i32 {S1}, {S1}, 0")
            self.o(f"s_lshl_b32 {S1}, {S1}, 3")
            self.o(f"s_bfm_b64 {S23}, {S1}, 0")
            self.o(f"s_and_b32 {MASK}, {S2}, {K1F}")
            self.o(f"s_lshl_b64 {S23}, 16, {S1}")
            self.o(f"s_cmp_ge_i32 {S0}, 0")
            self.o(f"s_cselect_b32 {PLANT}, {S2}, 0")
            self.o(f"v_and_b32 {regs[j]}, {MASK}, {regs[j]}")
            self.o(f"v_or_b32 {regs[j]}, {PLANT}, {regs[j]}")
        self.o(f"s_branch L_masked_{tag}_%=")
        self.o(f"L_full_{tag}_%=:")
        for j in range(4):
            self.o(f"v_and_b32 {regs[j]}, {K1F}, {regs[j]}")
        self.o(f"L_masked_{tag}_%=:")

    def load_group(self, regs, skip):
        """Code words of the next group not loaded yet (CPTR), zeros behind the last one (SCC: there is one)."""
        self.o(f"s_cbranch_scc0 L_nl_{skip}_%=")
        self.o(f"global_load_dwordx4 v[{regs[0][1:]}:{regs[3][1:]}], %[codeoff], {CPTR}")
        self.o(f"s_branch L_ld_{skip}_%=")
        self.o(f"L_nl_{skip}_%=:")
        for r in regs:
            self.o(f"v_mov_b32 {r}, 0")
        self.o(f"L_ld_{skip}_%=:")

    def next_code(self):
        self.o(f"s_add_u32 {CPTR_LO}, {CPTR_LO}, %[gstride_lo]")
        self.o(f"s_addc_u32 {CPTR_HI}, {CPTR_HI}, %[gstride_hi]")

    def next_pos(self):
        self.o(f"s_add_u32 {PPTR_LO}, {PPTR_LO}, 256")
        self.o(f"s_addc_u32 {PPTR_HI}, {PPTR_HI}, 0")

    def group_flags(self):
        if self.time:
            return
        self.o(f"v_and_b32 {T1}, 1, {POSV}")
        self.o(f"v_and_b32 {T2}, 2, {POSV}")
        self.o(f"v_cmp_ne_u32_e64 {NKEEP}, {T1}, 0")
        self.o(f"v_cmp_ne_u32_e64 {ORD}, {T2}, 0")

    def build(self):
        o, c = self.o, self.c
        c("---- set-up")
        o(f"s_add_u32 {NGRP}, %[n_ops], 15")
        o(f"s_lshr_b32 {NGRP}, {NGRP}, 4")
        o(f"v_mov_b64 {GLOGS}, %[glogs]")
        o(f"v_mov_b32 {LUT2}, %[lut2]")
        o(f"s_mov_b64 {CPTR}, %[codes]")
        o(f"s_mov_b64 {PPTR}, %[pos]")
        o(f"s_mov_b32 {K07}, 0x07070707")
        o(f"s_mov_b32 {K08}, 0x08080808")
        o(f"s_mov_b32 {K1F}, 0x1f1f1f1f")
        o(f"s_mov_b32 {GRP}, %[grp]")
        o(f"s_lshl_b32 {POSBASE}, {GRP}, 4")
        o(f"s_mov_b32 {PREVORD}, 0")
        o(f"v_mbcnt_lo_u32_b32 {LANE4}, -1, 0")
        o(f"v_mbcnt_hi_u32_b32 {LANE4}, -1, {LANE4}")
        o(f"v_lshlrev_b32 {LANE4}, 2, {LANE4}")
        o(f"global_load_dwordx4 v[{WORD[0][1:]}:{WORD[3][1:]}], %[codeoff], {CPTR}")
        self.next_code()
        o(f"s_add_u32 {S0}, {GRP}, 1")
        o(f"s_cmp_lt_u32 {S0}, {NGRP}")
        self.load_group(NEXT, "n0")
        c("(one group of position entries follows the last group's)")
        o(f"global_load_dword {POSV}, {LANE4}, {PPTR}")
        self.next_pos()
        o(f"global_load_dword {POSN}, {LANE4}, {PPTR}")
        o(f"v_mov_b32 {POSF}, 0")
        for r in ((FWD, BWD, FB, RCS, RSF, RSB) if self.time else (W_, A_, SAVED, PEAK, RUN, RFM, RBM)):
            o(f"v_mov_b64 {r}, 0")
        o(f"v_mov_b32 {WSOFF}, %[recoff]")
        o(f"v_mov_b32 {WSNEXT}, %[recnext]")
        o(f"s_lshl_b32 {WSLIMIT}, %[wsstride], 4")
        o(f"s_mov_b64 {PIECE(0)}, %[recbase]")
        for i in range(1, 5):
            o(f"s_add_u32 s{82 + 2 * i}, s{80 + 2 * i}, %[wspiece]")
            o(f"s_addc_u32 s{83 + 2 * i}, s{81 + 2 * i}, 0")
        if self.rsh:
            o(f"v_mov_b32 {ZEROPV}, %[zerop]")
        self.stage_fetch(ZVRK)
        self.stage_fetch(NZVRK)
        o("s_waitcnt vmcnt(0) lgkmcnt(0)")
        o(f"s_sub_i32 {LEFT}, %[n_ops], {POSBASE}")
        self.apply_masks(WORD, "w0")
        o(f"s_sub_i32 {LEFT}, {LEFT}, 16")
        self.apply_masks(NEXT, "w1")
        self.prep(0, WORD[0], WORD[1])
        self.group_flags()
        if self.rsh:
            o(f"v_readlane_b32 {SHOT}, {POSV}, 0")
            o(f"v_readlane_b32 {SZ}, {POSV}, 1")
            o("s_nop 4")
            o(f"s_sub_u32 {ZDELTA}, {SZ}, {SHOT}")
        for j in range(1, 5):
            self.compare_stage(j)
        for k in range(-4, 0):
            self.scalars(k)
            o("s_nop 1")
            self.ahead_a(k, k > -4, f"p{-k}_%=")
            o("s_waitcnt lgkmcnt(0)")
            if k + 2 >= 0:
                self.ahead_b(k, drain=True)
        if not self.time:
            o(f"v_cmp_ne_u32_sdwa {MRC[0]}, {D(0)['r8']}, 0 src0_sel:BYTE_0 src1_sel:DWORD")
        self.prep(1, WORD[1], WORD[2])
        o("s_waitcnt lgkmcnt(0)")
        c("---- one 16-op group per iteration")
        o("L_group_%=:")
        self.next_code()
        self.next_pos()
        o(f"s_add_u32 {S0}, {GRP}, 2")
        o(f"s_cmp_lt_u32 {S0}, {NGRP}")
        self.load_group(FAR, "f")
        o(f"s_cmp_le_u32 {S0}, {NGRP}")
        o("s_cbranch_scc0 L_np_%=")
        o(f"global_load_dword {POSF}, {LANE4}, {PPTR}")
        o("L_np_%=:")
        o(f"s_mov_b32 {VMN}, 0")
        c("(the stage that starts with an op at or behind the cut is the next part's)")
        o(f"s_cmp_ge_u32 {POSBASE}, %[cut]")
        o(f"s_cselect_b32 {CUTA}, 0x80000000, 0")
        o(f"s_add_u32 {S0}, {POSBASE}, 16")
        o(f"s_cmp_ge_u32 {S0}, %[cut]")
        o(f"s_cselect_b32 {CUTB}, 0x80000000, 0")
        for k in range(16):
            self.step(k, False)
        o("L_op_16_%=:")
        c("---- next group: what was asked for at this one's start is in (vector-memory instructions complete in order: the record")
        c("stores of the last few ops need not be waited for)")
        steps = (12, 8, 4, 2) if self.time else (12, 9, 6, 3)
        for n in steps:
            o(f"s_cmp_ge_u32 {VMN}, {n}")
            o(f"s_cbranch_scc1 L_vm{n}_%=")
        o("s_waitcnt vmcnt(0)")
        o("s_branch L_vmd_%=")
        for n in steps:
            o(f"L_vm{n}_%=:")
            o(f"s_waitcnt vmcnt({n})")
            if n != steps[-1]:
                o("s_branch L_vmd_%=")
        o("L_vmd_%=:")
        for j in range(4):
            o(f"v_mov_b32 {WORD[j]}, {NEXT[j]}")
        for j in range(4):
            o(f"v_mov_b32 {NEXT[j]}, {FAR[j]}")
        if not self.time:
            o(f"s_bitcmp1_b64 {ORD}, 63")
            o(f"s_cselect_b32 {PREVORD}, 1, 0")
        o(f"v_mov_b32 {POSV}, {POSN}")
        o(f"v_mov_b32 {POSN}, {POSF}")
        o(f"s_add_u32 {POSBASE}, {POSBASE}, 16")
        o(f"s_sub_i32 {LEFT}, %[n_ops], {POSBASE}")
        o(f"s_sub_i32 {LEFT}, {LEFT}, 16")
        self.apply_masks(NEXT, "nx")
        self.group_flags()
        o(f"s_add_u32 {GRP}, {GRP}, 1")
        c("behind the cut: done when every lane has closed the stage it was in")
        o(f"s_cmp_ge_u32 {POSBASE}, %[cut]")
        o("s_cbranch_scc0 L_more_%=")
        o(f"v_cmp_gt_u32_e32 vcc, {WSLIMIT}, {WSOFF}")
        o("s_andn2_b64 exec, -1, vcc")
        c("(the stage starts of the lanes that have are none of ours)")
        for r in WORD + NEXT:
            o(f"v_and_b32 {r}, 0x0f0f0f0f, {r}")
        o("s_mov_b64 exec, -1")
        o("s_cmp_lg_u64 vcc, 0")
        o("s_cbranch_scc0 L_exit_%=")
        o("L_more_%=:")
        o(f"s_cmp_lt_u32 {GRP}, {NGRP}")
        o("s_cbranch_scc1 L_group_%=")
        o("s_branch L_exit_%=")
        c("---- steps in which a stage starts")
        for k in range(16):
            self.step(k, True)
        o("L_exit_%=:")
        o("s_mov_b64 exec, -1")
        o("s_waitcnt vmcnt(0) lgkmcnt(0)")
        return self.lines


def c_string(lines):
    out = []
    for ln in lines:
        assert '"' not in ln and "\\" not in ln
        out.append('    "' + ln + '\\n"')
    return " \\\n".join(out)


def render():
    """The text of ace_duo_loop_asm.inc."""
    parts = ["// Generated by gen_duo_loop_asm.py -- do not edit.  gfx950 assembly of the op loop of ace_duo.h; see the generator.",
             "#pragma once", ""]
    texts = [("TIME_RSH1", Duo(True, True)), ("TIME_RSH0", Duo(True, False))] + [(f"MEMORY_{m.upper()}", Duo(False, mode=m)) for m in ("max", "min", "none")]
    for name, d in texts:
        parts += [f"#define ACE_DUO_ASM_{name} \\", c_string(d.build()), ""]
    clob = ", ".join(f'"v{i}"' for i in range(28, 128)) + ", " + ", ".join(f'"s{i}"' for i in range(24, 100) if i not in (32, 33))   # (s32 / s33 are the ABI's stack registers)
    parts += [f"#define ACE_DUO_ASM_CLOBBERS {clob}, \"vcc\", \"scc\", \"memory\"", ""]
    return "\n".join(parts)


def main():
    path = os.path.join(HERE, "ace_duo_loop_asm.inc")
    with open(path, "w") as f:
        f.write(render())
    print("wrote", path)


if __name__ == "__main__":
    main()
