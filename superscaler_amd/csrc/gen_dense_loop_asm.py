"""Writes ace_dense_loop_asm.inc: the op loop over the dense tables (ace_dense.h) as gfx950 assembly.

    python3 superscaler_amd/csrc/gen_dense_loop_asm.py

Same operations per plan, in the same order, as the loop of gen_score_loop_asm.py: a plan per lane, stage tails parked in
records and evaluated after the loop, recompute rules as execution masks, pacing by arrival counters.  What differs is what
an op costs beside the reference's own additions:
  * addresses: one v_dot4_u32_u8 each for the op's table entry and for its pair's cost.  The word a lane's codes are
    kept in holds three consecutive codes and a constant byte; its dot product with a scalar of the position (byte strides
    of the codes, and the place of the row in units of the constant byte) plus the lane's stage offset is the LDS address.
  * costs: the pair table names the 16 bytes {forward, backward} by their LDS address; equal pairs are stored once.
  * reserved memory: the largest of a finite set of values is the one of the largest rank; forward and backward ranks are
    16 bits each, one v_pk_max_u16 for both.
  * tables: 40 bytes per entry, a ds_read_b64 per value (neighbouring codes and stage sizes in different banks; the values' offsets
    are the same for all tables).
  * records: a stage that ends is parked in registers, and the parked records of all lanes are stored when one of them is
    about to park its second, some ten at a time, one behind the other in the wavefront's own part of the workspace; a
    record says whose it is.  (Stored at [stage][lane], the records were what the loop waited for: 1,048,576 plans of 16
    stages took 1,300 us with these stores and 600 without; lines of which a few bytes at a time are written leave the L2
    cache many times over.  One behind the other: 650.)
Measured with this loop's instructions on four wavefronts per SIMD: any of them about 4 cycles; ds_read_b64 at 8-byte stride
over 56 entries 4 cycles per wavefront and CU, ds_read_b128 at 48-byte stride 12, ds_read2st64_b64 24.

v_dot4's result may be read by another instruction only three issue slots later: every use keeps that distance.

Instructions of every kind count: with four wavefronts per SIMD a scalar instruction costs about a quarter of a vector one, and a
lone wavefront needs five to six cycles for either.  So a step has one wait (for all it asked for in the step before), one branch
(vcc says whether any lane's stage ends here), and its conditional additions run under masks that follow from one another.
Masks compared a step ahead, or the rule for layer starts as a branch, were 3 % slower; the table offsets of the next stage set in a
part of their own in front of the sums (so that the reads go out earlier) 1.5 %.

The "_WIN" texts are for rows that do not fit in LDS together: windows of rows in alternate halves of the rows' space.  At a window's
first position all wavefronts of the workgroup meet at a barrier, after which each issues its share of the LDS-direct loads of the
window AFTER the one being entered (fetch_event; the records come from ace_dense.h), which arrive while the workgroup walks a whole
window.  A lane's offsets are those of the half in use: they and the table they come from change sides with the window.

One text per (rows resident / windowed, resharding on / off).  Register use: v28-v127 and s24-s99 belong to the loop; operands live below.
"""
import os

HERE = os.path.dirname(os.path.abspath(__file__))

# ---- vector registers ---------------------------------------------------------------------------------------
RINGV = "v28"                                # records this wavefront has stored
M0707, M07, KV = "v29", "v30", "v31"         # masks of the two codes of a record; the constant byte(s)
# the parked record of a lane, as it is stored
PIECES = [f"v[{b}:{b + 3}]" for b in (32, 36, 40, 44, 48)]
P_FB, P_RCS, P_RSF, P_RSB, P_W, P_A, P_SAVED, P_PEAK = (f"v[{32 + 2 * i}:{33 + 2 * i}]" for i in range(8))
P_RANK, P_META, P_PREV = "v48", "v49", "v50"
PLACE = "v51"                                # stage * 128 + lane * 2 (it counts the stages)
# the running stage
RCS, RSF, RSB, W_, A_, SAVED, PEAK, FWD, BWD, RUN = (f"v[{52 + 2 * i}:{53 + 2 * i}]" for i in range(10))
RANK = "v72"


def E(x):                                   # entries of an op: fwd, bwd, weights, act, ranks
    b = 74 + 10 * x
    return [f"v[{b + 2 * i}:{b + 2 * i + 1}]" for i in range(5)]


def RANKS(x):
    return f"v{74 + 10 * x + 8}"


def ZQ(x):                                  # cost of an op's input: forward, backward
    b = 94 + 4 * x
    return f"v[{b}:{b + 3}]", f"v[{b}:{b + 1}]", f"v[{b + 2}:{b + 3}]"


def R(x):                                   # LDS address of an op pair's cost
    return f"v{102 + x}"


WORD = [f"v{104 + j}" for j in range(4)]    # code words of the current 16-op group
NEXT = [f"v{108 + j}" for j in range(4)]    # ... of the next group


def D(y):                                   # per 4-op word: codes 0 1 2 + constant, codes 2 3 4 + constant, recompute bits
    b = 112 + 3 * y
    return dict(a01=f"v{b}", a23=f"v{b + 1}", r8=f"v{b + 2}")


ZVRK, ZV, RK, NZVRK, NZV = "v[118:119]", "v118", "v119", "v[120:121]", "v120"
GLOGS, GLOGS_LO = "v[122:123]", "v122"       # log2 of the sizes of the plan's stages to come, 4 bits each, the next one at bit 3
LUT2, PACE = "v124", "v125"
T1, T2, T3 = "v126", "v127", "v73"

# ---- scalar registers ---------------------------------------------------------------------------------------
SRD = "s[24:27]"
CPTR, CPTR_LO, CPTR_HI = "s[28:29]", "s28", "s29"
PPTR, PPTR_LO, PPTR_HI = "s[36:37]", "s36", "s37"
GRP, LEFT, K1F, KC, K08, POSBASE = "s30", "s31", "s38", "s39", "s40", "s41"
MRC = ["s[42:43]", "s[58:59]"]
PEND = "s[46:47]"                            # lanes with a parked record that is not stored yet


LASTPLACE, ROOM = "s45", "s[48:49]"          # PLACE of a seventeenth stage; the lanes of a flush that may store
SOFF = ("0", "s53", "s57", "s60", "s61")     # where each piece of the wavefront's records begins

K78, VMN, NGRP, MASK, PLANT, PREVFL = "s44", "s50", "s51", "s52", "s56", "s62"
S0, S1, S2, S23 = "s96", "s97", "s98", "s[98:99]"
# windowed rows: the next window's first position, the next fetch event, "a window was entered since the next group's code words
# were asked for", how far the other half of the rows (of the offsets table) lies from the current one
NEXTWIN, EVT, ARRIVED, HALF, LUTHALF, DMAPTR, DMAOFF = "s34", "s35", "s55", "s54", "s57", "s[60:61]", "s63"


def P(y, q):                                # position entry: dot4 scalars of the op's row and of its pair, record word, flags
    b = 64 + 16 * y + 4 * q
    return dict(hot=f"s{b}", pk=f"s{b+1}", meta=f"s{b+2}", fl=f"s{b+3}")


def PBUF(y):
    return f"s[{64 + 16 * y}:{79 + 16 * y}]"


class Dense:
    def __init__(self, rsh, win=False):
        self.rsh, self.win, self.lines = rsh, win, []
        # (windowed rows: no scalar register is left to keep them in)
        self.soff = ("0", "s97", "s98", "s99", DMAOFF) if win else SOFF

    def o(self, s):
        self.lines.append(s)

    def c(self, s):
        self.lines.append("; " + s)

    def prep(self, y, wa, wb):
        d = D(y)
        self.c(f"word-level: codes with the constant byte, recompute bits (buffer {y})")
        self.o(f"v_alignbit_b32 {d['a23']}, {wb}, {wa}, 16")
        self.o(f"v_and_or_b32 {d['a01']}, {wa}, {KC}, {KV}")
        self.o(f"v_and_or_b32 {d['a23']}, {d['a23']}, {KC}, {KV}")
        self.o(f"v_and_b32 {d['r8']}, {K08}, {wa}")

    def code_word(self, k1):
        return D((k1 >> 2) & 1)["a01" if (k1 & 3) < 2 else "a23"]

    def stage_fetch(self):
        """Asks for the table offsets of the stage after the one that begins (the table is 128-byte aligned)."""
        self.o(f"v_bfi_b32 {T3}, {K78}, {GLOGS_LO}, {LUT2}")
        self.o(f"v_lshrrev_b64 {GLOGS}, 4, {GLOGS}")
        self.o(f"ds_read_b64 {NZVRK}, {T3}")

    def flush(self, lanes):
        """Stores the parked records of `lanes` behind those stored so far; lanes with sixteen stages store no more (and go on
        counting).  Leaves exec as `lanes`."""
        self.o(f"s_mov_b64 exec, {lanes}")
        self.o(f"v_cmp_gt_u32_e64 {ROOM}, {LASTPLACE}, {PLACE}")
        self.o(f"s_mov_b64 exec, {ROOM}")
        self.o(f"s_cmp_lg_u64 {ROOM}, 0")                      # (no such lane: the stores may not be issued at all)
        self.o(f"s_cselect_b32 {S0}, 5, 0")
        self.o(f"s_add_u32 {VMN}, {VMN}, {S0}")
        self.o(f"v_mbcnt_lo_u32_b32 {T1}, s48, {RINGV}")
        self.o(f"v_mbcnt_hi_u32_b32 {T1}, s49, {T1}")
        self.o(f"v_lshlrev_b32 {T1}, 4, {T1}")
        if self.win:
            for i in range(1, 5):
                self.o(f"s_mov_b32 {self.soff[i]}, {16384 * i}")
        for regs, off in zip(PIECES, self.soff):
            self.o(f"buffer_store_dwordx4 {regs}, {T1}, {SRD}, {off} offen")
        self.o(f"s_bcnt1_i32_b64 {S0}, {ROOM}")
        self.o("s_mov_b64 exec, -1")
        self.o(f"v_add_u32_e32 {RINGV}, {S0}, {RINGV}")
        self.o(f"s_mov_b64 exec, {lanes}")
        self.o(f"v_add_u32_e32 {PLACE}, 0x80, {PLACE}")

    def addresses(self, k1):
        p = P((k1 >> 2) & 1, k1 & 3)
        self.c(f"op {k1}: addresses of its entry and of its pair's cost address")
        self.o(f"v_dot4_u32_u8 {T1}, {self.code_word(k1)}, {p['hot']}, {ZV}")
        if self.rsh:
            self.o(f"v_dot4_u32_u8 {T2}, {self.code_word(k1)}, {p['pk']}, {RK}")

    def reads(self, k1):
        x1 = k1 & 1
        for i, e in enumerate(E(x1)):
            self.o(f"ds_read_b64 {e}, {T1}" + (f" offset:{8 * i}" if i else ""))
        if self.rsh:
            self.o(f"ds_read_u16 {R(1 - x1)}, {T2}")           # where the cost of the (k1, k1 + 1) pair is

    def fetch_event(self, L, pq):
        """Windowed rows, one fetch event: the wavefront's record {first position of the window after the one being entered,
        bit 0: wait for the fetch | number of loads << 8, address of the rows} and four loads {byte offset in the rows, LDS
        address} (through s[pq:pq+7]); all wavefronts of the workgroup meet, then each issues its loads (LDS-direct, 1 KB each)."""
        self.o(f"s_mul_i32 {DMAOFF}, {EVT}, %[eventsize]")
        self.o(f"s_add_u32 {DMAOFF}, {DMAOFF}, %[waveoff]")
        self.o(f"s_load_dwordx4 s[96:99], {DMAPTR}, {DMAOFF}")
        self.o(f"s_add_u32 {DMAOFF}, {DMAOFF}, 16")
        self.o(f"s_load_dwordx8 s[{pq}:{pq + 7}], {DMAPTR}, {DMAOFF}")
        self.o("s_waitcnt vmcnt(0) lgkmcnt(0)")             # this wavefront's reads of the old rows and its loads so far have landed
        self.o("s_barrier")
        self.o(f"s_mov_b32 {ARRIVED}, 1")                   # (so have the next group's code words, if they were asked for)
        self.o(f"s_add_u32 {EVT}, {EVT}, 1")
        self.o(f"v_mbcnt_lo_u32_b32 {T1}, -1, 0")
        self.o(f"v_mbcnt_hi_u32_b32 {T1}, -1, {T1}")
        self.o(f"v_lshlrev_b32 {T1}, 4, {T1}")
        self.o(f"s_bfe_u32 {DMAOFF}, s97, 0x40008")         # number of loads
        for j in range(4):
            self.o(f"s_cmp_le_u32 {DMAOFF}, {j}")
            self.o(f"s_cbranch_scc1 L_fd_{L}")
            self.o(f"s_mov_b32 m0, s{pq + 2 * j + 1}")
            self.o(f"v_add_u32_e32 {T2}, s{pq + 2 * j}, {T1}")
            self.o("s_nop 0")
            self.o(f"global_load_lds_dwordx4 {T2}, s[98:99]")
        self.o(f"L_fd_{L}:")
        self.o(f"s_mov_b32 {NEXTWIN}, s96")
        self.o("s_bitcmp1_b32 s97, 0")
        self.o(f"s_cbranch_scc0 L_fa_{L}")
        self.o("s_waitcnt vmcnt(0)")
        self.o("s_barrier")
        self.o(f"L_fa_{L}:")

    def window_switch(self, k1, L, y):
        """Windowed rows: if op k1 of the group (a multiple of four) is the first of the next window, the next fetch event; the
        lanes' offsets go over to the other half."""
        self.c("rows of the next window, if it starts with the next op")
        self.o(f"s_add_u32 {S0}, {POSBASE}, {k1}")
        self.o(f"s_cmp_eq_u32 {S0}, {NEXTWIN}")
        self.o(f"s_cbranch_scc0 L_nw_{L}")
        self.fetch_event(L, 64 + 16 * y)                    # (the first two position entries of this word are done with)
        self.o(f"v_add_u32_e32 {ZV}, {HALF}, {ZV}")
        self.o(f"v_add_u32_e32 {NZV}, {HALF}, {NZV}")
        self.o(f"v_add_u32_e32 {LUT2}, {LUTHALF}, {LUT2}")
        self.o(f"s_sub_u32 {HALF}, 0, {HALF}")
        self.o(f"s_sub_u32 {LUTHALF}, 0, {LUTHALF}")
        self.o(f"L_nw_{L}:")

    def slot(self, k):
        j, b = k >> 2, k & 3
        y, x, k1 = j & 1, k & 1, k + 1
        x1 = k1 & 1
        p = P(y, b)
        fwd, bwd, w, act, _ = E(x)
        L = f"{k}_%="
        self.c(f"================ op {k} of the group")
        if b == 2:
            if k == 2 and not self.win:
                self.c("pacing: the wavefronts of a SIMD that entered this group last get the issue priority, those ahead yield")
                self.o(f"v_readfirstlane_b32 {S0}, {PACE}")
                self.o(f"s_and_b32 {S0}, {S0}, %[pacemask]")
                self.o("s_cbranch_scc0 L_pp0_%=")
                self.o("s_setprio 3")
                self.o("s_branch L_ppd_%=")
                self.o("L_pp0_%=:")
                self.o("s_setprio 0")
                self.o("L_ppd_%=:")
        if k == 11:
            self.next_group_words()
        if b == 3:
            if j < 3:
                self.prep((j + 1) & 1, WORD[j + 1], WORD[j + 2] if j + 2 < 4 else NEXT[0])
            else:
                self.prep(0, NEXT[0], NEXT[1])
        word1 = WORD[k1 >> 2] if k1 < 16 else NEXT[0]
        self.c("\"recomputed\" of the next op; vcc: lanes whose next op starts a stage")
        self.o(f"v_cmp_ne_u32_sdwa {MRC[x1]}, {D((k1 >> 2) & 1)['r8']}, 0 src0_sel:BYTE_{k1 & 3} src1_sel:DWORD")
        self.o(f"v_cmp_gt_u32_sdwa vcc, {word1}, 15 src0_sel:BYTE_{k1 & 3} src1_sel:DWORD")
        self.o("s_waitcnt lgkmcnt(0)")                         # all that was asked for in the last step
        if b == 0:
            self.c("position entries of the next word")
            self.o(f"s_load_dwordx16 {PBUF((j + 1) & 1)}, {PPTR}, {64 * (j + 1)}")
        self.c(f"op {k}: sums")
        for acc, v in ((FWD, fwd), (BWD, bwd), (W_, w), (A_, act)) + (((RSF, ZQ(x)[1]), (RSB, ZQ(x)[2])) if self.rsh else ()):
            self.o(f"v_add_f64 {acc}, {acc}, {v}")
        self.o(f"s_cbranch_vccz L_ne_{L}")
        self.c("lanes whose stage ends with this op: park the stage's values, start the next stage from zero")
        self.c("(a lane that still has a record parked: store all parked ones first)")
        self.o(f"s_and_b64 {S23}, {PEND}, vcc")
        self.o(f"s_cbranch_scc0 L_nf_{L}")
        self.flush(PEND)
        self.o(f"s_mov_b64 {PEND}, 0")
        self.o(f"L_nf_{L}:")
        self.o("s_mov_b64 exec, vcc")
        self.o(f"s_or_b64 {PEND}, {PEND}, vcc")
        prevfl = P(y, b - 1)["fl"] if b else PREVFL
        self.c("the last segment closes into the peak if the op before this one is an ordinary one")
        self.o(f"s_bitcmp1_b32 {prevfl}, 1")
        self.o("s_cselect_b64 exec, vcc, 0")
        self.o(f"v_max_f64 {PEAK}, {PEAK}, {RUN}")
        self.o(f"s_and_b64 exec, vcc, {MRC[x]}")
        self.o(f"v_add_f64 {RCS}, {RCS}, {fwd}")
        self.o("s_mov_b64 exec, vcc")
        self.o(f"v_add_f64 {P_FB}, {FWD}, {BWD}")
        self.o(f"v_mov_b32 {P_PREV}, {P_META}")
        if self.rsh:
            self.o(f"v_and_or_b32 {P_META}, {self.code_word(k)}, {M0707 if b & 1 else M07}, {p['meta']}")
        else:
            word = WORD[j]
            if b:
                self.o(f"v_alignbit_b32 {P_META}, {WORD[j + 1] if j < 3 else NEXT[0]}, {word}, {8 * b}")
                word = P_META
            self.o(f"v_and_or_b32 {P_META}, {word}, {M07}, {p['meta']}")
        for to, r in ((P_RCS, RCS), (P_W, W_), (P_A, A_), (P_SAVED, SAVED), (P_PEAK, PEAK)) + (((P_RSF, RSF), (P_RSB, RSB)) if self.rsh else ()):
            self.o(f"v_mov_b64 {to}, {r}")
            self.o(f"v_mov_b64 {r}, 0")
        self.o(f"v_mov_b32 {P_RANK}, {RANK}")
        self.o(f"v_mov_b32 {RANK}, 0")
        self.o(f"v_mov_b64 {FWD}, 0")
        self.o(f"v_mov_b64 {BWD}, 0")
        self.o(f"v_mov_b64 {RUN}, 0")
        self.c("the reserved maxima run over every op but the stage's last; the next stage's offsets; its first op pays no resharding")
        self.o(f"v_mov_b32 {RANKS(x)}, 0")
        self.o(f"v_mov_b64 {ZVRK}, {NZVRK}")
        if self.rsh:
            self.o(f"v_mov_b32 {R(x1)}, 0")
        self.stage_fetch()
        self.o("s_mov_b64 exec, -1")
        self.c("that was the plan's last op (for every lane: the mark planted behind it): the padding positions need no walk")
        self.o(f"s_add_u32 {S0}, {POSBASE}, {k1}")
        self.o(f"s_cmp_eq_u32 {S0}, %[n_ops]")
        self.o("s_cbranch_scc1 L_exit_%=")
        self.o(f"L_ne_{L}:")
        if self.win and b == 3:
            self.window_switch(k1, L, y)
        self.addresses(k1)
        self.o(f"v_pk_max_u16 {RANK}, {RANK}, {RANKS(x)}")
        self.o("s_nop 0" if self.rsh else "s_nop 1")
        self.reads(k1)
        if self.rsh:
            self.o(f"ds_read_b128 {ZQ(x1)[0]}, {R(x1)}")
        self.o(f"s_andn2_b64 exec, {MRC[x]}, vcc")
        self.o(f"v_add_f64 {RCS}, {RCS}, {fwd}")
        self.c("recompute pair (this op, next op): running segment, saved activations, peak")
        self.o(f"s_and_b64 exec, exec, {MRC[x1]}")
        self.o(f"v_add_f64 {RUN}, {RUN}, {act}")
        self.o(f"s_bitcmp1_b32 {p['fl']}, 0")
        self.o("s_cselect_b64 exec, exec, 0")
        self.o(f"v_add_f64 {SAVED}, {SAVED}, {act}")
        self.o("s_not_b64 exec, exec")
        self.o(f"v_max_f64 {PEAK}, {PEAK}, {RUN}")
        self.o(f"v_mov_b64 {RUN}, 0")
        self.o("s_mov_b64 exec, -1")
        if b == 3:
            self.o(f"s_mov_b32 {PREVFL}, {p['fl']}")

    def apply_masks(self, regs, tag):
        """Code bytes of positions past the last op read as zero, and the byte right after the last op gets a stage-start
        bit, which is what ends the plan's last stage (LEFT = N - (first position of the group); five code bits used)."""
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

    def next_group_words(self):
        self.c("the next group's code words have arrived (zeros after the last group): padding and end-of-plan mark")
        if self.win:
            # (not if a window was entered since the words were asked for: they were waited for there, and the window
            # loads now in flight need not be)
            self.o(f"s_cmp_eq_u32 {ARRIVED}, 1")
            self.o("s_cbranch_scc1 L_arr_%=")
        # (vector-memory instructions complete in the order they were issued: only what was issued before the load and
        # the load itself have to be waited for, not the record stores of the last few ops)
        for n in (15, 10, 5):
            self.o(f"s_cmp_ge_u32 {VMN}, {n}")
            self.o(f"s_cbranch_scc1 L_vm{n}_%=")
        self.o("s_waitcnt vmcnt(0)")
        self.o("s_branch L_vmd_%=")
        for n in (15, 10, 5):
            self.o(f"L_vm{n}_%=:")
            self.o(f"s_waitcnt vmcnt({n})")
            if n != 5:
                self.o("s_branch L_vmd_%=")
        self.o("L_vmd_%=:")
        if self.win:
            self.o("L_arr_%=:")
        self.o(f"s_sub_i32 {LEFT}, %[n_ops], {POSBASE}")
        self.o(f"s_sub_i32 {LEFT}, {LEFT}, 16")
        self.apply_masks(NEXT, "nx")

    def pace_count(self):
        self.c("pacing: count this wavefront into this group's arrival counter of its SIMD (the count before it: its rank there)")
        self.o(f"s_and_b32 {S0}, {GRP}, 7")
        self.o(f"s_lshl_b32 {S0}, {S0}, 2")
        self.o(f"s_add_u32 {S0}, {S0}, %[pace]")
        self.o(f"v_mov_b32 {T3}, {S0}")
        self.o(f"v_mov_b32 {T2}, 1")
        self.o("s_mov_b64 exec, 1")
        self.o(f"ds_add_rtn_u32 {PACE}, {T3}, {T2}")
        self.o("s_mov_b64 exec, -1")

    def build(self):
        o, c = self.o, self.c
        c("---- set-up (all 64 lanes are active)")
        o(f"s_add_u32 {NGRP}, %[n_ops], 15")
        o(f"s_lshr_b32 {NGRP}, {NGRP}, 4")
        o(f"v_mov_b64 {GLOGS}, %[glogs]")
        o(f"v_mov_b32 {LUT2}, %[lut2]")
        o(f"v_mov_b64 {ZVRK}, %[zvrk]")
        o(f"s_mov_b64 {CPTR}, %[codes]")
        o(f"s_mov_b64 {PPTR}, %[pos]")
        o("s_mov_b64 s[24:25], %[recbase]")
        o("s_and_b32 s25, s25, 0xffff")
        o(f"s_mov_b32 s26, {5 * 16384}")
        o("s_mov_b32 s27, 0x00020000")
        o(f"s_mov_b32 {KC}, 0x{'00070707' if self.rsh else '00000707'}")
        o(f"s_mov_b64 {PEND}, 0")
        if not self.win:
            for i in range(1, 5):
                o(f"s_mov_b32 {SOFF[i]}, {16384 * i}")
        o(f"s_movk_i32 {LASTPLACE}, {16 * 128}")
        o(f"v_mov_b32 {P_META}, %[meta0]")
        o(f"v_mov_b32 {RINGV}, 0")
        o(f"v_mov_b32 {KV}, %[kv]")
        o(f"v_mov_b32 {M07}, 0x00000707")
        o(f"v_mov_b32 {M0707}, 0x00070700")
        o(f"s_mov_b32 {K08}, 0x08080808")
        o(f"s_mov_b32 {K1F}, 0x1f1f1f1f")
        o(f"s_movk_i32 {K78}, 0x78")
        o(f"s_mov_b32 {GRP}, 0")
        o(f"s_mov_b32 {POSBASE}, 0")
        o(f"s_mov_b32 {PREVFL}, 0")
        if self.win:
            c("issue priority of this wavefront: the deeper its plans, the higher (the others wait for it at every window)")
            for lvl in (3, 2, 1):
                o(f"s_cmp_eq_u32 %[prio], {lvl}")
                o(f"s_cbranch_scc0 L_np{lvl}_%=")
                o(f"s_setprio {lvl}")
                o(f"L_np{lvl}_%=:")
            o(f"s_mov_b64 {DMAPTR}, %[dma]")
            o(f"s_mov_b32 {HALF}, %[half]")
            o(f"s_mov_b32 {LUTHALF}, %[luthalf]")
            o(f"s_mov_b32 {ARRIVED}, 0")
            o(f"s_mov_b32 {EVT}, 0")
            c("window 0 (waited for), then window 1")
            self.fetch_event("s0_%=", 80)
            self.fetch_event("s1_%=", 80)
        o(f"global_load_dwordx4 v[104:107], %[codeoff], {CPTR}")
        o(f"s_load_dwordx16 {PBUF(0)}, {PPTR}, 0")
        for r in (FWD, BWD, RUN, PEAK, RCS, RSF, RSB, W_, A_, SAVED, P_RSF, P_RSB):
            o(f"v_mov_b64 {r}, 0")
        o(f"v_mov_b32 {RANK}, 0")
        o(f"v_mov_b32 {PLACE}, %[place]")
        o(f"v_mov_b32 {R(0)}, 0")
        self.stage_fetch()
        o("s_waitcnt vmcnt(0) lgkmcnt(0)")
        o(f"s_mov_b32 {LEFT}, %[n_ops]")
        self.apply_masks(WORD, "w0")
        self.prep(0, WORD[0], WORD[1])
        o(f"v_cmp_ne_u32_sdwa {MRC[0]}, {D(0)['r8']}, 0 src0_sel:BYTE_0 src1_sel:DWORD")
        self.addresses(0)
        o("s_nop 2")
        self.reads(0)
        if self.rsh:
            o(f"ds_read_b128 {ZQ(0)[0]}, {R(0)}")
        c("---- one 16-op group per iteration")
        o("L_group_%=:")
        o(f"s_add_u32 {S0}, {GRP}, 1")
        o(f"s_cmp_lt_u32 {S0}, {NGRP}")
        o("s_cbranch_scc0 L_last_%=")
        o(f"s_add_u32 {CPTR_LO}, {CPTR_LO}, %[gstride_lo]")
        o(f"s_addc_u32 {CPTR_HI}, {CPTR_HI}, %[gstride_hi]")
        o(f"global_load_dwordx4 v[108:111], %[codeoff], {CPTR}")
        o("s_branch L_loaded_%=")
        o("L_last_%=:")
        for r in NEXT:
            o(f"v_mov_b32 {r}, 0")
        o("L_loaded_%=:")
        o(f"s_mov_b32 {VMN}, 0")
        if self.win:
            o(f"s_mov_b32 {ARRIVED}, 0")
        else:
            self.pace_count()
        for k in range(16):
            self.slot(k)
        c("---- next group")
        for j in range(4):
            o(f"v_mov_b32 {WORD[j]}, {NEXT[j]}")
        o(f"s_add_u32 {PPTR_LO}, {PPTR_LO}, 256")
        o(f"s_addc_u32 {PPTR_HI}, {PPTR_HI}, 0")
        o(f"s_add_u32 {POSBASE}, {POSBASE}, 16")
        o(f"s_add_u32 {GRP}, {GRP}, 1")
        o(f"s_cmp_lt_u32 {GRP}, {NGRP}")
        o("s_cbranch_scc1 L_group_%=")
        o("L_exit_%=:")
        c("the records parked last (the plan's last op closed a stage of every lane)")
        self.flush("-1")
        o("s_waitcnt vmcnt(0) lgkmcnt(0)")
        o("s_setprio 0")
        o(f"v_mov_b32 %[placed], {PLACE}")
        o(f"v_mov_b32 %[stored], {RINGV}")
        return self.lines


def c_string(lines):
    out = []
    for ln in lines:
        assert '"' not in ln.replace('"recomputed"', "") and "\\" not in ln
        out.append('    "' + ln.replace('"', "'") + '\\n"')
    return " \\\n".join(out)


def render():
    """The text of ace_dense_loop_asm.inc."""
    parts = ["// Generated by gen_dense_loop_asm.py -- do not edit.  gfx950 assembly of the op loop over the dense tables,",
             "// one text per (rows resident / windowed, resharding on / off); see the generator for the design.", "#pragma once", ""]
    for win in (0, 1):
        for rsh in (1, 0):
            parts.append(f"#define ACE_DENSE_ASM{'_WIN' if win else ''}_RSH{rsh} \\")
            parts.append(c_string(Dense(bool(rsh), bool(win)).build()))
            parts.append("")
    clob = ", ".join(f'"v{i}"' for i in range(28, 128)) + ", " + ", ".join(f'"s{i}"' for i in range(24, 100) if i not in (32, 33))   # (s32 / s33 are the ABI's stack registers)
    parts.append(f"#define ACE_DENSE_ASM_CLOBBERS {clob}, \"vcc\", \"scc\", \"memory\"")
    parts.append("")
    return "\n".join(parts)


def main():
    path = os.path.join(HERE, "ace_dense_loop_asm.inc")
    with open(path, "w") as f:
        f.write(render())
    print("wrote", path)


if __name__ == "__main__":
    main()
