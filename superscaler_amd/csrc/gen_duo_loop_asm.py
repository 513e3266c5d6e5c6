"""Writes ace_duo_loop_asm.inc: the op loop of the scoring kernel for mid-sized batches (ace_duo.h) as gfx950 assembly.

    python3 superscaler_amd/csrc/gen_duo_loop_asm.py

Same operations per plan, in the same order, as the loop of gen_dense_loop_asm.py and over the same tables (which that file and
ace_dense.h describe), split over two lanes of different wavefronts:
  time     forward, backward, recompute and resharding sums; stores 32 bytes of a stage's record
  memory   weights, activations, saved activations, running segment and peak, reserved ranks; stores the other 40
and, along the sequence, over the wavefronts of several parts: a part's lane walks from the part's first group on, stores
the stages that start in the part, and stops behind the last of them (at or behind `cut`, the next part's first position).
What it adds up before the first stage that starts there belongs to the part before it and is not stored.

Written for one to four wavefronts per SIMD, where what counts is how long a wavefront takes per op: five to six cycles for an
instruction of any kind and more where a lone one's follow each other, 60 for an LDS read, 22 for a taken branch.  So a step has as
few instructions as the role allows (time 19, memory 24 where no lane ends a stage), one wait and one branch; the code words of
group g + 2 are asked for while group g is walked; the two scalars per position are loaded for eight ops at once.  (Measured at 8,192
plans of 523 ops, and all the same: the reads in front of the sums, so that nothing waits for them; the code of a stage's end out of the
way of the steps without one; the position scalars always in the scalar cache.  It is the number of instructions that counts: the
longest wavefront spends 250 cycles per op while 64 plans' stages end, 160 afterwards.)  Records are stored where a stage ends (few
plans per CU: what the stores cost the large batches does not show here), through a buffer whose bounds drop what belongs to
another part and what a seventeenth stage would write.
The loop ends with the plan's last op, behind which a stage start is planted, if not with its part.

One text per (role, resharding on / off).  v28-v95 and s24-s99 belong to the loop.
"""
import os

HERE = os.path.dirname(os.path.abspath(__file__))

# time: record pieces {forward + backward, recompute} {resharding forward, backward}
FB, RCS, RSF, RSB, FWD, BWD = (f"v[{32 + 2 * i}:{33 + 2 * i}]" for i in range(6))
# memory: {weights, activations} {saved, peak} {ranks, record word}
W_, A_, SAVED, PEAK = (f"v[{32 + 2 * i}:{33 + 2 * i}]" for i in range(4))
RANK, META, RUN = "v40", "v41", "v[42:43]"


def pair(b):
    return f"v[{b}:{b + 1}]"


def quad(b):
    return f"v[{b}:{b + 3}]"


def R(x):                                    # LDS address of an op pair's cost
    return f"v{60 + x}"


WORD = [f"v{62 + j}" for j in range(4)]
NEXT = [f"v{66 + j}" for j in range(4)]
FAR = [f"v{70 + j}" for j in range(4)]


def D(y):                                    # per 4-op word: codes 0 1 2 + constant, codes 2 3 4 + constant, recompute bits
    b = 74 + 3 * y
    return dict(a01=f"v{b}", a23=f"v{b + 1}", r8=f"v{b + 2}")


ZVRK, ZV, RK, NZVRK = "v[80:81]", "v80", "v81", "v[82:83]"
GLOGS, GLOGS_LO = "v[84:85]", "v84"
LUT2 = "v86"
WSOFF, WSNEXT = "v87", "v88"                 # where the lane's current record and the one after it go (0x80000000: nowhere)
T1, T2, T3, KV, M07, M0707 = "v89", "v90", "v91", "v92", "v93", "v94"

SRD = "s[24:27]"
CPTR, CPTR_LO, CPTR_HI = "s[28:29]", "s28", "s29"
PPTR, PPTR_LO, PPTR_HI = "s[36:37]", "s36", "s37"
GRP, LEFT, K1F, KC, K08, POSBASE = "s30", "s31", "s38", "s39", "s40", "s41"
MRC = ["s[42:43]", "s[58:59]"]
CUTA, CUTB, K78, PIECE1, PIECE2 = "s34", "s35", "s44", "s45", "s46"
VMN, NGRP, MASK, WSLIMIT, PLANT, PREVFL = "s50", "s51", "s52", "s54", "s56", "s62"
S0, S1, S2, S23 = "s96", "s97", "s98", "s[98:99]"


def P(k):                                    # entry of op k (0 .. 16): dot4 scalar of its row; of its pair (time), record word with flags (memory)
    b = 64 + 16 * ((k >> 3) & 1) + 2 * (k & 7)
    return f"s{b}", f"s{b + 1}"


def PBUF(h):
    return f"s[{64 + 16 * h}:{79 + 16 * h}]"


class Duo:
    def __init__(self, time, rsh):
        self.time, self.resharding, self.rsh, self.lines = time, rsh, time and rsh, []

    def o(self, s):
        self.lines.append(s)

    def c(self, s):
        self.lines.append("; " + s)

    def E(self, x):                          # entries of an op: time {fwd, bwd}, memory {weights, act, ranks}
        return [pair(44 + 4 * x), pair(46 + 4 * x)] if self.time else [pair(44 + 6 * x), pair(46 + 6 * x), pair(48 + 6 * x)]

    def ranks(self, x):
        return f"v{48 + 6 * x}"

    def Z(self, x):
        return quad(52 + 4 * x), pair(52 + 4 * x), pair(54 + 4 * x)

    def prep(self, y, wa, wb):
        d = D(y)
        self.o(f"v_alignbit_b32 {d['a23']}, {wb}, {wa}, 16")
        self.o(f"v_and_or_b32 {d['a01']}, {wa}, {KC}, {KV}")
        self.o(f"v_and_or_b32 {d['a23']}, {d['a23']}, {KC}, {KV}")
        self.o(f"v_and_b32 {d['r8']}, {K08}, {wa}")

    def code_word(self, k):
        return D((k >> 2) & 1)["a01" if (k & 3) < 2 else "a23"]

    def stage_fetch(self):
        self.o(f"v_bfi_b32 {T3}, {K78}, {GLOGS_LO}, {LUT2}")
        self.o(f"v_lshrrev_b64 {GLOGS}, 4, {GLOGS}")
        self.o(f"ds_read_b64 {NZVRK}, {T3}")

    def addresses(self, k1):
        hot, pk = P(k1)
        self.o(f"v_dot4_u32_u8 {T1}, {self.code_word(k1)}, {hot}, {ZV}")
        if self.rsh:
            self.o(f"v_dot4_u32_u8 {T2}, {self.code_word(k1)}, {pk}, {RK}")

    def reads(self, k1):
        x1 = k1 & 1
        for e, i in zip(self.E(x1), (0, 1) if self.time else (2, 3, 4)):
            self.o(f"ds_read_b64 {e}, {T1}" + (f" offset:{8 * i}" if i else ""))
        if self.rsh:
            self.o(f"ds_read_u16 {R(1 - x1)}, {T2}")
            self.o(f"ds_read_b128 {self.Z(x1)[0]}, {R(x1)}")

    def compares(self, i):
        """Op i (1 .. 16): recomputed; vcc: starts a stage."""
        word = WORD[i >> 2] if i < 16 else NEXT[0]
        self.o(f"v_cmp_ne_u32_sdwa {MRC[i & 1]}, {D((i >> 2) & 1)['r8']}, 0 src0_sel:BYTE_{i & 3} src1_sel:DWORD")
        self.o(f"v_cmp_gt_u32_sdwa vcc, {word}, 15 src0_sel:BYTE_{i & 3} src1_sel:DWORD")

    def stage_end(self, k):
        """Lanes whose stage ends with op k (vcc): its record, the next one's place (none if the next op is the next part's)."""
        j, b, x = k >> 2, k & 3, k & 1
        if self.time:
            self.o(f"s_and_b64 exec, vcc, {MRC[x]}")
            self.o(f"v_add_f64 {RCS}, {RCS}, {self.E(x)[0]}")
            self.o("s_mov_b64 exec, vcc")
            self.o(f"v_add_f64 {FB}, {FWD}, {BWD}")
            stores = [("dwordx4", "v[32:35]", "0"), ("dwordx4", "v[36:39]", PIECE1)]
        else:
            self.c("(the last segment closes into the peak if the op before this one is an ordinary one)")
            prev = P(k - 1)[1] if k & 7 else PREVFL
            self.o(f"s_bitcmp1_b32 {prev}, 13")
            self.o("s_cselect_b64 exec, vcc, 0")
            self.o(f"v_max_f64 {PEAK}, {PEAK}, {RUN}")
            self.o("s_mov_b64 exec, vcc")
            if self.resharding:
                self.o(f"v_and_or_b32 {META}, {self.code_word(k)}, {M0707 if b & 1 else M07}, {P(k)[1]}")
            else:
                word = WORD[j]
                if b:
                    self.o(f"v_alignbit_b32 {META}, {WORD[j + 1] if j < 3 else NEXT[0]}, {word}, {8 * b}")
                    word = META
                self.o(f"v_and_or_b32 {META}, {word}, {M07}, {P(k)[1]}")
            stores = [("dwordx4", "v[32:35]", "0"), ("dwordx4", "v[36:39]", PIECE1), ("dwordx2", "v[40:41]", PIECE2)]
        self.o(f"s_add_u32 {VMN}, {VMN}, {len(stores)}")
        for width, regs, off in stores:
            self.o(f"buffer_store_{width} {regs}, {WSOFF}, {SRD}, {off} offen")
        self.o(f"v_max_u32_e32 {WSOFF}, {CUTA if k < 15 else CUTB}, {WSNEXT}")
        self.o(f"v_add_u32_e32 {WSNEXT}, %[wsstride], {WSNEXT}")
        self.c("the next stage: from zero, its offsets; its first op pays no resharding, and the reserved maxima did not take this one")
        self.o(f"v_mov_b64 {ZVRK}, {NZVRK}")
        for r in (FWD, BWD, RCS) + ((RSF, RSB) if self.rsh else ()) if self.time else (RUN, W_, A_, SAVED, PEAK):
            self.o(f"v_mov_b64 {r}, 0")
        if self.rsh:
            self.o(f"v_mov_b32 {R(1 - x)}, 0")
        if not self.time:
            self.o(f"v_mov_b32 {RANK}, 0")
            self.o(f"v_mov_b32 {self.ranks(x)}, 0")
        self.stage_fetch()
        self.o("s_mov_b64 exec, -1")
        self.o(f"s_add_u32 {S0}, {POSBASE}, {k + 1}")
        self.o(f"s_cmp_eq_u32 {S0}, %[n_ops]")
        self.o("s_cbranch_scc1 L_exit_%=")

    def step(self, k):
        j, b, x, k1 = k >> 2, k & 3, k & 1, k + 1
        e = self.E(x)
        self.c(f"================ op {k} of the group")
        if b == 3:
            n = j + 1
            self.prep(n & 1, WORD[n] if n < 4 else NEXT[0], WORD[n + 1] if n + 1 < 4 else NEXT[n - 3])
        self.compares(k1)
        self.o("s_waitcnt lgkmcnt(0)")                         # all that was asked for in the last step
        if k & 7 == 0:
            self.o(f"s_load_dwordx16 {PBUF(((k >> 3) + 1) & 1)}, {PPTR}, {64 * ((k >> 3) + 1)}")
        if self.time:
            sums = [(FWD, e[0]), (BWD, e[1])] + ([(RSF, self.Z(x)[1]), (RSB, self.Z(x)[2])] if self.rsh else [])
        else:
            sums = [(W_, e[0]), (A_, e[1])]
        for acc, v in sums:
            self.o(f"v_add_f64 {acc}, {acc}, {v}")
        self.o(f"s_cbranch_vccz L_ne_{k}_%=")
        self.stage_end(k)
        self.o(f"L_ne_{k}_%=:")
        self.addresses(k1)
        if self.time:
            self.o(f"s_andn2_b64 exec, {MRC[x]}, vcc")
            self.o(f"v_add_f64 {RCS}, {RCS}, {e[0]}")
            self.o("s_mov_b64 exec, -1")
            self.reads(k1)
        else:
            self.o(f"v_pk_max_u16 {RANK}, {RANK}, {self.ranks(x)}")
            self.o("s_nop 1")
            self.reads(k1)
            self.c("recompute pair (this op, next op): running segment, saved activations, peak")
            self.o(f"s_and_b64 exec, {MRC[0]}, {MRC[1]}")
            self.o("s_andn2_b64 exec, exec, vcc")
            self.o(f"v_add_f64 {RUN}, {RUN}, {e[1]}")
            self.o(f"s_bitcmp1_b32 {P(k)[1]}, 12")
            self.o("s_cselect_b64 exec, exec, 0")
            self.o(f"v_add_f64 {SAVED}, {SAVED}, {e[1]}")
            self.o("s_not_b64 exec, exec")
            self.o(f"v_max_f64 {PEAK}, {PEAK}, {RUN}")
            self.o(f"v_mov_b64 {RUN}, 0")
            self.o("s_mov_b64 exec, -1")
            if k & 7 == 7:
                self.o(f"s_mov_b32 {PREVFL}, {P(k)[1]}")

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
        o("s_lshl_b32 s26, %[wsstride], 4")
        o("s_mov_b32 s27, 0x00020000")
        o(f"s_mov_b32 {WSLIMIT}, s26")
        o(f"s_mov_b32 {PIECE1}, %[wspiece]")
        o(f"s_lshl_b32 {PIECE2}, {PIECE1}, 1")
        o(f"s_mov_b32 {KC}, 0x{'00070707' if self.resharding else '00000707'}")
        o(f"v_mov_b32 {KV}, %[kv]")
        o(f"v_mov_b32 {M07}, 0x00000707")
        o(f"v_mov_b32 {M0707}, 0x00070700")
        o(f"s_mov_b32 {K08}, 0x08080808")
        o(f"s_mov_b32 {K1F}, 0x1f1f1f1f")
        o(f"s_movk_i32 {K78}, 0x78")
        o(f"s_mov_b32 {GRP}, %[grp]")
        o(f"s_lshl_b32 {POSBASE}, {GRP}, 4")
        o(f"s_mov_b32 {PREVFL}, 0")
        o(f"global_load_dwordx4 v[{WORD[0][1:]}:{WORD[3][1:]}], %[codeoff], {CPTR}")
        self.next_code()
        o(f"s_add_u32 {S0}, {GRP}, 1")
        o(f"s_cmp_lt_u32 {S0}, {NGRP}")
        self.load_group(NEXT, "n0")
        o(f"s_load_dwordx16 {PBUF(0)}, {PPTR}, 0")
        for r in ((FWD, BWD, FB, RCS, RSF, RSB) if self.time else (W_, A_, SAVED, PEAK, RUN)):
            o(f"v_mov_b64 {r}, 0")
        if not self.time:
            o(f"v_mov_b32 {RANK}, 0")
        o(f"v_mov_b32 {WSOFF}, %[recoff]")
        o(f"v_mov_b32 {WSNEXT}, %[recnext]")
        if self.rsh:
            o(f"v_mov_b32 {R(0)}, 0")
        self.stage_fetch()
        o("s_waitcnt vmcnt(0) lgkmcnt(0)")
        o(f"s_sub_i32 {LEFT}, %[n_ops], {POSBASE}")
        self.apply_masks(WORD, "w0")
        o(f"s_sub_i32 {LEFT}, {LEFT}, 16")
        self.apply_masks(NEXT, "w1")
        self.prep(0, WORD[0], WORD[1])
        o(f"v_cmp_ne_u32_sdwa {MRC[0]}, {D(0)['r8']}, 0 src0_sel:BYTE_0 src1_sel:DWORD")
        self.addresses(0)
        o("s_nop 2")
        self.reads(0)
        c("---- one 16-op group per iteration")
        o("L_group_%=:")
        self.next_code()
        o(f"s_add_u32 {S0}, {GRP}, 2")
        o(f"s_cmp_lt_u32 {S0}, {NGRP}")
        self.load_group(FAR, "f")
        o(f"s_mov_b32 {VMN}, 0")
        c("(the stage that starts with an op at or behind the cut is the next part's)")
        o(f"s_cmp_ge_u32 {POSBASE}, %[cut]")
        o(f"s_cselect_b32 {CUTA}, 0x80000000, 0")
        o(f"s_add_u32 {S0}, {POSBASE}, 16")
        o(f"s_cmp_ge_u32 {S0}, %[cut]")
        o(f"s_cselect_b32 {CUTB}, 0x80000000, 0")
        for k in range(16):
            self.step(k)
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
        o(f"s_add_u32 {PPTR_LO}, {PPTR_LO}, 128")
        o(f"s_addc_u32 {PPTR_HI}, {PPTR_HI}, 0")
        o(f"s_add_u32 {POSBASE}, {POSBASE}, 16")
        o(f"s_sub_i32 {LEFT}, %[n_ops], {POSBASE}")
        o(f"s_sub_i32 {LEFT}, {LEFT}, 16")
        self.apply_masks(NEXT, "nx")
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
        o("L_exit_%=:")
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
    for role, time in (("TIME", True), ("MEMORY", False)):
        for rsh in (1, 0):
            parts += [f"#define ACE_DUO_ASM_{role}_RSH{rsh} \\", c_string(Duo(time, bool(rsh)).build()), ""]
    clob = ", ".join(f'"v{i}"' for i in range(28, 96)) + ", " + ", ".join(f'"s{i}"' for i in range(24, 100) if i not in (32, 33))   # (s32 / s33 are the ABI's stack registers)
    parts += [f"#define ACE_DUO_ASM_CLOBBERS {clob}, \"vcc\", \"scc\", \"memory\"", ""]
    return "\n".join(parts)


def main():
    path = os.path.join(HERE, "ace_duo_loop_asm.inc")
    with open(path, "w") as f:
        f.write(render())
    print("wrote", path)


if __name__ == "__main__":
    main()
