"""The kernel of mid-sized batches (superscaler_amd/csrc/ace_duo.h: a plan walked by several lanes of different wavefronts).

On the GPU: around the batch sizes at which the launcher changes the workgroup, every plan against the C oracle, statuses of
malformed plans against the emulation.  On the CPU: the committed op loop is what its generator writes."""
import importlib.util
import os
import re

import numpy as np
import pytest

from superscaler_amd import synth
from superscaler_amd.plan import PlanBatch
from tests.helpers import c_oracle_scores, emu_score
from tests.test_small_batches import SETTINGS, WORKLOADS, tables_for, with_recompute

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "superscaler_amd", "csrc")


def test_committed_duo_loop_is_the_generators_output():
    spec = importlib.util.spec_from_file_location("gen_duo_loop_asm", os.path.join(CSRC, "gen_duo_loop_asm.py"))
    gen = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(gen)
    text = gen.render()
    with open(os.path.join(CSRC, "ace_duo_loop_asm.inc")) as f:
        assert f.read() == text
    # the operands of the statement live below v28 / s24, the stack registers are s32 / s33
    body = text.split("#define ACE_DUO_ASM_CLOBBERS")[0]
    for kind, low, high in (("v", 28, 127), ("s", 24, 99)):
        for m in re.finditer(rf"\b{kind}(\d+)\b|\b{kind}\[(\d+):(\d+)\]", body):
            a, b = int(m.group(1) or m.group(2)), int(m.group(1) or m.group(3))
            assert low <= a <= b <= high and not (kind == "s" and a <= 33 and b >= 32), m.group(0)


@pytest.mark.gpu
@pytest.mark.parametrize("name,mode,sizes", [("gpt3_13b", "plain", (3840, 4096, 4097, 16385)), ("t5_770m", "min", (8191,)), ("gpt3_175b", "noreserved", (4999,)),
                                             ("gpt3_1_3b", "min", (16384,)), ("gpt_wide_stages", "plain", (5000, 32768, 32769, 65537)),
                                             ("gpt_16ops", "noreserved", (65536,)), ("gpt_3tp", "min", (20001, 100001)),
                                             ("t5_1layer", "plain", (16383, 70000))])
def test_mid_sized_batches_on_the_gpu(name, mode, sizes):
    from superscaler_amd.evaluator import PlanEvaluator
    w = WORKLOADS[name]
    tables = tables_for(w, **SETTINGS[mode])
    assert tables.n_windows == 1
    ev = PlanEvaluator(tables)
    for n in sizes:
        print(f"[case] {name} {mode} plans={n}", flush=True)
        batch = with_recompute(synth.make_plans(w, tables, n_plans=n, seed_offset=n), 0.6, n)
        it, pk, fe, st = ev.score_host(batch)
        cit, cpk, cfe, cer = c_oracle_scores(tables, batch, threads=8)
        assert not cer.any() and (st == 0).all()
        assert np.array_equal(it, cit) and np.array_equal(pk, cpk) and np.array_equal(fe, cfe)
    # malformed plans among good ones: status and NaN as everywhere
    bad = PlanBatch(batch.codes.copy(), batch.hdr.copy())
    bad.codes[0, 0] &= 0xEF                 # no stage start in front
    bad.codes[1, 1:] |= 16                  # a stage per op
    bad.hdr[2, 0] = 40                      # more stages than there may be
    bad.hdr[3, 0] |= 0xff00                 # no such micro-batch size
    got = [x.cpu().numpy() for x in ev.score(ev.upload(bad, validate=False))[:4]]
    want = emu_score(tables, bad.slice(0, 64))
    for g, x in zip(got, want):
        assert x is None or np.array_equal(g[:64], x, equal_nan=True)
    assert np.array_equal(got[0][64:], it[64:]) and np.array_equal(got[1][64:], pk[64:])
    ev.close()


@pytest.mark.gpu
@pytest.mark.parametrize("name,mode,sizes", [("gpt_16ops", "plain", (65537, 131072, 200001, 262144)), ("gpt_wide_stages", "min", (262145, 300003)),
                                             ("t5_1layer", "noreserved", (147456, 600001)), ("gpt3_1_3b", "plain", (270000,)),
                                             ("wresnet_1b", "plain", (7680, 7681, 16385, 270001)), ("resnet_1111", "min", (8000, 70000)),
                                             ("resnet_16gpus", "noreserved", (16384, 33333)),
                                             # (windowed rows of which the table compiler's are too short to be fetched)
                                             ("resnet_2tp", "plain", (4096, 4097, 131073))])
def test_large_batches_in_even_shares_on_the_gpu(name, mode, sizes):
    from superscaler_amd.evaluator import PlanEvaluator
    w = WORKLOADS[name]
    tables = tables_for(w, **SETTINGS[mode])
    ev = PlanEvaluator(tables)
    base = synth.make_plans(w, tables, n_plans=40000, seed_offset=7)
    rng = np.random.default_rng(1)
    for n in sizes:
        print(f"[case] {name} {mode} plans={n}", flush=True)
        pick = rng.integers(0, base.n_plans, n)
        want = c_oracle_scores(tables, base, threads=8)
        batch = PlanBatch(base.codes[pick], base.hdr[pick])
        it, pk, fe, st = ev.score_host(batch)
        assert (st == 0).all() and np.array_equal(it, want[0][pick]) and np.array_equal(pk, want[1][pick]) and np.array_equal(fe, want[2][pick])
    ev.close()


def with_rows_in_another_order(tables, seed):
    """The same tables with the resident rows in other LDS slots."""
    import copy
    t = copy.copy(tables)
    n = len(t.win_rows)
    assert t.n_windows == 1 and np.array_equal(t.win_rows[:, 1], np.arange(n) * t.rows.shape[1] * 8)
    slot = np.random.default_rng(seed).permutation(n).astype(np.uint32)
    t.win_rows = np.stack([t.win_rows[:, 0], slot * np.uint32(t.rows.shape[1] * 8)], axis=1)
    info = t.pos_info
    t.pos_info = (info & np.uint32(0xffff0000)) | slot[info & 0xff] | slot[(info >> 8) & 0xff] << np.uint32(8)
    return t


@pytest.mark.gpu
@pytest.mark.parametrize("name,sizes", [("gpt_wide_stages", (100, 4097, 131073)), ("t5_1layer", (5000,))])
def test_rows_in_another_order_on_the_gpu(name, sizes):
    from superscaler_amd.evaluator import PlanEvaluator
    w = WORKLOADS[name]
    tables = tables_for(w)
    ev = PlanEvaluator(with_rows_in_another_order(tables, 3))
    for n in sizes:
        print(f"[case] {name} plans={n}", flush=True)
        batch = synth.make_plans(w, tables, n_plans=n, seed_offset=n)
        it, pk, fe, st = ev.score_host(batch)
        want = c_oracle_scores(tables, batch, threads=8)
        assert (st == 0).all() and np.array_equal(it, want[0]) and np.array_equal(pk, want[1]) and np.array_equal(fe, want[2])
    ev.close()
