"""The dense tables of large batches (superscaler_amd/csrc/ace_dense.h).

On the CPU: the tables as the library builds them, walked like the assembly loop walks them (one dot product per address, ranks of the
reserved sizes, parked records), against the C oracle and, for codes that name no profiled entry, against the per-plan state
machine; the committed loop text is what its generator writes.  On the GPU: every plan against the C oracle at the sizes where the
division into workgroups changes, and malformed plans among good ones."""
import dataclasses
import importlib.util
import os
import re

import numpy as np
import pytest

from superscaler_amd import synth
from superscaler_amd.plan import PlanBatch
from tests.helpers import c_oracle_scores, emu_dense_score, emu_score
from tests.test_small_batches import SETTINGS, WORKLOADS, tables_for, with_recompute

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "superscaler_amd", "csrc")
#: the tables that fit (not: memory of collectives)
DENSE = {"gpt3_1_3b", "gpt3_13b", "gpt3_175b", "t5_770m", "gpt_1tp_1mbs", "gpt_16ops", "gpt_wide_stages", "gpt_3tp", "t5_1layer", "t5_1tp",
         "wresnet_1b", "resnet_1111", "resnet_16gpus", "resnet_2tp", "gpt_6mbs_64gpus"}


def test_committed_dense_loop_is_the_generators_output():
    spec = importlib.util.spec_from_file_location("gen_dense_loop_asm", os.path.join(CSRC, "gen_dense_loop_asm.py"))
    gen = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(gen)
    text = gen.render()
    with open(os.path.join(CSRC, "ace_dense_loop_asm.inc")) as f:
        assert f.read() == text
    # the operands of the statement live below v28 / s24, the stack registers are s32 / s33
    body = text.split("#define ACE_DENSE_ASM_CLOBBERS")[0]
    for kind, low, high in (("v", 28, 127), ("s", 24, 99)):
        for m in re.finditer(rf"\b{kind}(\d+)\b|\b{kind}\[(\d+):(\d+)\]", body):
            a, b = int(m.group(1) or m.group(2)), int(m.group(1) or m.group(3))
            assert low <= a <= b <= high and not (kind == "s" and a <= 33 and b >= 32), m.group(0)
    dot_products_are_read_late_enough(body)


def test_duo_loops_dot_products_are_read_late_enough():
    with open(os.path.join(CSRC, "ace_duo_loop_asm.inc")) as f:
        dot_products_are_read_late_enough(f.read().split("#define ACE_DUO_ASM_CLOBBERS")[0])


def dot_products_are_read_late_enough(body):
    """A dot product is read three issue slots later at the earliest."""
    lines = [ln.strip(' "\\').replace("\\n", "") for ln in body.splitlines()]
    ops = [ln for ln in lines if ln and not ln.startswith((";", "#", "//")) and not ln.endswith(":")]
    for i, ln in enumerate(ops):
        if ln.startswith("v_dot4"):
            dst = re.search(r"(v\d+)", ln).group(1)
            slots = 0
            for nxt in ops[i + 1:]:
                if slots >= 3:
                    break
                # (another dot product is an issue slot; it reads none of these)
                assert not re.search(rf"\b{dst}\b", nxt), (ln, nxt)
                slots += 1 + (int(nxt.split()[1]) if nxt.startswith("s_nop") else 0)


@pytest.mark.parametrize("mode", SETTINGS)
@pytest.mark.parametrize("name", WORKLOADS)
def test_dense_tables_score_like_the_oracle(name, mode):
    w = WORKLOADS[name]
    tables = tables_for(w, **SETTINGS[mode])
    batch = with_recompute(synth.make_plans(w, tables, n_plans=150, seed_offset=11), 0.6, 11)
    got = emu_dense_score(tables, batch)
    if got is None:
        # (memory of collectives is on only where something is resharded)
        assert name not in DENSE or mode == "collective"
        return
    assert name in DENSE
    it, pk, fe, er = c_oracle_scores(tables, batch)
    assert np.array_equal(got[0], it) and np.array_equal(got[1], pk) and np.array_equal(got[2], fe) and not got[3].any() and not er.any()
    # an op with another code (every fifth plan: many), stage sizes outside the tables: what the tables say there as well
    rng = np.random.default_rng(5)
    bad = PlanBatch(batch.codes.copy(), batch.hdr.copy())
    hit = np.zeros(bad.codes.shape, dtype=bool)
    hit[np.arange(len(hit)), rng.integers(0, hit.shape[1], len(hit))] = True
    hit[::5] = rng.random(hit[::5].shape) < 0.05
    codes = 8 if name in synth.WORKLOADS else len(tables.db.tp_list) * tables.db.n_algo
    bad.codes[hit] = rng.integers(0, codes, hit.sum()) | (bad.codes[hit] & 24)
    bad.hdr[::9, 1] = rng.integers(0, 2 ** 32, len(bad.hdr[::9]), dtype=np.uint64).astype(np.uint32)
    bad.codes[7] |= 16                      # a stage per op
    for g, x in zip(emu_dense_score(tables, bad)[:4], emu_score(tables, bad)[:4]):
        assert np.array_equal(g, x, equal_nan=True)


@pytest.mark.gpu
@pytest.mark.parametrize("name,mode,sizes", [("gpt_wide_stages", "plain", (65537, 131073, 262145)), ("t5_1tp", "min", (65600, 262144)),
                                             ("gpt_3tp", "noreserved", (70001,)), ("gpt3_1_3b", "min", (65537,)), ("t5_770m", "plain", (98304,)),
                                             # (rows in windows)
                                             ("wresnet_1b", "min", (6145, 6537, 16385, 262145)), ("resnet_1111", "plain", (65537,)),
                                             ("resnet_16gpus", "noreserved", (6200,)), ("gpt_6mbs_64gpus", "plain", (70001,)), ("270 types", "plain", (20001,))])
def test_large_batches_over_dense_tables_on_the_gpu(name, mode, sizes):
    from superscaler_amd.evaluator import PlanEvaluator
    # (more op types than fit eight bits)
    w = WORKLOADS[name] if name in WORKLOADS else dataclasses.replace(WORKLOADS["wresnet_1b"], resnet_blocks=(3, 4, 23, 3))
    tables = tables_for(w, **SETTINGS[mode])
    assert emu_dense_score(tables, synth.make_plans(w, tables, n_plans=1)) is not None
    ev = PlanEvaluator(tables)
    base = with_recompute(synth.make_plans(w, tables, n_plans=20000, seed_offset=3), 0.6, 3)
    want = c_oracle_scores(tables, base, threads=8)
    rng = np.random.default_rng(2)
    for n in sizes:
        print(f"[case] {name} {mode} plans={n}", flush=True)
        pick = rng.integers(0, base.n_plans, n)
        batch = PlanBatch(base.codes[pick], base.hdr[pick])
        # malformed plans among good ones, in one wavefront and apart
        bad = [0, 1, 2, 3, n // 2, n - 1]
        batch.codes[bad[0], 0] &= 0xEF          # no stage start in front
        batch.codes[bad[1], 1:] |= 16           # a stage per op
        batch.hdr[bad[2], 0] = 40               # more stages than there may be
        batch.hdr[bad[3], 0] |= 0xff00          # no such micro-batch size
        batch.codes[bad[4], ::3] |= 16
        batch.codes[bad[5], 1:] |= 16
        it, pk, fe, st = [x.cpu().numpy() for x in ev.score(ev.upload(batch, validate=False))[:4]]
        good = np.ones(n, dtype=bool)
        good[bad] = False
        assert (st[good] == 0).all()
        assert np.array_equal(it[good], want[0][pick][good]) and np.array_equal(pk[good], want[1][pick][good])
        assert np.array_equal(fe[good], want[2][pick][good])
        for g, x in zip((it, pk, fe, st), emu_score(tables, PlanBatch(batch.codes[bad], batch.hdr[bad]))[:4]):
            assert np.array_equal(g[bad], x, equal_nan=True)
    ev.close()
