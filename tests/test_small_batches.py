"""The kernel of small batches (superscaler_amd/csrc/ace_spread.h: one plan or single-stage query per workgroup).

On the CPU: its phases, lane after lane, with every array (LDS included) flush against an inaccessible page, in a child
process per case (`python -m tests.test_small_batches WORKLOAD MODE`), against the state-machine emulation, which the other
CPU tests pin to the oracle.  On the GPU: around the batch sizes at which the launcher changes kernels, every plan against
the C oracle and the stage records against the emulation."""
import os
import subprocess
import sys

import numpy as np
import pytest

from superscaler_amd import synth
from superscaler_amd.plan import PlanBatch
from tests.helpers import c_oracle_scores, emu_kernel_score, emu_lib, emu_score, kernel_layout, odd_workloads

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
WORKLOADS = {**synth.WORKLOADS, **{w.name: w for w in odd_workloads()}}
SETTINGS = {"plain": {}, "min": {"memory_pred_type": "MIN"}, "noreserved": {"consider_reserved_space": False},
            "collective": {"consider_collective_memory": True}}


def tables_for(w, **settings):
    import dataclasses
    from superscaler_amd.tables import compile_tables
    graph = synth.make_graph(w)
    return compile_tables(graph, synth.make_db(w, graph), dataclasses.replace(synth.make_settings(w), **settings))


def stage_queries(batch):
    """Every stage of every plan as a single-stage query: (batch, ranges)."""
    plan, lo = np.nonzero(batch.codes & 16)
    hi = np.append(lo[1:], batch.num_ops)
    hi[np.append(plan[1:] != plan[:-1], True)] = batch.num_ops
    first = np.searchsorted(plan, plan)
    s = np.arange(len(plan)) - first
    sizes = batch.hdr[plan, 1].astype(np.uint64) | (batch.hdr[plan, 2].astype(np.uint64) << np.uint64(32))
    hdr = np.zeros((len(plan), 4), dtype=np.uint32)
    hdr[:, 0] = ((batch.hdr[plan, 0] & 0xff) - s) | (batch.hdr[plan, 0] & 0xff00)
    hdr[:, 1] = ((sizes >> (4 * s).astype(np.uint64)) & np.uint64(15)).astype(np.uint32)
    return PlanBatch(np.ascontiguousarray(batch.codes[plan]), hdr), np.stack([lo, hi], axis=1).astype(np.uint32)


def same(a, b):
    return all(np.array_equal(x, y, equal_nan=True) for x, y in zip(a, b) if x is not None)


def with_recompute(batch, p, seed):
    """A copy with other recompute bits: long runs of them (segments that reach over chunks of 256 ops)."""
    rng = np.random.default_rng(seed)
    return PlanBatch((batch.codes & np.uint8(0xF7)) | ((rng.random(batch.codes.shape) < p).astype(np.uint8) << 3), batch.hdr)


def main(name, mode):
    w = WORKLOADS[name]
    n = 12 if w.name in synth.WORKLOADS else 40
    tables = tables_for(w, **SETTINGS.get(mode, {}))
    base = synth.make_plans(w, tables, n_plans=n, seed_offset=5)
    if mode == "junk":
        # random bytes everywhere, headers and ranges included: not compared, the kernel only has to stay inside its arrays
        rng = np.random.default_rng(3)
        raw = rng.integers(0, 256, size=kernel_layout(base.codes).shape, dtype=np.uint8)
        hdr = rng.integers(0, 2 ** 32, size=base.hdr.shape, dtype=np.uint64).astype(np.uint32)
        rg = rng.integers(0, 2 * base.num_ops, size=(n, 2), dtype=np.uint64).astype(np.uint32)
        for kw in ({}, {"breakdown": True}, {"ranges": rg}):
            emu_kernel_score(tables, PlanBatch(base.codes, hdr), raw_codes=raw, spread=True, **kw)
        order = rng.integers(0, 2 ** 32, size=n, dtype=np.uint64).astype(np.uint32)
        emu_kernel_score(tables, base, order=order, spread=True)
        return
    for batch in (base, with_recompute(base, 0.97, 1), with_recompute(base, 1.0, 2)):
        assert same(emu_kernel_score(tables, batch, spread=True), emu_score(tables, batch))
        assert same(emu_kernel_score(tables, batch, breakdown=True, spread=True), emu_score(tables, batch, breakdown=True))
        q, ranges = stage_queries(batch)
        got, want = emu_kernel_score(tables, q, ranges=ranges, spread=True), emu_score(tables, q, ranges=ranges)
        assert np.array_equal(got[3], want[3]) and np.array_equal(got[4], want[4])
    # malformed plans: status and NaN as everywhere
    bad = PlanBatch(base.codes.copy(), base.hdr.copy())
    bad.codes[0, 0] &= 0xEF
    bad.codes[1, 1:] |= 16
    bad.hdr[2, 0] = 40
    bad.hdr[3, 0] |= 0xff00
    assert same(emu_kernel_score(tables, bad, spread=True), emu_score(tables, bad))


@pytest.mark.parametrize("mode", [*SETTINGS, "junk"])
@pytest.mark.parametrize("name", list(WORKLOADS))
def test_phases_on_the_cpu(name, mode):
    emu_lib()
    proc = subprocess.run([sys.executable, "-m", "tests.test_small_batches", name, mode], cwd=ROOT, stdout=subprocess.PIPE,
                          stderr=subprocess.STDOUT, text=True, timeout=600)
    assert proc.returncode == 0, f"child ended with {proc.returncode} (negative: killed by that signal)\n{proc.stdout[-2000:]}"


@pytest.mark.gpu
@pytest.mark.parametrize("name,mode,sizes", [("gpt3_13b", "plain", (1, 4096, 4097)), ("t5_770m", "min", (3, 1000)),
                                             ("gpt3_175b", "plain", (17, 1024)), ("wresnet_1b", "noreserved", (33, 4096, 4097)),
                                             ("gpt3_1_3b", "collective", (40, 1024))])
def test_small_batches_on_the_gpu(name, mode, sizes):
    from superscaler_amd.evaluator import PlanEvaluator
    w = WORKLOADS[name]
    tables = tables_for(w, **SETTINGS[mode])
    ev = PlanEvaluator(tables)
    for n in sizes:
        print(f"[case] {name} {mode} plans={n}", flush=True)
        batch = with_recompute(synth.make_plans(w, tables, n_plans=n, seed_offset=n), 0.6, n)
        it, pk, fe, st = ev.score_host(batch)
        cit, cpk, cfe, cer = c_oracle_scores(tables, batch, threads=8)
        assert not cer.any() and (st == 0).all()
        assert np.array_equal(it, cit) and np.array_equal(pk, cpk) and np.array_equal(fe, cfe)
        sub = batch.slice(0, min(n, 200))
        assert same(ev.score_host(sub, breakdown=True), emu_score(tables, sub, breakdown=True))
        q, ranges = stage_queries(sub)
        got, want = ev.score_host(q, ranges=ranges), emu_score(tables, q, ranges=ranges)
        assert np.array_equal(got[3], want[3]) and np.array_equal(got[4], want[4])
    ev.close()


if __name__ == "__main__":
    main(sys.argv[1], sys.argv[2])
