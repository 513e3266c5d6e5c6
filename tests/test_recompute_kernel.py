"""check_recompute for a whole batch in one launch (superscaler_amd/csrc/ace_recompute.h): the kernel's phases on the CPU,
arrays and LDS flush against inaccessible pages, in a child process per case (`python -m tests.test_recompute_kernel WORKLOAD
SETTINGS`), against the numpy form of the loop; on the GPU the same comparison and the error cases."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

from superscaler_amd import opgraph as og
from superscaler_amd import synth
from superscaler_amd.aceso_cost_model import CostModel
from superscaler_amd.plan import PlanBatch
from superscaler_amd.recompute import update_recompute_arrays
from tests.helpers import EmuEvaluator, emu_lib, emu_score, kernel_layout
from tests.test_small_batches import ROOT, SETTINGS, WORKLOADS


def cost_model(w, emu=True, **settings):
    import dataclasses
    graph = synth.make_graph(w)
    cm = CostModel(dataclasses.replace(synth.make_settings(w), **settings), synth.make_db(w, graph), graph)
    if emu:
        cm._evaluator = EmuEvaluator(cm.tables)
    return cm


def emu_recompute(cm, batch, codes=None):
    """(codes [P, N], flags) of ace_recompute_batch's kernel on the CPU."""
    t, lib = cm.tables, emu_lib()
    raw = kernel_layout(batch.codes) if codes is None else codes
    out, flags = np.zeros_like(raw), np.zeros(4, dtype=np.int32)
    types = np.ascontiguousarray(t.graph.type_of_pos, dtype=np.int32)
    act = np.ascontiguousarray(t.db.tables["activations"], dtype=np.float64)
    norec = ((np.asarray(t.graph.flags)[:len(t.db.op_names)] & og.F_NO_RECOMPUTE) != 0).astype(np.uint8)
    status = np.ascontiguousarray(emu_score(t, batch)[3]) if codes is None else np.zeros(batch.n_plans, dtype=np.uint8)
    hdr, ts = np.ascontiguousarray(batch.hdr), t.as_struct()
    vp = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    assert lib.ace_emu_recompute(ctypes.byref(ts), vp(raw), vp(hdr), ctypes.c_longlong(batch.n_plans), ctypes.c_double(cm.settings.memory_limit),
                                 ctypes.c_double(cm.settings.peak_mem_in_backward), vp(types), vp(act), vp(norec), vp(status), vp(out), vp(flags)) == 0
    G, P, _ = out.shape
    return np.ascontiguousarray(out.transpose(1, 0, 2).reshape(P, G * 16)[:, :batch.num_ops]), flags


def limits(cm, batch):
    """No stage, some stages, nearly all stages above it."""
    cleared = PlanBatch(batch.codes & np.uint8(0xF7), batch.hdr)
    peak = emu_score(cm.tables, cleared)[1]
    return [float(np.max(peak)), float(np.quantile(peak, 0.6)), float(np.min(peak)) * 0.7]


def main(name, mode):
    w = WORKLOADS[name]
    cm = cost_model(w, **SETTINGS.get(mode, {}))
    batch = synth.make_plans(w, cm.tables, n_plans=16 if w.name in synth.WORKLOADS else 60, seed_offset=9)
    if mode == "junk":
        rng = np.random.default_rng(2)
        raw = rng.integers(0, 256, size=kernel_layout(batch.codes).shape, dtype=np.uint8)
        hdr = rng.integers(0, 2 ** 32, size=batch.hdr.shape, dtype=np.uint64).astype(np.uint32)
        # (as many stages as the bits say, so that the stages are walked; first op opens one; 1 to 16 of them)
        raw &= np.where(rng.random(raw.shape) < 0.02, 0xff, 0xef).astype(np.uint8)
        raw[0, :, 0] |= 16
        P, N = batch.codes.shape
        codes = np.ascontiguousarray(raw.transpose(1, 0, 2).reshape(P, -1)[:, :N])
        hdr[:, 0] = (hdr[:, 0] & 0xf00) | ((codes >> 4) & 1).sum(axis=1)
        cm.settings.memory_limit = 1.0
        emu_recompute(cm, PlanBatch(codes, hdr), raw)
        return
    for limit in limits(cm, batch):
        for backward in (0, 700):
            cm.settings.memory_limit, cm.settings.peak_mem_in_backward = limit, backward
            codes, flags = emu_recompute(cm, batch)
            assert not flags.any() and np.array_equal(codes, update_recompute_arrays(cm, batch).codes)
    bad = PlanBatch(batch.codes.copy(), batch.hdr.copy())
    bad.hdr[0, 0] += 1
    assert emu_recompute(cm, bad)[1][0] == -1
    bad.hdr[0, 0] = batch.hdr[0, 0]
    bad.codes[1, 0] &= 0xEF
    assert emu_recompute(cm, bad)[1][1] == 1


@pytest.mark.parametrize("mode", [*SETTINGS, "junk"])
@pytest.mark.parametrize("name", list(WORKLOADS))
def test_phases_on_the_cpu(name, mode):
    emu_lib()
    proc = subprocess.run([sys.executable, "-m", "tests.test_recompute_kernel", name, mode], cwd=ROOT, stdout=subprocess.PIPE,
                          stderr=subprocess.STDOUT, text=True, timeout=600)
    assert proc.returncode == 0, f"child ended with {proc.returncode} (negative: killed by that signal)\n{proc.stdout[-2000:]}"


@pytest.mark.gpu
@pytest.mark.parametrize("name,mode,n", [("gpt3_13b", "plain", 700), ("t5_770m", "min", 300), ("wresnet_1b", "plain", 700),
                                         ("gpt3_175b", "noreserved", 100), ("gpt3_1_3b", "collective", 300), ("gpt_16ops", "plain", 33)])
def test_one_launch_on_the_gpu(name, mode, n):
    w = WORKLOADS[name]
    cm, ref = cost_model(w, emu=False, **SETTINGS[mode]), cost_model(w, **SETTINGS[mode])
    batch = synth.make_plans(w, cm.tables, n_plans=n, seed_offset=n)
    print(f"[case] {name} {mode} plans={n}", flush=True)
    for limit in limits(ref, batch):
        cm.settings.memory_limit = ref.settings.memory_limit = limit
        assert np.array_equal(cm.update_recompute_arrays(batch).codes, update_recompute_arrays(ref, batch).codes)
    # (ranges that a batch carries for single-stage queries do not matter: every stage of the whole plans is looked at)
    ranged = cm.evaluator.upload(batch, ranges=np.tile(np.array([[0, 1]], dtype=np.uint32), (n, 1)))
    assert np.array_equal(cm.evaluator.download(cm.update_recompute_device(ranged)).codes, update_recompute_arrays(ref, batch).codes)
    bad = PlanBatch(batch.codes.copy(), batch.hdr.copy())
    bad.hdr[0, 0] += 1
    with pytest.raises(ValueError):
        cm.update_recompute_device(cm.evaluator.upload(bad, validate=False))
    cm.close()


if __name__ == "__main__":
    main(sys.argv[1], sys.argv[2])
