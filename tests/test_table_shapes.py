"""Scoring over tables of other shapes than the configured workloads': more or fewer micro-batch sizes, devices per node and op types, so
that rows are of other lengths, fit where the configured ones do not, or go through windows.

On the CPU: the tables as the library builds them, their sizes, and every plan against the C oracle.  On the GPU: the same at batch sizes
on both sides of what decides about the kernel."""
import ctypes
import dataclasses
import time

import numpy as np
import pytest

from superscaler_amd import synth
from superscaler_amd.plan import PlanBatch
from superscaler_amd.tables import compile_tables
from tests.helpers import c_oracle_scores, emu_dense_score, emu_lib, emu_score
from tests.test_mid_batches import with_rows_in_another_order
from tests.test_small_batches import with_recompute


def workload(name, sizes, per_node=None, gpus=None, blocks=None):
    w = synth.WORKLOADS[name]
    gpus = gpus or w.num_gpus
    if blocks:
        w = dataclasses.replace(w, resnet_blocks=blocks)
    return dataclasses.replace(w, mbs_list=[1 << i for i in range(sizes)], gpus_per_node=per_node or w.gpus_per_node, num_gpus=gpus,
                               pp_choices=[s for s in w.pp_choices if s <= gpus])


#: (workload, micro-batch sizes, devices per node, devices): entries per row between 10 and 96
SHAPES = {"t5, 6 sizes": ("t5_770m", 6), "t5, 8 sizes": ("t5_770m", 8), "t5, 2 of 2": ("t5_770m", 2, 2, 8), "gpt, 6 sizes": ("gpt3_13b", 6),
          "gpt, 8 sizes": ("gpt3_1_3b", 8, 8, 32), "gpt, 7 of 4": ("gpt3_13b", 7, 4), "gpt, 8 of 2": ("gpt3_1_3b", 8, 2), "gpt, 3 of 8": ("gpt3_175b", 3, 8, 64),
          "conv, 1 of 1": ("wresnet_1b", 1, 1, 4), "conv, 3 of 1": ("wresnet_1b", 3, 1, 4), "conv, 5 of 1": ("wresnet_1b", 5, 1, 4),
          "conv, 1 of 2": ("wresnet_1b", 1, 2, 4), "conv, 6 sizes": ("wresnet_1b", 6), "conv, 38 ops": ("wresnet_1b", 4, 8, None, (1, 1, 1, 1)),
          "gpt, 10 sizes": ("gpt3_175b", 10), "gpt, 10 sizes, 523 ops": ("gpt3_13b", 10)}


#: ... over databases in which no two sizes and no two collectives' times are equal: large images
DISTINCT = {"t5, all sizes differ": ("t5_770m", 5), "t5, 8 differing": ("t5_770m", 8), "gpt, all sizes differ": ("gpt3_175b", 4), "gpt, 8 differing": ("gpt3_1_3b", 8),
            "gpt, 6 differing": ("gpt3_13b", 6)}
SHAPES.update(DISTINCT)
#: ... and that the dense form has no room for: rows resident; in windows that the assembly loop fetches; in windows of rows too short for it
OUTSIDE = {"conv, 4 of 1 differing": ("wresnet_1b", 4, 1, 4), "conv, 4 of 4 differing": ("wresnet_1b", 4, 4), "conv, 8 of 1 differing": ("wresnet_1b", 8, 1, 4),
           "gpt, 8 of 8 differing": ("gpt3_13b", 8, 8), "conv, 38 ops, 8 differing": ("wresnet_1b", 8, 8, None, (1, 1, 1, 1))}


def distinct_sizes(db, seed):
    """Every input and output size, and every collective's time, a value of its own."""
    rng = np.random.default_rng(seed)
    for key in ("input_size", "output_size"):
        a = db.tables[key]
        db.tables[key] = np.round(a * rng.uniform(0.7, 1.3, a.shape) + rng.uniform(0, 1, a.shape), 3)
    keys = sorted({"{:.0f}".format(float(x)) for x in db.tables["input_size"].ravel()}, key=float)
    for groups in db.collectives.values():
        for n in groups:
            groups[n] = {k: round(float(rng.uniform(0.1, 2.0)) * (1 + float(k) * 0.01), 3) for k in keys}
    return db


def tables_of(shape, **settings):
    """(workload, its compiled tables)"""
    w = workload(*{**SHAPES, **OUTSIDE}[shape])
    graph = synth.make_graph(w)
    db = synth.make_db(w, graph)
    return w, compile_tables(graph, distinct_sizes(db, 1) if shape in DISTINCT or shape in OUTSIDE else db, dataclasses.replace(synth.make_settings(w), **settings))


def shape_of(tables):
    """(fits, windows, LDS of a workgroup, bytes of the image, from row to row, most rows of a window)"""
    out = np.zeros(6, dtype=np.int32)
    ts = tables.as_struct()
    emu_lib().ace_emu_dense_shape(ctypes.byref(ts), out.ctypes.data_as(ctypes.c_void_p))
    return [int(x) for x in out]


@pytest.mark.parametrize("shape", SHAPES)
def test_rows_take_what_their_entries_need(shape):
    w, tables = tables_of(shape)
    ok, windows, lds, _, pitch, _ = shape_of(tables)
    entries = tables.n_diag * tables.C + 8
    # (one entry to keep banks apart; up to 255 multiples of one constant name the places of rows: of `n` rows one is a 255th of all,
    # rounded up to eight bytes, longer at most; a window's rows are fetched 1 KB at a time, in pieces of 16 bytes)
    need = 40 * (entries + 1)
    assert ok and pitch <= max(need + 8 * (need // 255 + 2), 1024 if windows else 0) and lds <= 160 * 1024


@pytest.mark.parametrize("shape", [s for s in SHAPES if s not in ("conv, 1 of 2", "conv, 6 sizes", "conv, 38 ops", "gpt, 10 sizes", "gpt, 10 sizes, 523 ops")])
def test_rows_that_fit_a_cu_are_resident(shape):
    """So that mid-sized batches have their kernel, whatever the table compiler's own rows need."""
    ok, windows, *_ = shape_of(tables_of(shape)[1])
    assert ok and windows == 0


@pytest.mark.parametrize("shape", SHAPES)
def test_every_shape_scores_like_the_oracle(shape):
    w, tables = tables_of(shape)
    batch = with_recompute(synth.make_plans(w, tables, n_plans=120, seed_offset=21), 0.6, 21)
    got = emu_dense_score(tables, batch)
    it, pk, fe, er = c_oracle_scores(tables, batch)
    assert np.array_equal(got[0], it) and np.array_equal(got[1], pk) and np.array_equal(got[2], fe) and not got[3].any() and not er.any()


def test_many_types_of_distinct_sizes_are_left_soon():
    """1,046 op types, every size and time of its own: that they do not fit is known long before all pairs of values have been compared, which
    took 1.14 s; now 0.06."""
    w = workload("wresnet_1b", 4, 8, None, (3, 4, 120, 3))
    graph = synth.make_graph(w)
    tables = compile_tables(graph, distinct_sizes(synth.make_db(w, graph), 1), synth.make_settings(w))
    shape_of(tables)
    took = []
    for _ in range(3):
        at = time.perf_counter()
        assert shape_of(tables)[0] == 0
        took.append(time.perf_counter() - at)
    assert min(took) < 0.5


def on_the_gpu(shape, sizes, **settings):
    from superscaler_amd.evaluator import PlanEvaluator
    w, tables = tables_of(shape, **settings)
    ev = PlanEvaluator(tables)
    base = with_recompute(synth.make_plans(w, tables, n_plans=9000, seed_offset=31), 0.6, 31)
    want = c_oracle_scores(tables, base, threads=8)
    rng = np.random.default_rng(4)
    for n in sizes:
        print(f"[case] {shape} plans={n}", flush=True)
        pick = rng.integers(0, base.n_plans, n)
        it, pk, fe, st = ev.score_host(PlanBatch(base.codes[pick], base.hdr[pick]))
        assert (st == 0).all() and np.array_equal(it, want[0][pick]) and np.array_equal(pk, want[1][pick]) and np.array_equal(fe, want[2][pick])
    ev.close()


@pytest.mark.gpu
@pytest.mark.parametrize("shape,sizes", [("t5, 6 sizes", (70001,)), ("gpt, 6 sizes", (65537, 262145)), ("gpt, 8 sizes", (70000,)), ("t5, 2 of 2", (65537,)),
                                         ("conv, 1 of 1", (5000, 70001)), ("conv, 1 of 2", (6537, 70001)), ("conv, 6 sizes", (65536,))])
def test_large_batches_over_other_shapes_on_the_gpu(shape, sizes):
    on_the_gpu(shape, sizes)


@pytest.mark.gpu
@pytest.mark.parametrize("shape,sizes", [("t5, 6 sizes", (5000, 8192, 65536)), ("t5, 8 sizes", (16385,)), ("gpt, 6 sizes", (4097, 32768, 65536)), ("conv, 5 of 1", (5000, 33000)),
                                         ("conv, 1 of 1", (16384,)), ("t5, all sizes differ", (8192, 65536)), ("t5, 8 differing", (5000, 70001)),
                                         ("gpt, all sizes differ", (4097, 65537)), ("gpt, 8 differing", (8192, 262145)), ("gpt, 6 differing", (20000, 131073))])
def test_mid_sized_batches_over_other_shapes_on_the_gpu(shape, sizes):
    on_the_gpu(shape, sizes)
    on_the_gpu(shape, sizes[:1], resharding=False, memory_pred_type="MIN")


@pytest.mark.gpu
@pytest.mark.parametrize("shape,sizes", [("conv, 6 sizes", (6536, 6537)), ("conv, 38 ops", (4724, 4725)), ("gpt, 10 sizes", (11004, 11005, 65537))])
def test_windows_on_both_sides_of_their_limit_on_the_gpu(shape, sizes):
    on_the_gpu(shape, sizes)


def outside_on_the_gpu(shape, sizes, order=False, **settings):
    """Tables that the dense form has no room for: every plan, malformed ones among them."""
    from superscaler_amd.evaluator import PlanEvaluator
    w, tables = tables_of(shape, **settings)
    base = with_recompute(synth.make_plans(w, tables, n_plans=9000, seed_offset=33), 0.6, 33)
    assert emu_dense_score(tables, base.slice(0, 1)) is None
    want = c_oracle_scores(tables, base, threads=8)
    ev = PlanEvaluator(with_rows_in_another_order(tables, 5) if order else tables)
    rng = np.random.default_rng(6)
    for n in sizes:
        print(f"[case] {shape} {settings} plans={n}", flush=True)
        pick = rng.integers(0, base.n_plans, n)
        batch = PlanBatch(base.codes[pick], base.hdr[pick])
        bad = [0, 1, 2, 3, n - 1, *range(64, 144)]
        batch.codes[0, 0] &= 0xEF               # no stage start in front
        batch.codes[1, 1:] |= 16                # a stage per op
        batch.hdr[2, 0] = 40                    # more stages than there may be
        batch.hdr[3, 0] |= 0xff00               # no such micro-batch size
        batch.codes[n - 1, 1:] |= 16
        some = rng.random(batch.codes[64:144].shape) < 0.03
        batch.codes[64:144] ^= np.where(some, rng.choice([8, 16], some.shape), 0).astype(np.uint8)     # stage and recompute bits
        got = [x.cpu().numpy() for x in ev.score(ev.upload(batch, validate=False))[:4]]
        good = np.ones(n, dtype=bool)
        good[bad] = False
        assert (got[3][good] == 0).all() and all(np.array_equal(g[good], x[pick][good]) for g, x in zip(got, want))
        for g, x in zip(got, emu_score(tables, PlanBatch(batch.codes[bad], batch.hdr[bad]))[:4]):
            assert np.array_equal(g[bad], x, equal_nan=True)
    ev.close()


@pytest.mark.gpu
@pytest.mark.parametrize("shape,sizes", [("conv, 4 of 1 differing", (8632, 8633, 65537, 270001)), ("conv, 4 of 4 differing", (8800, 8801, 262145)),
                                         ("conv, 8 of 1 differing", (15900, 15901, 131073)), ("gpt, 8 of 8 differing", (8801, 70001)), ("conv, 38 ops, 8 differing", (6825,))])
def test_tables_outside_the_dense_form_on_the_gpu(shape, sizes):
    outside_on_the_gpu(shape, sizes)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", ["conv, 4 of 1 differing", "conv, 4 of 4 differing", "conv, 8 of 1 differing"])
def test_every_variant_of_the_older_loops_on_the_gpu(shape):
    """One text each per resharding on or off and rule of the reserved memory, rows resident or in windows; the C++ loop likewise."""
    for resharding in (True, False):
        for pred, reserved in (("MAX", True), ("MIN", True), ("MAX", False)):
            outside_on_the_gpu(shape, (131149,), resharding=resharding, memory_pred_type=pred, consider_reserved_space=reserved)


@pytest.mark.gpu
def test_resident_rows_in_another_order_outside_the_dense_form_on_the_gpu():
    """... which no assembly loop walks."""
    outside_on_the_gpu("conv, 4 of 1 differing", (13400, 13401, 131073), order=True)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", ["conv, 4 of 1 differing", "conv, 4 of 4 differing", "conv, 8 of 1 differing", "conv, 1 of 2"])
def test_static_scratch_over_other_shapes_on_the_gpu(shape):
    import torch
    from superscaler_amd.evaluator import PlanEvaluator
    from tests.test_zz_no_alloc import _raw_scores
    w, tables = tables_of(shape)
    base = with_recompute(synth.make_plans(w, tables, n_plans=4000, seed_offset=35), 0.6, 35)
    want = c_oracle_scores(tables, base, threads=8)
    ev = PlanEvaluator(tables)
    for n in (16384, 8801):
        print(f"[case] {shape} plans={n}", flush=True)
        pick = np.random.default_rng(n).integers(0, base.n_plans, n)
        d = ev.upload(PlanBatch(base.codes[pick], base.hdr[pick]))
        for entry in ("static", "plain"):
            got = _raw_scores(ev, torch, entry, d, float(tables.settings.memory_limit))
            assert (got[3] == 0).all() and all(np.array_equal(g, x[pick]) for g, x in zip(got, want))
    ev.close()
