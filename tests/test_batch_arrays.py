"""What a host batch's arrays may look like where native code reads them: other integer types and layouts are converted, one
header row stands for all plans, and arrays that are too short (or too long) are refused before anything reads them."""
import contextlib
import ctypes
import types

import numpy as np
import pytest

from superscaler_amd import plan as plan_mod
from superscaler_amd import synth
from superscaler_amd.evaluator import PlanEvaluator, load_library, pack_small_inputs, rows_to_device
from superscaler_amd.neighbours import _draw_moves, _draws_struct, sample_moves
from superscaler_amd.plan import PlanBatch, validate_batch
from tests.helpers import odd_workloads

W = odd_workloads()[2]
TYPES = [np.uint8, np.int8, np.int32, np.int64, np.uint64, ">i4"]


def tables_and_plans(n):
    tables = synth.make_tables(W)
    return tables, synth.make_plans(W, tables, n_plans=n, seed_offset=3)


def forms(batch):
    """The same plans in other integer types and memory layouts."""
    for t in TYPES:
        yield PlanBatch(batch.codes.astype(t), batch.hdr.astype(np.int64 if t != np.uint64 else np.uint64))
    yield PlanBatch(np.asfortranarray(batch.codes), np.asfortranarray(batch.hdr))
    yield PlanBatch(np.repeat(batch.codes, 2, axis=1)[:, ::2], np.repeat(batch.hdr, 2, axis=0)[::2])


def at(pointer, like):
    """What stands at `pointer`, as an array like `like`."""
    return np.frombuffer(ctypes.string_at(pointer, like.nbytes), dtype=like.dtype).reshape(like.shape)


def test_moves_are_drawn_from_the_plans_values():
    tables, batch = tables_and_plans(4)
    for p in range(4):
        base = batch.slice(p, p + 1)
        want = sample_moves(base, tables, 400, np.random.default_rng(p))
        for b in forms(base):
            templates, moves = sample_moves(b, tables, 400, np.random.default_rng(p))
            assert np.array_equal(moves, want[1]) and np.array_equal(templates.codes, want[0].codes) and np.array_equal(templates.hdr, want[0].hdr)
    N = tables.graph.num_ops
    for bad in (PlanBatch(base.codes[:, :N - 1], base.hdr), PlanBatch(base.codes, base.hdr[:, :3])):
        with pytest.raises(ValueError):
            sample_moves(bad, tables, 400, np.random.default_rng(0))
    with pytest.raises(TypeError):
        sample_moves(PlanBatch(base.codes.astype(float), base.hdr), tables, 400, np.random.default_rng(0))


def test_a_search_step_reads_the_plans_values():
    tables, batch = tables_and_plans(1)
    seen = []

    def ace_search_step(handle, row, hdr, *_):
        seen.append((at(row, batch.codes[0]), at(hdr, batch.hdr[0])))
        return 0
    ev = types.SimpleNamespace(tables=tables, lib=types.SimpleNamespace(ace_search_step=ace_search_step), handle=None, _stream=lambda: None)
    draws = _draws_struct(_draw_moves(10, int(batch.hdr[0, 0] & 0xff), tables, np.random.default_rng(0)))
    for b in forms(batch):
        PlanEvaluator.search_step(ev, b, draws)
        assert np.array_equal(seen[-1][0], batch.codes[0]) and np.array_equal(seen[-1][1], batch.hdr[0])
    with pytest.raises(ValueError):
        PlanEvaluator.search_step(ev, PlanBatch(batch.codes[:, :-1], batch.hdr), draws)


def test_the_structural_check_wants_a_header_per_plan():
    tables, batch = tables_and_plans(8)
    for b in forms(batch):
        assert validate_batch(b, tables) is None
    for rows in (0, 4, 7, 9):
        with pytest.raises(ValueError):
            validate_batch(PlanBatch(batch.codes, np.resize(batch.hdr, (rows, 4))), tables)
    for bad in (batch.hdr[:, :3], batch.hdr[:, 0], np.repeat(batch.hdr, 2, axis=1)):
        with pytest.raises(ValueError):
            validate_batch(PlanBatch(batch.codes, bad), tables)
    with pytest.raises(TypeError):
        validate_batch(PlanBatch(batch.codes.astype(float), batch.hdr), tables)
    # one header for all of them: checked against every plan's stage starts
    same = PlanBatch(np.repeat(batch.codes[:1], 8, axis=0), batch.hdr[:1])
    assert validate_batch(same, tables) is None
    same.codes[5, 1:] |= 16
    assert validate_batch(same, tables) == plan_mod.FINDINGS[1]


def fake_evaluator(tables, calls):
    """A PlanEvaluator whose library only records what it is handed."""
    import torch
    ev = PlanEvaluator.__new__(PlanEvaluator)
    ev._plan_bytes = 16 * ((tables.graph.num_ops + 15) // 16)
    ev.tables, ev.device, ev.handle, ev._torch = tables, torch.device("cuda", 0), None, types.SimpleNamespace(
        _C=types.SimpleNamespace(_cuda_getCurrentRawStream=lambda device: device))

    def ace_score_host(handle, codes, hdr, ranges, P, *_):
        shape = (P, tables.graph.num_ops)
        calls.append((at(codes, np.empty(shape, np.uint8)), at(hdr, np.empty((P, 4), np.uint32)),
                      None if ranges is None else at(ranges, np.empty((P, 2), np.uint32)), _[-1]))
        return 0
    ev.lib = types.SimpleNamespace(ace_score_host=ace_score_host, ace_check_plans=load_library().ace_check_plans)
    return ev


def test_scores_are_asked_for_the_plans_values():
    import torch
    tables, batch = tables_and_plans(8)
    P, N = batch.codes.shape
    calls = []
    ev = fake_evaluator(tables, calls)
    ranges = np.tile(np.array([[0, N]], dtype=np.uint32), (P, 1))
    want = np.zeros(1 << 16, dtype=np.uint8)
    used = pack_small_inputs(want, batch, ranges)
    one = PlanBatch(np.repeat(batch.codes[:1], P, axis=0), batch.hdr[:1])
    for b in [*forms(batch), one]:
        ref = batch if b is not one else PlanBatch(one.codes, np.repeat(one.hdr, P, axis=0))
        for rg in (None, ranges):
            ev.score_host(b, ranges=rg)
            codes, hdr = calls[-1][:2]
            assert np.array_equal(codes, ref.codes) and np.array_equal(hdr, ref.hdr)
        rows, hdr = rows_to_device(b, "cpu")
        assert rows.dtype == torch.uint8 and np.array_equal(rows.numpy(), ref.codes) and np.array_equal(hdr.numpy().view(np.uint32), ref.hdr)
        if b is not one:
            got = np.zeros_like(want)
            assert pack_small_inputs(got, b, ranges) == used and np.array_equal(got, want)
    for bad in (PlanBatch(batch.codes, batch.hdr[:4]), PlanBatch(batch.codes, batch.hdr[:, :3])):
        for call in (lambda: ev.score_host(bad), lambda: ev.score_host(bad, ranges=ranges), lambda: rows_to_device(bad, "cpu"),
                     lambda: pack_small_inputs(np.zeros_like(want), bad, None)):
            with pytest.raises(ValueError):
                call()


def test_ranges_stand_for_every_query():
    tables, batch = tables_and_plans(8)
    P, N = batch.codes.shape
    calls = []
    ev = fake_evaluator(tables, calls)
    per_query = np.stack([np.arange(P), np.arange(P) + 2], axis=1)
    for rg, want in ((per_query, per_query), (per_query.astype(np.uint32), per_query), (np.asfortranarray(per_query), per_query),
                     (per_query.tolist(), per_query), ((3, 5), np.tile([[3, 5]], (P, 1))), (np.array([[3, 5]]), np.tile([[3, 5]], (P, 1)))):
        ev.score_host(batch, ranges=rg)
        assert np.array_equal(calls[-1][2], want)
        buf = np.zeros(1 << 16, dtype=np.uint8)
        used = pack_small_inputs(buf, batch, rg)
        assert np.array_equal(buf[used - 8 * P:used].view(np.uint32).reshape(P, 2), want)
    for buf in (np.zeros(1 << 16, dtype=np.int8), np.zeros(1 << 17, dtype=np.uint8)[::2], np.frombuffer(bytes(1 << 16), dtype=np.uint8)):
        with pytest.raises(ValueError):
            pack_small_inputs(buf, batch, per_query)
    made = len(calls)
    for rg in (per_query[:4], per_query[:0], np.zeros((P, 3)), np.zeros(P), np.zeros((P, 1, 2))):
        with pytest.raises(ValueError):
            ev.score_host(batch, ranges=rg)
        with pytest.raises(ValueError):
            pack_small_inputs(np.zeros(1 << 16, dtype=np.uint8), batch, rg)
    assert len(calls) == made


def test_plans_without_ops_have_no_code_words():
    buf = np.full(4096, 7, dtype=np.uint8)
    b = PlanBatch(np.zeros((3, 0), dtype=np.uint8), np.arange(12, dtype=np.uint32).reshape(3, 4))
    assert pack_small_inputs(buf[1024:], b, None) == 48
    assert np.array_equal(buf[1024:1072].view(np.uint32), np.arange(12)) and (buf[:1024] == 7).all() and (buf[1072:] == 7).all()


def test_queries_have_the_graphs_ops():
    tables, batch = tables_and_plans(8)
    calls = []
    ev = fake_evaluator(tables, calls)
    ranges = np.tile([[0, 1]], (8, 1))
    for bad in (PlanBatch(batch.codes[:, :-1], batch.hdr), PlanBatch(np.repeat(batch.codes, 2, axis=1), batch.hdr)):
        for kw in ({}, {"ranges": ranges}, {"ranges": ranges, "group_by_depth": True}):
            with pytest.raises(ValueError, match="ops per plan"):
                ev.score_host(bad, **kw)
        with pytest.raises(ValueError, match="ops per plan"):
            ev.upload(bad, ranges=ranges)
    assert not calls


def test_a_device_without_an_index_is_the_one_that_was_current(monkeypatch):
    """The library's handle lives on that one: its stream is the one a call must be ordered on, whatever is current later."""
    import torch
    from superscaler_amd import evaluator
    tables, batch = tables_and_plans(2)
    calls = []
    made = fake_evaluator(tables, calls).lib
    made.ace_create = lambda tables, handle: 0
    current = [3]
    monkeypatch.setattr(evaluator, "load_library", lambda: made)
    monkeypatch.setattr(torch.cuda, "is_available", lambda: True)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: current[0])
    monkeypatch.setattr(torch.cuda, "device", lambda d: contextlib.nullcontext())
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda index: 1000 + index, raising=False)
    ev = {d: PlanEvaluator(tables, d) for d in ("cuda", "cuda:1", 2, torch.device("cuda"))}
    current[0] = 0
    for d, index in (("cuda", 3), ("cuda:1", 1), (2, 2), (torch.device("cuda"), 3)):
        assert ev[d].device == torch.device("cuda", index)
        ev[d].score_host(batch)
        assert calls[-1][3] == 1000 + index


def test_device_batches_hold_the_graphs_ops():
    """A batch that was not checked when it was made (from_device, upload(validate=False)): fewer 16-op groups than the graph has
    would be read past their end."""
    import torch
    from superscaler_amd.evaluator import DeviceBatch
    from superscaler_amd.neighbours import _draw_moves, _draws_struct
    tables, batch = tables_and_plans(4)
    calls = []
    ev = fake_evaluator(tables, calls)
    P, N = batch.codes.shape
    assert 16 < N < 32
    hdr = torch.from_numpy(batch.hdr.view(np.int32))
    small = DeviceBatch.from_device(torch.zeros((1, P, 16), dtype=torch.uint8), hdr, 16)
    short = DeviceBatch.from_device(torch.zeros((2, P - 1, 16), dtype=torch.uint8), hdr, N)
    for d in (small, short):
        for call in (lambda: ev.score(d), lambda: ev.time_score_kernel(d, 1), lambda: ev.recompute(d, 1e4, 0.0)):
            with pytest.raises(ValueError, match="16-op groups"):
                call()
    # op positions of a search's moves have 16 bits
    ev.tables = types.SimpleNamespace(graph=types.SimpleNamespace(num_ops=65536), settings=tables.settings, stage_lut=tables.stage_lut)
    with pytest.raises(ValueError, match="16-bit"):
        ev.search_step(PlanBatch(np.zeros((1, 65536), dtype=np.uint8), batch.hdr[:1]),
                       _draws_struct(_draw_moves(1, 1, tables, np.random.default_rng(0))))


def test_queries_of_other_types_are_converted():
    tables, batch = tables_and_plans(8)
    calls = []
    ev = fake_evaluator(tables, calls)
    ev.score_host(PlanBatch(batch.codes.astype(float), batch.hdr.astype(float)), ranges=(0, 3))
    assert np.array_equal(calls[-1][0], batch.codes) and np.array_equal(calls[-1][1], batch.hdr)
    with pytest.raises(TypeError):
        ev.score_host(PlanBatch(batch.codes.astype(float), batch.hdr))


@pytest.mark.gpu
def test_empty_batches_and_other_integers_on_the_gpu():
    import torch
    tables, batch = tables_and_plans(8)
    ev = PlanEvaluator(tables)
    empty = ev.upload(batch.slice(0, 0), validate=False)
    assert empty.n_plans == 0 and empty.codes.shape == (2, 0, 16) and empty.hdr.shape == (0, 4)
    with pytest.raises(ValueError):
        ev.upload(batch.slice(0, 0))
    d = ev.upload(batch)
    none = ev.download(d, torch.zeros(0, dtype=torch.int64, device="cuda"))
    assert none.codes.shape == (0, tables.graph.num_ops) and none.hdr.shape == (0, 4) and none.hdr.dtype == np.uint32
    want = ev.top_k(batch, 3)
    for k in (np.int64(3), np.uint8(3)):
        got = ev.top_k(batch, k)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
        assert ev.score_stream([batch], k)[0].tolist() == want[0].tolist()
    with pytest.raises(TypeError):
        ev.top_k(batch, 3.0)
    ev.close()
