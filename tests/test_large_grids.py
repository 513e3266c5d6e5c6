"""Batches whose grids have 2^32 work items and more: kernels with many lanes per plan are launched in parts."""
import ctypes

import numpy as np
import pytest

from tests.helpers import emu_lib


@pytest.mark.parametrize("lanes", [32, 256, 1024])
def test_parts_cover_the_grid_and_can_be_launched(lanes):
    lib = emu_lib()
    most = 2 ** 31 // lanes
    for groups in (1, most - 1, most, most + 1, 2 * most, 2 ** 24, 2 ** 24 + 5, 2 ** 26, 2 ** 31 - 1):
        out = np.zeros((1024, 2), dtype=np.uint64)
        n = lib.ace_emu_grid_parts(ctypes.c_ulonglong(groups), ctypes.c_uint(lanes), out.ctypes.data_as(ctypes.c_void_p), 1024)
        parts = out[:n].astype(object)
        assert n == -(-groups // most) <= 1024
        assert parts[0][0] == 0 and all(a + b == c for (a, b), (c, _) in zip(parts, parts[1:])) and sum(parts[-1]) == groups
        assert all(0 < count * lanes < 2 ** 32 for _, count in parts)


@pytest.mark.gpu
def test_recompute_for_sixteen_million_plans():
    """A workgroup of 256 lanes per plan: 2^24 plans have 2^32 work items."""
    import torch
    from superscaler_amd import opgraph as og
    from superscaler_amd import synth
    from superscaler_amd.evaluator import DeviceBatch, PlanEvaluator, _check
    from tests.test_recompute_kernel import cost_model
    from tests.test_small_batches import WORKLOADS
    w = WORKLOADS["gpt_16ops"]
    cm = cost_model(w, emu=False)
    ev = PlanEvaluator(cm.tables)
    t = cm.tables
    assert ev.prepare_recompute(((np.asarray(t.graph.flags)[:len(t.db.op_names)] & og.F_NO_RECOMPUTE) != 0).astype(np.uint8))
    small, tiles = 4096, 4097
    assert small * tiles > 2 ** 24
    d = ev.upload(synth.make_plans(w, t, n_plans=small, seed_offset=1))
    limit = float(ev.score(d)[1].median().item())
    want, status, flags = ev.recompute(d, limit, 0.0)
    assert flags.tolist() == [0, 0, 0, 0] and not torch.equal(want.codes & 8, want.codes & 0)
    G = d.codes.shape[0]
    big = DeviceBatch.from_device(d.codes.repeat(1, tiles, 1), d.hdr.repeat(tiles, 1), d.num_ops)
    out, flags = torch.zeros_like(big.codes), torch.zeros(4, dtype=torch.int32, device="cuda")
    _check(ev.lib, ev.lib.ace_recompute_batch(ev.handle, ctypes.byref(big.struct), limit, 0.0, status.repeat(tiles).data_ptr(), out.data_ptr(),
                                              flags.data_ptr(), ev._stream()), "ace_recompute_batch")
    torch.cuda.synchronize()
    assert flags.tolist() == [0, 0, 0, 0]
    same = bool((out.view(G, tiles, small, 16) == want.codes.view(G, 1, small, 16)).all())
    assert same
    ev.close()


@pytest.mark.gpu
def test_half_a_billion_plans_change_layout():
    """A workgroup of 256 lanes per 32 plans: 2^29 plans have 2^32 work items."""
    import torch
    from superscaler_amd.evaluator import _check, load_library, pack_rows
    P, N = 2 ** 29 + 37, 3
    rows = (torch.arange(P * N, dtype=torch.int32, device="cuda") % 251).to(torch.uint8).view(P, N)
    codes = pack_rows(rows, None)
    same, padded = bool((codes[0, :, :N] == rows).all()), not bool(codes[0, :, N:].any())
    assert same and padded
    back = torch.zeros_like(rows)
    lib = load_library()
    _check(lib, lib.ace_unpack_plans(codes.data_ptr(), P, N, back.data_ptr(), None), "ace_unpack_plans")
    torch.cuda.synchronize()
    same = torch.equal(back, rows)
    assert same
