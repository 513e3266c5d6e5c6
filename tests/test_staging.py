"""Uploads through the caller's staging buffer: as many bytes as the plans have are enough, the plans go through it whatever their
size, and nothing waits for the device (checked or not)."""
import numpy as np
import pytest

from superscaler_amd import synth
from tests.helpers import kernel_layout


@pytest.mark.gpu
@pytest.mark.parametrize("n", [5, 4001, 100_003])           # less than a piece of the library's own staging; more than three of them
def test_staged_uploads_do_not_wait(n):
    import torch
    from superscaler_amd.evaluator import STAGING_PIECE, STAGING_SLOTS, DeviceBatch, PlanEvaluator
    w = synth.WORKLOADS["gpt3_13b"]
    tables = synth.make_tables(w)
    N = tables.graph.num_ops
    batch = synth.make_plans(w, tables, n_plans=n, seed_offset=n, workers=8)
    assert (n * N > STAGING_PIECE * STAGING_SLOTS) == (n == 100_003)
    ev = PlanEvaluator(tables)
    staging = torch.zeros(n * N, dtype=torch.uint8, pin_memory=True)
    DeviceBatch(batch, staging=staging)                      # (what is allocated once is allocated)
    for upload in (lambda: DeviceBatch(batch, staging=staging), lambda: ev.upload(batch, staging=staging)):
        staging.zero_()
        torch.cuda.synchronize()
        torch.cuda._sleep(1 << 28)                           # (cycles: a tenth of a second and more)
        done = torch.cuda.Event()
        done.record()
        d = upload()
        assert not done.query()
        torch.cuda.synchronize()
        assert np.array_equal(staging.numpy().reshape(n, N), batch.codes)
        assert np.array_equal(d.codes.cpu().numpy(), kernel_layout(batch.codes)) and np.array_equal(d.hdr.cpu().numpy().view(np.uint32), batch.hdr)
    with pytest.raises(RuntimeError):
        DeviceBatch(batch, staging=staging[:-1])
    bad = batch.slice(0, n)
    bad.codes = bad.codes.copy()
    bad.codes[n // 2, 0] &= 0xEF
    with pytest.raises(ValueError):
        ev.upload(bad, staging=staging)
    ev.close()
