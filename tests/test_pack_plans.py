"""Plans between the host's rows and the kernels' layout (superscaler_amd/csrc/ace_pack.h) and the structural check of a batch
that rides along: on the CPU behind guard pages in a child process (`python -m tests.test_pack_plans`), on the GPU through
upload() and download(), against numpy."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

from superscaler_amd import plan as plan_mod
from superscaler_amd import synth
from superscaler_amd.plan import PlanBatch, validate_batch
from tests.helpers import emu_lib, kernel_layout

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# ops: less than a group, a full one, one more; 64 groups and around them; several column tiles; plans: around tiles of 32
SHAPES = [(1, 1), (1, 15), (33, 16), (31, 17), (32, 134), (65, 523), (3, 1024), (34, 1025), (2, 1023), (40, 1251), (1, 4097)]


def batch_of(P, N, rng, n_mbs, C):
    """Plans whose structure is right: 1 to 16 stages, op 0 opens one, codes and micro-batch indices in range."""
    codes = (rng.integers(0, C, (P, N)) | (rng.integers(0, 2, (P, N)) << 3)).astype(np.uint8)
    hdr = rng.integers(0, 2 ** 32, (P, 4), dtype=np.uint64).astype(np.uint32)
    for p in range(P):
        S = int(rng.integers(1, min(N, 16) + 1))
        codes[p, np.append(0, rng.choice(np.arange(1, N), S - 1, replace=False)).astype(int)] |= 16
        hdr[p, 0] = S | int(rng.integers(0, n_mbs)) << 8
    return PlanBatch(codes, hdr)


def broken(batch, rng, n_mbs, C):
    """(what is wrong, batch) with one plan broken."""
    P, N = batch.codes.shape
    p = int(rng.integers(0, P))
    for k in range(5):
        b = PlanBatch(batch.codes.copy(), batch.hdr.copy())
        S = int(b.hdr[p, 0] & 0xff)
        if k == 0:
            b.hdr[p, 0] = (b.hdr[p, 0] & 0xff00) | rng.choice([0, 17, 200])
        elif k == 1:
            b.hdr[p, 0] = (b.hdr[p, 0] & 0xff00) | (S % 16 + 1)
        elif k == 2:
            if N < 2 or S == min(N, 16):
                continue
            b.codes[p, 0] &= 0xEF
            b.codes[p, np.flatnonzero((b.codes[p, 1:] & 16) == 0)[0] + 1] |= 16      # (as many as the header says)
        elif k == 3:
            b.hdr[p, 0] = S | n_mbs << 8
        else:
            if C == 8:
                continue
            i = int(rng.integers(0, N))
            b.codes[p, i] = (b.codes[p, i] & 0xF8) | C
        yield k, b


def main():
    lib, rng = emu_lib(), np.random.default_rng(4)
    vp = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    for P, N in SHAPES:
        for n_mbs, C in ((5, 8), (2, 4), (1, 3)):
            batch = batch_of(P, N, rng, n_mbs, C)
            for k, b in [(None, batch), *broken(batch, rng, n_mbs, C)]:
                codes, hdr = np.ascontiguousarray(b.codes), np.ascontiguousarray(b.hdr)
                out = np.empty(((N + 15) // 16, P, 16), dtype=np.uint8)
                found = lib.ace_emu_pack(vp(codes), vp(hdr), ctypes.c_longlong(P), N, n_mbs, C, vp(out))
                assert np.array_equal(out, kernel_layout(codes))
                assert found == 0 if k is None else plan_mod.finding(found) == plan_mod.FINDINGS[k], (P, N, k, found)
            back = np.empty_like(codes)
            assert lib.ace_emu_unpack(vp(out), ctypes.c_longlong(P), N, vp(back)) == 0 and np.array_equal(back, codes)


def test_phases_on_the_cpu():
    emu_lib()
    proc = subprocess.run([sys.executable, "-m", "tests.test_pack_plans"], cwd=ROOT, stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                          text=True, timeout=600)
    assert proc.returncode == 0, f"child ended with {proc.returncode} (negative: killed by that signal)\n{proc.stdout[-2000:]}"


class Stub:
    """What validate_batch reads of the tables."""

    def __init__(self, N, n_mbs, C):
        import types
        self.graph, self.db, self.C = types.SimpleNamespace(num_ops=N), types.SimpleNamespace(mbs_list=[0] * n_mbs), C


def test_the_host_check_names_what_is_wrong():
    rng = np.random.default_rng(6)
    for P, N in SHAPES + [(2, 5000)]:
        for n_mbs, C in ((5, 8), (2, 4), (1, 3)):
            batch = batch_of(P, N, rng, n_mbs, C)
            assert validate_batch(batch, Stub(N, n_mbs, C)) is None
            for k, b in broken(batch, rng, n_mbs, C):
                assert validate_batch(b, Stub(N, n_mbs, C)) == plan_mod.FINDINGS[k]
    assert "ops per plan" in validate_batch(batch, Stub(N + 1, n_mbs, C))
    assert validate_batch(batch.slice(0, 0), Stub(N, n_mbs, C)) == "empty batch"


@pytest.mark.gpu
@pytest.mark.parametrize("name,n", [("gpt3_13b", 4001), ("wresnet_1b", 33), ("t5_770m", 1000)])
def test_upload_and_download_on_the_gpu(name, n):
    from superscaler_amd.evaluator import PlanEvaluator
    w = synth.WORKLOADS[name]
    tables = synth.make_tables(w)
    ev = PlanEvaluator(tables)
    rng = np.random.default_rng(n)
    batch = synth.make_plans(w, tables, n_plans=n, seed_offset=n)
    pinned = ev.pinned_plan_batch(n)
    pinned.codes[...], pinned.hdr[...] = batch.codes, batch.hdr
    ev.HOST_CHECK_BYTES = 0                     # the check of the packing kernel, whatever the size
    for b in (batch, pinned):
        d = ev.upload(b)
        assert np.array_equal(d.codes.cpu().numpy(), kernel_layout(batch.codes))
        for limit in (0, ev.PINNED_RESULT_BYTES):
            ev.PINNED_RESULT_BYTES = limit
            back = ev.download(d)
            assert np.array_equal(back.codes, batch.codes) and np.array_equal(back.hdr, batch.hdr)
    for k, b in broken(batch, rng, len(tables.db.mbs_list), tables.C):
        with pytest.raises(ValueError, match=plan_mod.FINDINGS[k].split()[0]):
            ev.upload(b)
    ev.close()


if __name__ == "__main__":
    main()
