"""ctypes binding of libace_eval.so and the torch-side plumbing (device buffers, streams).

`PlanEvaluator` owns one ace_handle_t (tables resident on the device).  It never computes a
score itself: if the HIP library is missing or no GPU is present it raises.
"""
import ctypes
import operator
import os
import threading
from typing import Optional

import numpy as np

from .plan import PlanBatch, check_plans, check_shape, finding, host_arrays, validate_batch
from .tables import ABI_VERSION, MAX_STAGES, STAGE_REC, AceTablesStruct, CompiledTables

_LIB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "libace_eval.so")
_lib = None

EXPORTS = ["ace_abi_version", "ace_strerror", "ace_last_hip_error", "ace_create", "ace_destroy",
           "ace_score_batch", "ace_score_batch_static", "ace_reserve", "ace_topk_workspace_bytes", "ace_topk", "ace_time_score_kernel", "ace_apply_moves",
           "ace_recompute_groups", "ace_recompute_select", "ace_group_keys", "ace_gather_plans",
           "ace_keyset_create", "ace_keyset_destroy", "ace_keyset_size", "ace_keyset_add", "ace_keyset_unseen", "ace_keyset_claim",
           "ace_keyset_move", "ace_keyset_keys", "ace_build_moves", "ace_new_moves", "ace_search_step", "ace_recompute_prepare", "ace_recompute_batch",
           "ace_pack_plans", "ace_unpack_plans", "ace_check_plans", "ace_score_host", "ace_pack_host"]


class AceBatchStruct(ctypes.Structure):
    _fields_ = [("d_codes", ctypes.c_void_p), ("d_hdr", ctypes.c_void_p), ("d_range", ctypes.c_void_p),
                ("n_plans", ctypes.c_size_t), ("d_order", ctypes.c_void_p)]


class AceRcTablesStruct(ctypes.Structure):
    _fields_ = [("d_codes", ctypes.c_void_p), ("n_plans", ctypes.c_size_t), ("d_type_of_pos", ctypes.c_void_p),
                ("d_activations", ctypes.c_void_p), ("d_no_recompute", ctypes.c_void_p), ("num_ops", ctypes.c_int32),
                ("num_types", ctypes.c_int32), ("n_mbs", ctypes.c_int32), ("n_tp", ctypes.c_int32), ("n_algo", ctypes.c_int32)]


class AceMoveDrawsStruct(ctypes.Structure):
    _fields_ = [("n", ctypes.c_size_t), ("count", ctypes.c_size_t * 6), ("rows", ctypes.c_void_p * 6),
                ("x", ctypes.c_void_p * 6), ("y", ctypes.c_void_p * 6)]


class AceStepResultStruct(ctypes.Structure):
    _fields_ = [("n_moves", ctypes.c_size_t), ("found", ctypes.c_int32), ("iter_ms", ctypes.c_double), ("peak_mb", ctypes.c_double)]


ACE_ETOOBIG = -2


class AceError(RuntimeError):
    pass


def load_library():
    """dlopen the in-tree HIP library; no fallback of any kind."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(_LIB_PATH):
        raise AceError(f"{_LIB_PATH} is missing: build it with `python -m superscaler_amd.build` "
                       "(there is no CPU fallback for plan scoring)")
    import torch  # noqa: F401  (its HIP runtime has to be the one the library binds to, also where the first call is a host one)
    lib = ctypes.CDLL(_LIB_PATH)
    lib.ace_abi_version.restype = ctypes.c_int
    lib.ace_strerror.restype = ctypes.c_char_p
    lib.ace_strerror.argtypes = [ctypes.c_int]
    lib.ace_last_hip_error.restype = ctypes.c_char_p
    lib.ace_create.restype = ctypes.c_int
    lib.ace_create.argtypes = [ctypes.POINTER(AceTablesStruct), ctypes.POINTER(ctypes.c_void_p)]
    lib.ace_destroy.restype = None
    lib.ace_destroy.argtypes = [ctypes.c_void_p]
    lib.ace_score_batch.restype = ctypes.c_int
    lib.ace_score_batch.argtypes = [ctypes.c_void_p, ctypes.POINTER(AceBatchStruct), ctypes.c_double, ctypes.c_int,
                                    ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p,
                                    ctypes.c_void_p, ctypes.c_void_p]
    lib.ace_score_batch_static.restype = ctypes.c_int
    lib.ace_score_batch_static.argtypes = [ctypes.c_void_p, ctypes.POINTER(AceBatchStruct), ctypes.c_double, ctypes.c_int,
                                           ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p]
    lib.ace_reserve.restype = ctypes.c_int
    lib.ace_reserve.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
    lib.ace_topk_workspace_bytes.restype = ctypes.c_size_t
    lib.ace_topk_workspace_bytes.argtypes = [ctypes.c_size_t, ctypes.c_int]
    lib.ace_topk.restype = ctypes.c_int
    lib.ace_topk.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int,
                             ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t,
                             ctypes.c_void_p]
    lib.ace_time_score_kernel.restype = ctypes.c_int
    lib.ace_time_score_kernel.argtypes = [ctypes.c_void_p, ctypes.POINTER(AceBatchStruct), ctypes.c_double,
                                          ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p,
                                          ctypes.c_int, ctypes.c_void_p, ctypes.POINTER(ctypes.c_double)]
    lib.ace_apply_moves.restype = ctypes.c_int
    lib.ace_apply_moves.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p, ctypes.c_size_t,
                                    ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p]
    lib.ace_group_keys.restype = ctypes.c_int
    lib.ace_group_keys.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p]
    lib.ace_gather_plans.restype = ctypes.c_int
    lib.ace_gather_plans.argtypes = [ctypes.c_void_p] * 3 + [ctypes.c_size_t, ctypes.c_int] + [ctypes.c_void_p] * 3
    lib.ace_recompute_groups.restype = ctypes.c_int
    lib.ace_recompute_groups.argtypes = [ctypes.POINTER(AceRcTablesStruct), ctypes.c_int] + [ctypes.c_void_p] * 9
    lib.ace_recompute_select.restype = ctypes.c_int
    lib.ace_recompute_select.argtypes = ([ctypes.POINTER(AceRcTablesStruct), ctypes.c_void_p, ctypes.c_int] +
                                         [ctypes.c_void_p] * 9 + [ctypes.c_double, ctypes.c_void_p, ctypes.c_void_p])
    vp, sz = ctypes.c_void_p, ctypes.c_size_t
    lib.ace_keyset_create.argtypes = [ctypes.POINTER(vp)]
    lib.ace_keyset_destroy.restype = None
    lib.ace_keyset_destroy.argtypes = [vp]
    lib.ace_keyset_size.restype = sz
    lib.ace_keyset_size.argtypes = [vp]
    lib.ace_keyset_add.argtypes = [vp, vp, sz]
    lib.ace_keyset_unseen.argtypes = [ctypes.POINTER(vp), ctypes.c_int, vp, sz, vp]
    lib.ace_keyset_claim.argtypes = [ctypes.POINTER(vp), ctypes.c_int, vp, sz, vp]
    lib.ace_keyset_move.argtypes = [vp, vp]
    lib.ace_keyset_keys.argtypes = [vp, vp]
    lib.ace_pack_plans.argtypes = [vp, sz, ctypes.c_int, vp, ctypes.c_int, ctypes.c_int, vp, vp, vp]
    lib.ace_unpack_plans.argtypes = [vp, sz, ctypes.c_int, vp, vp]
    lib.ace_check_plans.argtypes = [vp, vp, sz, ctypes.c_int, ctypes.c_int, ctypes.c_int]
    lib.ace_score_host.argtypes = [vp, vp, vp, vp, sz, ctypes.c_double, ctypes.c_int, vp, vp, vp, vp]
    lib.ace_pack_host.restype = sz
    lib.ace_pack_host.argtypes = [vp, vp, vp, sz, ctypes.c_int, vp]
    lib.ace_recompute_prepare.argtypes = [vp] * 4
    lib.ace_recompute_batch.argtypes = [vp, ctypes.POINTER(AceBatchStruct), ctypes.c_double, ctypes.c_double] + [vp] * 4
    ci = ctypes.c_int
    lib.ace_search_step.argtypes = [vp, vp, vp, vp, ci, ctypes.POINTER(AceMoveDrawsStruct), ctypes.POINTER(vp), ci, ctypes.c_double, ci, vp, vp,
                                    ctypes.POINTER(AceStepResultStruct), vp]
    lib.ace_new_moves.argtypes = [vp, vp, ci, ci, ci, ci, vp, ci, ctypes.POINTER(AceMoveDrawsStruct), ctypes.POINTER(vp), ci, vp, ctypes.POINTER(sz),
                                  vp, vp, ci, ctypes.POINTER(ci)]
    lib.ace_build_moves.argtypes = [vp, vp, ci, ci, ci, ci, vp, ci, ctypes.POINTER(AceMoveDrawsStruct), vp, vp, vp, ci, ctypes.POINTER(ci)]
    if lib.ace_abi_version() != ABI_VERSION:
        raise AceError("libace_eval.so has a different ABI version")
    _lib = lib
    return lib


_objects = None


def load_objects():
    """The native module that walks plan objects (csrc/ace_objects.cpp)."""
    global _objects
    if _objects is None:
        try:
            from . import _ace_objects
        except ImportError as e:
            raise AceError(f"superscaler_amd/_ace_objects.so cannot be loaded ({e}): build it with `python -m superscaler_amd.build`") from e
        _objects = _ace_objects
    return _objects


def _check(lib, rc, what):
    if rc != 0:
        msg = lib.ace_strerror(rc).decode()
        hip = lib.ace_last_hip_error().decode()
        raise AceError(f"{what}: {msg}" + (f" ({hip})" if hip and rc == -3 else ""))


WAVE = 64            # lanes of a wavefront
WAVES_PER_GROUP = 16  # wavefronts of the scoring kernel's large workgroup
_SNAKE = np.array([0, 1, 2, 3, 7, 6, 5, 4, 8, 9, 10, 11, 15, 14, 13, 12])


def deal_slots(n_plans: int) -> np.ndarray:
    """For a batch sorted from deep to shallow: which sorted position goes into each storage slot.
    The sorted plans are cut into wavefronts of 64 and the wavefronts are dealt round-robin to the
    workgroups of 16, so that every workgroup (every CU) gets the same mix of deep and shallow
    wavefronts; inside a workgroup they are laid out boustrophedon, because wavefront w runs on SIMD
    w % 4 and the four SIMDs should get equal shares too.  The last n_plans % 64 plans keep their place."""
    full = n_plans // WAVE
    groups = (full + WAVES_PER_GROUP - 1) // WAVES_PER_GROUP
    chunk = np.arange(full)
    if groups > 1:
        dealt = []
        for b in range(groups):
            mine = chunk[b::groups]                       # deepest ... shallowest wavefront of this workgroup
            dealt.append(mine[_SNAKE] if len(mine) == WAVES_PER_GROUP else mine)
        chunk = np.concatenate(dealt)
    slots = (chunk[:, None] * WAVE + np.arange(WAVE)[None, :]).reshape(-1)
    return np.concatenate([slots, np.arange(full * WAVE, n_plans)])


def depth_order(batch: PlanBatch) -> np.ndarray:
    """Storage order for a batch: perm[i] = the caller's index of the plan stored in slot i.  The plans
    are sorted (stably) by pipeline depth, deepest first, and by the positions of their first two
    stage boundaries, so that plans that close their stages at the same ops share a wavefront; the
    wavefronts are then dealt to the workgroups (deal_slots)."""
    S = (batch.hdr[:, 0] & 0xff).astype(np.int64)
    P, N = batch.codes.shape
    if N < 2:
        perm = np.argsort(-S, kind="stable")
    else:
        cuts = (batch.codes[:, 1:] & 16) != 0
        c1 = cuts.argmax(axis=1) + 1
        c1[~cuts.any(axis=1)] = 0
        cuts[np.arange(P), c1 - 1] &= (c1 == 0)
        c2 = cuts.argmax(axis=1) + 1
        c2[~cuts.any(axis=1)] = 0
        perm = np.lexsort((c2, c1, -S))
    return perm[deal_slots(P)]


_U32 = np.dtype(np.uint32)


def _address(a: np.ndarray) -> int:
    """Address of an array made here (writable, contiguous): a quarter of the time that numpy's ctypes view takes."""
    return ctypes.addressof(ctypes.c_char.from_buffer(a)) if a.size else a.ctypes.data


def host_ranges(ranges, n_plans: int) -> np.ndarray:
    """The op ranges of single-stage queries as native code reads them: uint32 [n_plans, 2], contiguous; one range stands for all
    queries, other shapes are refused (ValueError)."""
    r = np.ascontiguousarray(ranges, _U32)
    if r.shape != (n_plans, 2):
        r, one = np.empty((n_plans, 2), dtype=_U32), r
        r[...] = one
    return r


def pack_small_inputs(buf: np.ndarray, batch: PlanBatch, ranges) -> int:
    """Lay a small batch out for the kernel in `buf` (uint8) as ace_score_host does: codes [ceil(N/16)][P][16] (zero padded),
    then the headers uint32 [P][4], then the ranges uint32 [P][2] if given.  Returns the number of bytes used."""
    codes, hdr = host_arrays(batch.codes, batch.hdr, integers=False)
    P, N = codes.shape
    rg = None if ranges is None else host_ranges(ranges, P)
    if buf.dtype != np.uint8 or not (buf.flags.c_contiguous and buf.flags.writeable):
        raise ValueError("a contiguous uint8 buffer expected")
    args = (codes.ctypes.data, hdr.ctypes.data, None if rg is None else rg.ctypes.data, P, N)
    lib = load_library()
    if lib.ace_pack_host(*args, None) > buf.nbytes:
        raise ValueError("the buffer is too small")
    return lib.ace_pack_host(*args, buf.ctypes.data)


# Ordinary host memory goes to the device through page-locked pieces: the copy into one, by the host's threads, runs beside the
# transfer of the one before.  Three batches of 200,003 plans of 523 ops: 8.4 -> 6.7 ms (5.5 ms is the bus), 8.8 MB 280 -> 200 us,
# 1.6 MB 104 -> 57 us, where copies straight from ordinary memory reach 29 GB/s.  A piece costs some 50 us of calls and of waking
# the threads (pieces of 4 MB: 7.5 ms); three of them are in use at most, whatever the size of the batch, and they come from and
# go back to torch's cache of page-locked memory.
STAGING_PIECE = 16 << 20
STAGING_SLOTS = 3


def rows_to_device(batch: PlanBatch, device, staging=None):
    """The code rows (uint8 [P, N]) and headers (int32 [P, 4]) of a host batch on the device, in the host's layout.  Plans in
    page-locked memory (PlanEvaluator.pinned_plan_batch) are read where they are, by copies that may still be under way;
    others are staged in page-locked memory and may be rewritten after the call (`staging`: the memory to use, see DeviceBatch)."""
    import torch
    pinned = getattr(batch, "pinned_tensors", None)
    if pinned is not None:
        return pinned[0].to(device, non_blocking=True), pinned[1].to(device, non_blocking=True)
    codes, hdr = host_arrays(batch.codes, batch.hdr)
    host_rows, host_hdr = torch.from_numpy(codes).view(-1), torch.from_numpy(hdr.view(np.uint8)).view(-1)
    P, N = codes.shape
    if torch.device(device).type != "cuda":
        return host_rows.view(P, N).to(device), host_hdr.view(torch.int32).view(P, 4).to(device)
    head, size = host_hdr.numel(), host_rows.numel()
    if staging is not None:
        # (the caller's buffer, whatever its size: nothing waits for the device)
        stage, stage_hdr = staging[:size].view(P, N), torch.empty((P, 4), dtype=torch.int32, pin_memory=True)
        stage.copy_(host_rows.view(P, N))
        stage_hdr.copy_(host_hdr.view(torch.int32).view(P, 4))
        return stage.to(device, non_blocking=True), stage_hdr.to(device, non_blocking=True)
    if head + size <= STAGING_PIECE:
        # (one transfer for both)
        stage = torch.empty(head + size, dtype=torch.uint8, pin_memory=True)
        stage[:head].copy_(host_hdr)
        stage[head:].copy_(host_rows)
        both = stage.to(device, non_blocking=True)
        return both[head:].view(P, N), both[:head].view(torch.int32).view(P, 4)
    stream = torch.cuda.current_stream(device)
    slots = []                       # (page-locked piece, when its last transfer has ended)

    def send(to, data):
        for lo in range(0, data.numel(), STAGING_PIECE):
            part = data[lo:lo + STAGING_PIECE]
            if len(slots) < STAGING_SLOTS:
                piece, sent = torch.empty(STAGING_PIECE, dtype=torch.uint8, pin_memory=True), torch.cuda.Event()
            else:
                piece, sent = slots.pop(0)
                sent.synchronize()
            piece[:part.numel()].copy_(part)
            to[lo:lo + STAGING_PIECE].copy_(piece[:part.numel()], non_blocking=True)
            sent.record(stream)
            slots.append((piece, sent))
    hdr = torch.empty(head, dtype=torch.uint8, device=device)
    rows = torch.empty(size, dtype=torch.uint8, device=device)
    send(hdr, host_hdr)
    send(rows, host_rows)
    return rows.view(P, N), hdr.view(torch.int32).view(P, 4)


def pack_rows(rows, hdr, check=None, findings=None):
    """Code rows [P, N] on the device -> [ceil(N / 16), P, 16] (plan-minor, sixteen ops per 16-byte word, zero padded);
    `check` and `findings` as in DeviceBatch."""
    import torch
    P, N = rows.shape
    G = (N + 15) // 16
    if P == 0:
        return torch.empty((G, 0, 16), dtype=torch.uint8, device=rows.device)
    if rows.device.type != "cuda":
        return torch.nn.functional.pad(rows, (0, G * 16 - N)).view(P, G, 16).permute(1, 0, 2).contiguous()
    lib = load_library()
    codes = torch.empty((G, P, 16), dtype=torch.uint8, device=rows.device)
    n_mbs, n_codes = check or (0, 8)
    flags = None if not check else torch.zeros(1, dtype=torch.int32, device=rows.device) if findings is None else findings
    with torch.cuda.device(rows.device):
        _check(lib, lib.ace_pack_plans(rows.data_ptr(), P, N, hdr.data_ptr() if check else None, n_mbs, n_codes, codes.data_ptr(),
                                       flags.data_ptr() if check else None,
                                       torch.cuda.current_stream(rows.device).cuda_stream), "ace_pack_plans")
    if check and findings is None:
        msg = finding(int(flags.item()))
        if msg:
            raise ValueError(msg)
    return codes


class DeviceBatch:
    """A PlanBatch resident in HBM in the layout the kernel streams."""

    def __init__(self, batch: PlanBatch, device="cuda:0", ranges: Optional[np.ndarray] = None, staging=None,
                 group_by_depth: bool = False, check=None, findings=None):
        """`staging`: a pinned uint8 host tensor of at least P * N bytes; the plan bytes then go through
        it and the copy to the device does not block the host (the caller must not reuse the tensor
        before that copy has completed).
        `group_by_depth`: store the plans sorted by pipeline depth (deepest first) and position of the
        first two stage boundaries, with the permutation alongside (`order`), so that the lanes of a
        wavefront close their stages together; results still come back in the caller's order.
        `check`: (micro-batch sizes, codes) of the tables; the plans' structure is then checked on the way
        (ValueError).  `findings`: a zeroed device int32 that takes what the check finds instead; the caller reads it,
        with what it reads anyway."""
        import torch
        P, N = batch.codes.shape
        order = None
        if group_by_depth and P > 1:
            perm = depth_order(batch)
            batch = PlanBatch(batch.codes[perm], batch.hdr[perm])
            if ranges is not None:
                ranges = np.asarray(ranges)[perm]
            order = torch.from_numpy(perm.astype(np.int32)).to(device)
        rows, hdr = rows_to_device(batch, device, staging)
        if ranges is not None:
            r = np.ascontiguousarray(ranges, dtype=np.uint32)
            assert r.shape == (P, 2)
            ranges = torch.from_numpy(r.view(np.int32)).to(device)
        self._set(pack_rows(rows, hdr, check, findings), hdr, N, ranges, order)

    def _set(self, codes, hdr, num_ops, ranges, order):
        self.n_plans, self.num_ops = int(hdr.shape[0]), int(num_ops)
        self.codes, self.hdr, self.ranges, self.order = codes, hdr, ranges, order
        self.struct = AceBatchStruct(codes.data_ptr(), hdr.data_ptr(), ranges.data_ptr() if ranges is not None else None,
                                     self.n_plans, order.data_ptr() if order is not None else None)

    @classmethod
    def from_device(cls, codes, hdr, num_ops: int, ranges=None, order=None):
        """Wrap tensors that are already on the device in the kernel's layout: codes uint8 [G, P, 16], hdr int32
        [P, 4], ranges (single-stage queries) int32 [P, 2] or None, order int32 [P] (result index of the plan in
        each slot) or None."""
        self = cls.__new__(cls)
        self._set(codes, hdr, num_ops, ranges, order)
        return self

    @property
    def bytes_moved_per_plan(self):
        return self.codes.shape[0] * 16 + 16 + (4 if self.order is not None else 0)


class PlanEvaluator:
    def __init__(self, tables: CompiledTables, device="cuda:0"):
        import torch
        if not torch.cuda.is_available():
            raise AceError("no GPU visible: plan scoring runs on the HIP kernels only")
        self.lib = load_library()
        self.tables = tables
        self._plan_bytes = 16 * ((tables.graph.num_ops + 15) // 16)
        # (a device without an index: the one that is current now, where the handle comes to live)
        self.device = torch.device(device)
        if self.device.index is None:
            self.device = torch.device(self.device.type, torch.cuda.current_device())
        self._torch = torch
        with torch.cuda.device(self.device):
            ts = tables.as_struct()
            h = ctypes.c_void_p()
            _check(self.lib, self.lib.ace_create(ctypes.byref(ts), ctypes.byref(h)), "ace_create")
        self.handle = h
        self._deal_cache = {}
        self._topk_ws = None
        self._rc_ready, self._rc_lock = None, threading.Lock()
        self._graphs_alive = 0
        self._copy_stream = None

    def close(self):
        if getattr(self, "handle", None):
            self.lib.ace_destroy(self.handle)
            self.handle = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def upload(self, batch: PlanBatch, validate: bool = True, ranges: Optional[np.ndarray] = None,
               staging=None, group_by_depth: bool = False, findings=None) -> DeviceBatch:
        """`validate` checks the encoding on the host first (a clear message instead of per-plan status
        bytes; the kernel itself is safe for any byte content).  `group_by_depth`, `findings`: see DeviceBatch."""
        check = None
        if validate and ranges is not None:
            host_arrays(batch.codes, batch.hdr, self.tables.graph.num_ops)       # (a query's plan need not be a whole one: no check of it)
        elif validate:
            # (small batches are checked before they go anywhere; for others the check rides on the device's packing of the
            # plans and costs the read-back of its findings; not where the call must not wait for the device)
            small = batch.codes.size <= self.HOST_CHECK_BYTES or (findings is None and (
                staging is not None or self._torch.cuda.is_current_stream_capturing()))
            msg = validate_batch(batch, self.tables) if small else check_shape(batch, self.tables)
            if msg:
                raise ValueError(msg)
            check = None if small else (len(self.tables.db.mbs_list), self.tables.C)
        return DeviceBatch(batch, self.device, ranges, staging, group_by_depth, check, findings)

    def pinned_plan_batch(self, n_plans: int) -> PlanBatch:
        """An empty PlanBatch (codes uint8 [n_plans, N], hdr uint32 [n_plans, 4]) whose arrays live in page-locked host
        memory: a producer that writes its plans there (synth.make_plans(out=...), neighbours on the host, a reader of
        plan files) hands them to upload() / score_stream() without the host-side staging copy, so the transfer runs at
        the bus's rate.  The caller must not rewrite the arrays while an upload of them is in flight."""
        torch = self._torch
        N = self.tables.graph.num_ops
        tc = torch.empty((n_plans, N), dtype=torch.uint8, pin_memory=True)
        th = torch.empty((n_plans, 4), dtype=torch.int32, pin_memory=True)
        b = PlanBatch(tc.numpy(), th.numpy().view(np.uint32))
        b.pinned_tensors = (tc, th)
        return b

    def device_context(self):
        """Context manager that makes this evaluator's GPU the current one (for raw library calls)."""
        return self._torch.cuda.device(self.device)

    def copy_stream(self):
        """A stream for copies beside the kernels, the same one every time (the allocator keeps memory by stream)."""
        if self._copy_stream is None:
            self._copy_stream = self._torch.cuda.Stream(self.device)
        return self._copy_stream

    def _stream(self):
        return ctypes.c_void_p(self._torch.cuda.current_stream(self.device).cuda_stream)

    def _fits(self, d: DeviceBatch):
        """The kernels read as many 16-op groups of every plan as the op graph has."""
        if d.codes.numel() < d.n_plans * self._plan_bytes:
            raise ValueError(f"{d.n_plans} plans of {self._plan_bytes // 16} 16-op groups expected, the batch's codes have {d.codes.numel()} bytes")

    def score(self, dbatch: DeviceBatch, memory_limit: Optional[float] = None, strict: bool = False,
              breakdown: bool = False, out=None):
        """Launch the scoring kernel; returns device tensors (iter_ms, peak_mb, feasible, status[, stage records
        [P, 16, STAGE_REC]; [P, 1, STAGE_REC] for single-stage queries]).  Where `status` is not 0 the scores are NaN and
        the records hold no particular values."""
        torch = self._torch
        self._fits(dbatch)
        P = dbatch.n_plans
        limit = float(self.tables.settings.memory_limit if memory_limit is None else memory_limit)
        if out is None:
            it = torch.empty(P, dtype=torch.float64, device=self.device)
            pk = torch.empty(P, dtype=torch.float64, device=self.device)
            fe = torch.empty(P, dtype=torch.uint8, device=self.device)
            st = torch.empty(P, dtype=torch.uint8, device=self.device)
        else:
            it, pk, fe, st = out
        breakdown = breakdown or dbatch.ranges is not None
        # (plain scoring with every row resident uses the handle's workspace, which the library reallocates for a larger
        # batch -- unless a captured step holds its address: then ace_reserve() has fixed it and the call is refused)
        # (a single-stage query has one record)
        n_rec = 1 if dbatch.ranges is not None else MAX_STAGES
        rec = torch.zeros((P, n_rec, STAGE_REC), dtype=torch.float64, device=self.device) if breakdown else None
        with torch.cuda.device(self.device):
            rc = self.lib.ace_score_batch(self.handle, ctypes.byref(dbatch.struct), limit, int(strict),
                                          it.data_ptr(), pk.data_ptr(), fe.data_ptr(), st.data_ptr(),
                                          rec.data_ptr() if breakdown else None, self._stream())
        _check(self.lib, rc, "ace_score_batch")
        return (it, pk, fe, st, rec) if breakdown else (it, pk, fe, st)

    def reserve(self, max_plans: int, fixed: bool = False):
        """Size the handle's scoring workspace for batches of up to `max_plans` plans now; `fixed`: a later, larger
        batch is refused (AceError) instead of reallocating it (what a captured step needs)."""
        with self._torch.cuda.device(self.device):
            _check(self.lib, self.lib.ace_reserve(self.handle, int(max_plans), int(fixed)), "ace_reserve")

    def topk(self, iter_ms, feasible, k: int):
        """Device-wide top-k: (indices int64[k], times f64[k], count)."""
        torch, k = self._torch, operator.index(k)
        buf = self.topk_packed(iter_ms, feasible, k)
        return buf[:8 * k].view(torch.int64), buf[8 * k:16 * k].view(torch.float64), buf[16 * k:16 * k + 4].view(torch.int32)

    def topk_packed(self, iter_ms, feasible, k: int, out=None):
        """topk() in one device buffer (indices, times, count: one copy brings all of them to the host); `out`: that buffer
        (uint8, at least 16 * k + 4)."""
        torch = self._torch
        n, k = iter_ms.numel(), operator.index(k)
        need = self.lib.ace_topk_workspace_bytes(n, k)
        if self._topk_ws is None or self._topk_ws.numel() < need:
            # (a captured step keeps its own reference to the workspace it recorded, so the old one stays alive for it)
            self._topk_ws = torch.empty(need, dtype=torch.uint8, device=self.device)
        buf = torch.empty(16 * k + 8, dtype=torch.uint8, device=self.device) if out is None else out
        at = buf.data_ptr()
        with torch.cuda.device(self.device):
            rc = self.lib.ace_topk(self.handle, iter_ms.data_ptr(), feasible.data_ptr(), n, k, at, at + 8 * k, at + 16 * k,
                                   self._topk_ws.data_ptr(), self._topk_ws.numel(), self._stream())
        _check(self.lib, rc, "ace_topk")
        return buf

    @staticmethod
    def read_topk(buf, k: int):
        """topk_packed's result on the host: (indices, times) of the feasible ones."""
        host = buf if isinstance(buf, np.ndarray) else buf.cpu().numpy()
        n = int(host[16 * k:16 * k + 4].view(np.int32)[0])
        return host[:8 * k].view(np.int64)[:n], host[8 * k:16 * k].view(np.float64)[:n]

    def top_k(self, batch: PlanBatch, k: int, memory_limit: Optional[float] = None, strict: bool = False):
        """(indices, times) of the k fastest feasible plans of a host batch.  Everything is asked for before anything is read:
        what the structural check of the plans has found comes back with the result (scoring is safe for any bytes)."""
        torch, k = self._torch, operator.index(k)
        buf = torch.zeros(16 * k + 16, dtype=torch.uint8, device=self.device)
        d = self.upload(batch, findings=buf[16 * k + 8:16 * k + 12].view(torch.int32))
        it, pk, fe, st = self.score(d, memory_limit, strict)
        host = self.topk_packed(it, fe, k, buf).cpu().numpy()
        msg = finding(int(host[16 * k + 8:16 * k + 12].view(np.int32)[0]))
        if msg:
            raise ValueError(msg)
        return self.read_topk(host, k)

    def capture_step(self, dbatch: DeviceBatch, k: int, memory_limit: Optional[float] = None, strict: bool = False):
        """Score + top-k of a resident batch recorded once in a HIP graph (the library's launches record into a
        capturing stream as they are; nothing in them clears memory with a memset node).  Returns a StepGraph:
        `replay()` runs the recorded launches again on the batch's current bytes and returns the same output
        tensors ((iter_ms, peak_mb, feasible, status), (indices, times, count)).  For a batch that is scored
        again and again after edits in place; the launches of a step (scoring, one or two of the top-k for k <= 256) then cost one submission."""
        return StepGraph(self, dbatch, k, memory_limit, strict)

    def time_score_kernel(self, dbatch: DeviceBatch, reps: int, memory_limit: Optional[float] = None) -> float:
        """Average scoring-kernel duration in ms over `reps` back-to-back launches (hipEvents on the
        launch stream)."""
        torch = self._torch
        self._fits(dbatch)
        P = dbatch.n_plans
        limit = float(self.tables.settings.memory_limit if memory_limit is None else memory_limit)
        it = torch.empty(P, dtype=torch.float64, device=self.device)
        pk = torch.empty(P, dtype=torch.float64, device=self.device)
        fe = torch.empty(P, dtype=torch.uint8, device=self.device)
        ms = ctypes.c_double()
        with torch.cuda.device(self.device):
            rc = self.lib.ace_time_score_kernel(self.handle, ctypes.byref(dbatch.struct), limit, 0, it.data_ptr(),
                                                pk.data_ptr(), fe.data_ptr(), reps, self._stream(), ctypes.byref(ms))
        _check(self.lib, rc, "ace_time_score_kernel")
        return ms.value

    def score_stream(self, batches, k: int, memory_limit: Optional[float] = None, strict: bool = False):
        """Score host-resident batches one after the other while the next one is uploaded: uploads go to a second
        stream (same priority), scoring and the per-batch top-k run on the current stream.  Plans are not validated on
        the host: malformed or unscorable ones come back infeasible.  Returns (global plan indices, times) of the k
        fastest feasible plans over all batches (ascending, ties -> lower global index) and the number of plans seen."""
        torch = self._torch
        copy_stream = self.copy_stream()
        main = torch.cuda.current_stream(self.device)
        best_idx = np.empty(0, dtype=np.int64)
        best_val = np.empty(0, dtype=np.float64)
        offset = 0
        it = iter(batches)

        def upload(b):
            # (only copies on the second stream, so that the bus never waits for a kernel)
            with torch.cuda.stream(copy_stream):
                rows, hdr = rows_to_device(b, self.device)
                ev = torch.cuda.Event()
                ev.record(copy_stream)
            return rows, hdr, ev

        nxt = next(it, None)
        pending = upload(nxt) if nxt is not None else None
        while pending is not None:
            rows, hdr, ready = pending
            main.wait_event(ready)
            d = DeviceBatch.from_device(pack_rows(rows, hdr), hdr, rows.shape[1])
            t, pk, fe, st = self.score(d, memory_limit, strict)
            top = self.topk_packed(t, fe, k)
            # (the next batch is on its way before this one's result is waited for: the bus has work all the time)
            nxt = next(it, None)
            pending = upload(nxt) if nxt is not None else None
            idx, val = self.read_topk(top, k)                          # synchronises this batch
            best_idx = np.concatenate([best_idx, idx + offset])
            best_val = np.concatenate([best_val, val])
            order = np.lexsort((best_idx, best_val))[:k]
            best_idx, best_val = best_idx[order], best_val[order]
            offset += d.n_plans
            del d, rows, hdr
        return best_idx, best_val, offset

    def apply_moves(self, templates: PlanBatch, moves: np.ndarray, with_keys: bool = False):
        """Expand move descriptors (neighbours.sample_moves) into a device-resident batch: only the
        templates and 16 bytes per neighbour cross the bus.  With `with_keys` also returns a device
        tensor int64[n] holding a 64-bit key of every plan's bytes (neighbours.plan_keys_host computes
        the same keys from a PlanBatch)."""
        torch = self._torch
        T, N = templates.codes.shape
        G = (N + 15) // 16
        n = int(moves.shape[0])
        # one upload: descriptors, template headers, template code rows
        off_hdr, off_codes = 16 * n, 16 * (n + T)
        up = np.zeros(off_codes + T * G * 16, dtype=np.uint8)
        up[:off_hdr].view(np.uint32).reshape(n, 4)[...] = moves
        up[off_hdr:off_codes].view(np.uint32).reshape(T, 4)[...] = templates.hdr
        up[off_codes:].reshape(T, G * 16)[:, :N] = templates.codes
        d_up = torch.from_numpy(up).to(self.device)
        at = d_up.data_ptr()
        codes = torch.empty((G, n, 16), dtype=torch.uint8, device=self.device)
        hdr = torch.empty((n, 4), dtype=torch.int32, device=self.device)
        keys = torch.zeros((n, 2), dtype=torch.int64, device=self.device) if with_keys else None
        with torch.cuda.device(self.device):
            rc = self.lib.ace_apply_moves(at + off_codes, at + off_hdr, T, at, n, N,
                                          self.tables.db.n_algo, codes.data_ptr(), hdr.data_ptr(),
                                          keys.data_ptr() if with_keys else None, self._stream())
        _check(self.lib, rc, "ace_apply_moves")
        d = DeviceBatch.from_device(codes, hdr, N)
        return (d, keys) if with_keys else d

    def search_step(self, plan: PlanBatch, draws: AceMoveDrawsStruct, sets=()):
        """One step of a search in one library call (ace_search_step): the new ones among the drawn moves on plan 0 of `plan`
        expanded, scored and the fastest feasible one picked: (plan, iteration ms, peak MB), or None.  `sets`: handles of
        the visited sets (empty: only repeated moves are dropped)."""
        t, best = self.tables, AceStepResultStruct()
        if t.graph.num_ops >= 65536:
            raise ValueError("move descriptors hold 16-bit op positions")
        codes, hdr = host_arrays(plan.codes[:1], plan.hdr[:1], t.graph.num_ops)
        codes_out, hdr_out = np.empty_like(codes), np.empty_like(hdr)
        handles = (ctypes.c_void_p * max(1, len(sets)))(*sets)
        _check(self.lib, self.lib.ace_search_step(self.handle, codes.ctypes.data, hdr.ctypes.data, t.stage_lut.ctypes.data,
                                                  t.settings.num_gpus_per_node, ctypes.byref(draws), handles, len(sets),
                                                  float(t.settings.memory_limit), 0, codes_out.ctypes.data, hdr_out.ctypes.data,
                                                  ctypes.byref(best), self._stream()), "ace_search_step")
        return (PlanBatch(codes_out, hdr_out), best.iter_ms, best.peak_mb) if best.found else None

    def prepare_recompute(self, no_recompute: np.ndarray) -> bool:
        """Upload what check_recompute needs beside the tables (once); False if the op graph is too long for the kernel."""
        with self._rc_lock:
            if self._rc_ready is None:
                t = self.tables
                types = np.ascontiguousarray(t.graph.type_of_pos, dtype=np.int32)
                act = np.ascontiguousarray(t.db.tables["activations"], dtype=np.float64)
                norec = np.ascontiguousarray(no_recompute, dtype=np.uint8)
                with self.device_context():
                    rc = self.lib.ace_recompute_prepare(self.handle, types.ctypes.data, act.ctypes.data, norec.ctypes.data)
                if rc != ACE_ETOOBIG:
                    _check(self.lib, rc, "ace_recompute_prepare")
                self._rc_ready = rc == 0
            return self._rc_ready

    def recompute(self, d: DeviceBatch, memory_limit: float, peak_backward: float):
        """check_recompute's choice for every stage of every plan, after prepare_recompute: (the new batch, status of the
        plans, int32[4] flags of ace_recompute_batch), on the device."""
        torch = self._torch
        status = self.score(d, memory_limit)[3]
        codes = torch.empty_like(d.codes)
        flags = torch.zeros(4, dtype=torch.int32, device=self.device)
        with self.device_context():
            _check(self.lib, self.lib.ace_recompute_batch(self.handle, ctypes.byref(d.struct), float(memory_limit), float(peak_backward),
                                                          status.data_ptr(), codes.data_ptr(), flags.data_ptr(), self._stream()),
                   "ace_recompute_batch")
        return DeviceBatch.from_device(codes, d.hdr, d.num_ops), status, flags

    def select(self, d: DeviceBatch, index) -> DeviceBatch:
        """The plans `index` (device int64 tensor) of a device-resident batch, as a new batch."""
        if d.order is not None:
            raise ValueError("select: the batch is stored in grouped order (group_by_depth)")
        return DeviceBatch.from_device(d.codes.index_select(1, index).contiguous(), d.hdr.index_select(0, index).contiguous(),
                                       d.num_ops)

    def download(self, d: DeviceBatch, index=None) -> PlanBatch:
        """A device-resident batch (or its plans `index`, a device int64 tensor) as a host PlanBatch."""
        if index is not None:
            d = self.select(d, index)
        if d.order is not None:
            raise ValueError("download: the batch is stored in grouped order (group_by_depth)")
        torch = self._torch
        P, N = d.n_plans, d.num_ops
        if P == 0:
            return PlanBatch(np.empty((0, N), dtype=np.uint8), np.empty((0, 4), dtype=np.uint32))
        both = torch.empty(16 * P + P * N, dtype=torch.uint8, device=self.device)
        both[:16 * P].copy_(d.hdr.view(torch.uint8).view(-1))
        with self.device_context():
            _check(self.lib, self.lib.ace_unpack_plans(d.codes.data_ptr(), P, N, both.data_ptr() + 16 * P, self._stream()), "ace_unpack_plans")
        # (up to PINNED_RESULT_BYTES the arrays handed out are page-locked: one copy at the bus's rate, no second one)
        if both.numel() <= self.PINNED_RESULT_BYTES:
            host = torch.empty(both.numel(), dtype=torch.uint8, pin_memory=True)
            host.copy_(both, non_blocking=True)
            torch.cuda.current_stream(self.device).synchronize()
        else:
            host = both.cpu()
        host = host.numpy()
        return PlanBatch(host[16 * P:].reshape(P, N), host[:16 * P].view(np.uint32).reshape(P, 4))

    def group(self, d: DeviceBatch) -> DeviceBatch:
        """A copy of a device-resident batch in grouped storage order (see DeviceBatch), made on the
        device: sort keys from the library (ace_group_keys), a stable sort, one gather of the plan
        bytes.  Worth it for a batch that is scored more than once; results of the copy come back in the
        order of `d`.  Equal to upload(batch, group_by_depth=True) of the same plans."""
        torch = self._torch
        if d.order is not None or d.ranges is not None:
            raise ValueError("group: a plain batch in its own order is expected")
        P = d.n_plans
        keys = torch.empty(P, dtype=torch.int64, device=self.device)
        with self.device_context():
            _check(self.lib, self.lib.ace_group_keys(d.codes.data_ptr(), d.hdr.data_ptr(), P, d.num_ops, keys.data_ptr(),
                                                     self._stream()), "ace_group_keys")
        by_key = torch.sort(keys, stable=True).indices       # (keys are below 2^48: signed order = unsigned order)
        slots = self._deal_cache.get(P)
        if slots is None:
            slots = torch.from_numpy(deal_slots(P)).to(self.device)
            self._deal_cache = {P: slots}
        perm = by_key.index_select(0, slots).to(torch.int32)
        codes, hdr = torch.empty_like(d.codes), torch.empty_like(d.hdr)
        with self.device_context():
            _check(self.lib, self.lib.ace_gather_plans(d.codes.data_ptr(), d.hdr.data_ptr(), perm.data_ptr(), P, d.num_ops,
                                                       codes.data_ptr(), hdr.data_ptr(), self._stream()), "ace_gather_plans")
        return DeviceBatch.from_device(codes, hdr, d.num_ops, order=perm)

    def stage_records_host(self, batch: PlanBatch, ranges: np.ndarray):
        """Single-stage queries: (status, stage record 0 of every query) as numpy arrays."""
        out = self.score(self.upload(batch, ranges=ranges), breakdown=True)
        return out[3].cpu().numpy(), out[4][:, 0, :].cpu().numpy()

    def picked_records_host(self, batch: PlanBatch, plan_idx: np.ndarray, stage_idx: np.ndarray):
        """Whole plans: (status of every plan, the stage records [plan_idx[k], stage_idx[k]]) as numpy arrays
        (picked on the device, so only those records cross the bus)."""
        torch = self._torch
        out = self.score(self.upload(batch), breakdown=True)
        pick = out[4][torch.from_numpy(np.ascontiguousarray(plan_idx)).to(self.device),
                      torch.from_numpy(np.ascontiguousarray(stage_idx)).to(self.device)]
        return out[3].cpu().numpy(), pick.cpu().numpy()

    PINNED_RESULT_BYTES = 64 << 20
    HOST_CHECK_BYTES = 128 << 10     # (the host checks 4 to 8 GB/s, the read-back is 20 us)

    # ---- small host-in / host-out calls ------------------------------------------------------------
    # The reference's search calls the cost model for one plan or one stage at a time, so the time of such
    # a call is what a host-side search sees.  Small batches therefore take one library call (ace_score_host): laid out in
    # page-locked memory, which the kernel reads and writes where it is.
    SMALL_IO_BYTES = 1 << 20

    def _score_small(self, batch: PlanBatch, limit: float, strict: bool, breakdown: bool, ranges):
        """score_host for a batch whose inputs and outputs fit the library's page-locked buffers; None if they do not."""
        P = batch.codes.shape[0]
        breakdown = breakdown or ranges is not None
        n_rec = 1 if ranges is not None else MAX_STAGES          # a single-stage query has one record
        # (a query's plan is not checked: it never had to be of integers)
        codes, hdr = host_arrays(batch.codes, batch.hdr, self.tables.graph.num_ops, integers=ranges is None)
        codes_at, hdr_at = codes.ctypes.data, hdr.ctypes.data
        if ranges is not None:
            ranges = host_ranges(ranges, P)
        else:
            msg = check_plans(self.lib, codes_at, hdr_at, P, self.tables) if P else check_shape(batch, self.tables)
            if msg:
                raise ValueError(msg)
        times = np.empty((2, P))
        flags = np.empty((2, P), dtype=np.uint8)
        rec = np.empty((P, n_rec, STAGE_REC)) if breakdown else None
        rc = self.lib.ace_score_host(self.handle, codes_at, hdr_at, ranges.ctypes.data if ranges is not None else None, P,
                                     limit, int(strict), _address(times), _address(flags), _address(rec) if breakdown else None,
                                     self._torch._C._cuda_getCurrentRawStream(self.device.index))
        if rc == ACE_ETOOBIG:
            return None
        _check(self.lib, rc, "ace_score_host")
        out = (times[0], times[1], flags[0], flags[1])
        return out + (rec,) if breakdown else out

    # convenience: host in, host out
    def score_host(self, batch: PlanBatch, memory_limit=None, strict=False, breakdown=False, ranges=None,
                   group_by_depth: bool = False):
        if not group_by_depth and batch.n_plans <= 4096 and batch.codes.size < self.SMALL_IO_BYTES:
            limit = float(self.tables.settings.memory_limit if memory_limit is None else memory_limit)
            out = self._score_small(batch, limit, strict, breakdown, ranges)
            if out is not None:
                return out
        d = self.upload(batch, ranges=ranges, group_by_depth=group_by_depth)
        out = self.score(d, memory_limit, strict, breakdown)
        self._torch.cuda.synchronize(self.device)
        return tuple(None if t is None else t.cpu().numpy() for t in out)


class StepGraph:
    """See PlanEvaluator.capture_step."""

    def __init__(self, ev: PlanEvaluator, dbatch: DeviceBatch, k: int, memory_limit=None, strict=False):
        torch = ev._torch
        self.batch = dbatch                       # the graph holds its addresses
        P = dbatch.n_plans
        self.scores = (torch.empty(P, dtype=torch.float64, device=ev.device), torch.empty(P, dtype=torch.float64, device=ev.device),
                       torch.empty(P, dtype=torch.uint8, device=ev.device), torch.empty(P, dtype=torch.uint8, device=ev.device))
        # one eager step on a side stream first: the handle's workspace and the top-k workspace are allocated
        # there, never inside the capture
        side = torch.cuda.Stream(device=ev.device)
        side.wait_stream(torch.cuda.current_stream(ev.device))
        with torch.cuda.stream(side):
            ev.score(dbatch, memory_limit, strict, out=self.scores)
            ev.topk(self.scores[0], self.scores[2], k)
        torch.cuda.current_stream(ev.device).wait_stream(side)
        torch.cuda.synchronize(ev.device)
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph):
            ev.score(dbatch, memory_limit, strict, out=self.scores)
            self.top = ev.topk(self.scores[0], self.scores[2], k)
        self._topk_ws = ev._topk_ws               # the recorded launches write into it: it must outlive a larger topk()
        self._ev = ev
        ev._graphs_alive += 1
        ev.reserve(0, fixed=True)                 # the handle's workspace may not move while the graph lives

    def replay(self):
        if self._ev is None or not self._ev.handle:
            raise AceError("the captured step was released, or its evaluator closed")
        self.graph.replay()
        return self.scores, self.top

    def release(self):
        """Forget the recorded launches (the evaluator may then score larger batches again)."""
        if self._ev is not None:
            self._ev._graphs_alive -= 1
            if self._ev._graphs_alive == 0 and self._ev.handle:
                self._ev.reserve(0, fixed=False)
            self._ev = None
            self.graph = None
            self._topk_ws = None

    def __del__(self):
        try:
            self.release()
        except Exception:
            pass
