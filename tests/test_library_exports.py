"""The C-ABI library loads without a GPU and exports every function include/ace_eval.h declares;
argument checking that needs no device is exercised too (no kernel is launched here)."""
import ctypes
import os
import re

import pytest

from superscaler_amd import evaluator, synth
from superscaler_amd.tables import AceTablesStruct

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_functions():
    text = open(os.path.join(ROOT, "include", "ace_eval.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(ace_[a-z_0-9]+)\s*\(", text)))


def test_every_declared_symbol_is_exported():
    lib = evaluator.load_library()
    names = declared_functions()
    assert {"ace_create", "ace_destroy", "ace_score_batch", "ace_topk", "ace_strerror"} <= set(names)
    for n in names:
        assert hasattr(lib, n), f"{n} is declared in include/ace_eval.h but not exported"
    assert sorted(evaluator.EXPORTS) == names
    assert lib.ace_abi_version() == 8


def test_error_strings_and_argument_checks():
    lib = evaluator.load_library()
    assert lib.ace_strerror(0) == b"ok"
    assert lib.ace_strerror(-1) == b"invalid argument"
    assert lib.ace_strerror(-99) == b"unknown error"
    h = ctypes.c_void_p()
    assert lib.ace_create(None, ctypes.byref(h)) == -1          # null tables
    ts = AceTablesStruct()
    ts.abi_version = 1
    assert lib.ace_create(ctypes.byref(ts), ctypes.byref(h)) == -5   # ABI version mismatch
    tables = synth.make_tables(synth.WORKLOADS["gpt3_1_3b"])
    bad = tables.as_struct()
    bad.n_tp = 9
    assert lib.ace_create(ctypes.byref(bad), ctypes.byref(h)) == -1  # geometry the encoding cannot hold
    bad = tables.as_struct()
    lut = tables.stage_lut.copy()
    lut[0, 0] = 0xFFF0                                              # a diag the tables do not have
    bad.stage_lut = lut.ctypes.data
    assert lib.ace_create(ctypes.byref(bad), ctypes.byref(h)) == -1
    assert lib.ace_topk_workspace_bytes(1 << 20, 64) > 0
    assert lib.ace_topk_workspace_bytes(1 << 20, 0) == 0


def test_missing_library_fails_loudly(monkeypatch):
    monkeypatch.setattr(evaluator, "_lib", None)
    monkeypatch.setattr(evaluator, "_LIB_PATH", "/nonexistent/libace_eval.so")
    with pytest.raises(evaluator.AceError):
        evaluator.load_library()


def test_host_side_work_on_plans_names_the_build_command_without_the_libraries(monkeypatch):
    """Encoding, the structural check, move descriptors and visited sets are native; tables, plans and plan files are not."""
    import sys
    import numpy as np
    import superscaler_amd
    from superscaler_amd.neighbours import VisitedKeys, sample_moves
    from superscaler_amd.plan import PlanBatch, validate_batch
    monkeypatch.setattr(evaluator, "_lib", None)
    monkeypatch.setattr(evaluator, "_objects", None)
    monkeypatch.setattr(evaluator, "_LIB_PATH", "/nonexistent/libace_eval.so")
    monkeypatch.setitem(sys.modules, "superscaler_amd._ace_objects", None)
    monkeypatch.delattr(superscaler_amd, "_ace_objects", raising=False)
    w = synth.WORKLOADS["gpt3_1_3b"]
    tables = synth.make_tables(w)
    batch = synth.make_plans(w, tables, n_plans=2)
    config = batch.to_config(0, tables)
    for call in (lambda: PlanBatch.from_configs([config], tables), lambda: validate_batch(batch, tables),
                 lambda: sample_moves(batch, tables, 10, np.random.default_rng(0)), VisitedKeys):
        with pytest.raises(evaluator.AceError, match="python -m superscaler_amd.build"):
            call()


def test_no_gpu_means_no_scoring():
    import torch
    if torch.cuda.is_available():
        pytest.skip("a GPU is present")
    tables = synth.make_tables(synth.WORKLOADS["gpt3_1_3b"])
    with pytest.raises(evaluator.AceError):
        evaluator.PlanEvaluator(tables)


OUT_OF_MEMORY = """
import ctypes, resource
import numpy as np
from superscaler_amd import evaluator
lib = evaluator.load_library()
d = evaluator.AceMoveDrawsStruct()
d.n = 1
codes, hdr, out = np.full(16, 16, dtype=np.uint8), np.array([1, 0, 0, 0], dtype=np.uint32), np.zeros(4096, dtype=np.uint32)
codes[1:] = 0
n = ctypes.c_int(0)
used = int(open("/proc/self/statm").read().split()[0]) * resource.getpagesize()
resource.setrlimit(resource.RLIMIT_AS, (used + (1 << 28), used + (1 << 28)))
# (a table of 2^30 micro-batch sizes: 16 GiB that are asked for before anything is read)
rc = lib.ace_build_moves(codes.ctypes.data, hdr.ctypes.data, 16, 2, 4, 1 << 30, out.ctypes.data, 8, ctypes.byref(d), out.ctypes.data, out.ctypes.data,
                         out.ctypes.data, 3, ctypes.byref(n))
print("code", rc)
"""


def test_a_call_that_runs_out_of_memory_returns_a_code():
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    proc = subprocess.run([sys.executable, "-c", OUT_OF_MEMORY], cwd=root, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert proc.returncode == 0 and "code -4" in proc.stdout, (proc.returncode, proc.stdout[-500:])


def test_header_is_plain_c_and_matches_the_library(tmp_path):
    """include/ace_eval.h compiles as C99 on its own, and a C program that takes the address of every
    declared function links against the library (the declarations and the exports agree)."""
    import shutil
    import subprocess
    if shutil.which("gcc") is None:
        pytest.skip("no gcc")
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    hdr = os.path.join(root, "include", "ace_eval.h")
    subprocess.run(["gcc", "-std=c99", "-Wall", "-Werror", "-pedantic", "-fsyntax-only", "-x", "c", hdr], check=True)
    src = tmp_path / "use.c"
    src.write_text('#include "ace_eval.h"\n#include <stdio.h>\nint main(void) {\n'
                   '  const void *f[] = {' + ", ".join(f"(const void *)&{n}" for n in evaluator.EXPORTS) + '};\n'
                   '  printf("%d %d\\n", ace_abi_version(), (int)(sizeof f / sizeof f[0]));\n  return 0;\n}\n')
    exe = tmp_path / "use"
    libdir = os.path.join(root, "superscaler_amd")
    subprocess.run(["gcc", "-std=c99", "-Wno-pedantic", "-I" + os.path.join(root, "include"), str(src), "-o", str(exe),
                    "-L" + libdir, "-l:libace_eval.so", "-Wl,-rpath," + libdir], check=True)
