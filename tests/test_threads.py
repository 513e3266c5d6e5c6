"""Several threads with one evaluator: the host calls share page-locked buffers and take turns, and what is made on first use is
made once."""
import types
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from superscaler_amd import synth
from superscaler_amd.evaluator import PlanEvaluator
from tests.test_small_batches import WORKLOADS, stage_queries


def test_recompute_is_prepared_once():
    import contextlib
    import threading
    import time
    tables = synth.make_tables(WORKLOADS["gpt_wide_stages"])
    calls = []

    def prepare(*_):
        calls.append(1)
        time.sleep(0.05)
        return 0
    ev = types.SimpleNamespace(tables=tables, handle=None, lib=types.SimpleNamespace(ace_recompute_prepare=prepare), _rc_ready=None,
                               _rc_lock=threading.Lock(), device_context=contextlib.nullcontext)
    none = np.zeros(len(tables.db.op_names), dtype=np.uint8)
    with ThreadPoolExecutor(4) as pool:
        assert list(pool.map(lambda _: PlanEvaluator.prepare_recompute(ev, none), range(4))) == [True] * 4
    assert len(calls) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["gpt3_1_3b", "wresnet_1b"])
def test_host_calls_of_several_threads(name):
    from superscaler_amd.neighbours import _draw_moves, _draws_struct
    w = WORKLOADS[name]
    tables = synth.make_tables(w)
    ev = PlanEvaluator(tables)
    batches = [synth.make_plans(w, tables, n_plans=n, seed_offset=n) for n in (1, 37, 400, 1000)]
    queries = [stage_queries(b.slice(0, 50)) for b in batches]
    bases = [b.slice(0, 1) for b in batches]
    draws = [_draw_moves(500, int(b.hdr[0, 0] & 0xff), tables, np.random.default_rng(k), 8) for k, b in enumerate(bases)]

    def work(k):
        out = []
        for _ in range(25):
            out.append(ev.score_host(batches[k], breakdown=True))
            out.append(ev.score_host(queries[k][0], ranges=queries[k][1]))
            best = ev.search_step(bases[k], _draws_struct(draws[k]))
            out.append(() if best is None else (best[0].codes, best[0].hdr, best[1], best[2]))
        return out
    alone = [work(k) for k in range(4)]
    with ThreadPoolExecutor(4) as pool:
        together = list(pool.map(work, range(4)))
    for a, b in zip(alone, together):
        for x, y in zip(a, b):
            assert len(x) == len(y) and all(np.array_equal(p, q, equal_nan=True) for p, q in zip(x, y))
    ev.close()
