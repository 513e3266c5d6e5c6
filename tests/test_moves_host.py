"""The native host side of the batched search: ace_build_moves (drawn choices -> descriptors) against the rules of
sample_moves written out row by row, ace_new_moves against the keys of the expanded plans, and the key set against a Python set."""
import numpy as np
import pytest

from superscaler_amd import synth
from superscaler_amd.neighbours import (OP_ALGO_TOGGLE, OP_MIGRATE, OP_RC_TOGGLE, OP_TP_STEP, VisitedKeys, _build_moves, _draw_moves,
                                        apply_moves_host, plan_keys_host)
from superscaler_amd.plan import validate_batch
from tests.helpers import odd_workloads

WORKLOADS = {**synth.WORKLOADS, **{w.name: w for w in odd_workloads()}}


def expected(base, tables, draws):
    """Per row: (what kind of template, (op, p0, p1)) by the rules."""
    row, A, N = base.codes[0], tables.db.n_algo, base.num_ops
    S, b = int(base.hdr[0, 0] & 0xff), int(base.hdr[0, 0] >> 8) & 0xff
    lo = np.append(np.flatnonzero(row & 16), N).tolist()
    tp = ((row & 7) // A).tolist()
    sizes = int(base.hdr[0, 1]) | int(base.hdr[0, 2]) << 32
    glog = [(sizes >> 4 * s) & 15 for s in range(S)]
    out = [("base", 0, 0, 0)] * draws["n"]
    for k, (rows, xs, ys) in enumerate(zip(draws["rows"], draws["x"], draws["y"])):
        for i, r in enumerate(rows.tolist()):
            x, y = int(xs[i]), int(ys[i]) if len(ys) else 0
            if k == 0 and lo[x - 1] < lo[x] + y < lo[x + 1]:
                out[r] = ("base", OP_MIGRATE, lo[x] | (lo[x] + y) << 16, tp[lo[x] - 1] if y > 0 else tp[lo[x]])
            elif k == 1 and all(t + y in tables.allowed_tp_logs(b, glog[x]) for t in tp[lo[x]:lo[x + 1]]):
                out[r] = ("base", OP_TP_STEP, lo[x] | lo[x + 1] << 16, int(y > 0))
            elif k == 2 and 0 <= b + x < len(tables.db.mbs_list) and all(
                    t in tables.allowed_tp_logs(b + x, glog[s]) for s in range(S) for t in tp[lo[s]:lo[s + 1]]):
                out[r] = (("mbs", b + x), 0, 0, 0)
            elif k == 3:
                out[r] = ("base", OP_RC_TOGGLE, x | min(N, x + y) << 16, 0)
            elif k == 4:
                out[r] = ("base", OP_ALGO_TOGGLE, x, 0)
            elif k == 5 and x != y and glog[x] - 1 == glog[y]:
                good = True
                for s, g in ((x, glog[x] - 1), (y, glog[y] + 1)):
                    ok = tables.allowed_tp_logs(b, g)
                    good = good and bool(ok) and all(min(max(t, min(ok)), max(ok)) in ok for t in tp[lo[s]:lo[s + 1]])
                if good:
                    out[r] = (("devices", x, y), 0, 0, 0)
    return out


@pytest.mark.parametrize("name", ["gpt3_1_3b", "t5_770m", "wresnet_1b", "gpt3_175b", "gpt_1tp_1mbs", "gpt_wide_stages", "t5_1tp"])
def test_drawn_moves_become_the_descriptors_of_the_rules(name):
    w = WORKLOADS[name]
    tables = synth.make_tables(w)
    for p in range(4):
        base = synth.make_plans(w, tables, n_plans=8, seed_offset=50).slice(p, p + 1)
        draws = _draw_moves(700, int(base.hdr[0, 0] & 0xff), tables, np.random.default_rng(p), 8)
        templates, moves = _build_moves(base, tables, draws)
        assert validate_batch(templates, tables) is None and validate_batch(apply_moves_host(templates, moves, tables.db.n_algo), tables) is None
        glog = [[(int(h[1]) | int(h[2]) << 32) >> 4 * s & 15 for s in range(16)] for h in templates.hdr]
        for m, (what, *edit) in zip(moves.tolist(), expected(base, tables, draws)):
            t = m[0] & 0xffff
            assert [m[0] >> 16, m[1], m[2], m[3]] == [*edit, 0]
            if what == "base":
                assert t == 0
            elif what[0] == "mbs":
                assert t > 0 and int(templates.hdr[t, 0] >> 8) == what[1] and np.array_equal(templates.codes[t], base.codes[0])
            else:
                moved = [g - h for g, h in zip(glog[t], glog[0])]
                assert moved[what[1]] == -1 and moved[what[2]] == 1 and sum(map(abs, moved)) == 2


@pytest.mark.parametrize("name", ["gpt3_1_3b", "t5_770m", "wresnet_1b", "gpt_16ops", "gpt_wide_stages", "t5_1tp"])
def test_moves_kept_are_those_whose_expanded_plans_are_new(name):
    w = WORKLOADS[name]
    tables = synth.make_tables(w)
    a, b = VisitedKeys(), VisitedKeys()
    for p in range(5):
        base = synth.make_plans(w, tables, n_plans=8, seed_offset=50).slice(p % 4, p % 4 + 1)
        draws = _draw_moves(3000, int(base.hdr[0, 0] & 0xff), tables, np.random.default_rng(p), [8, 40][p % 2])
        if p == 3:
            draws["y"][3] = draws["y"][3] * 3 - 3           # (runs that have no bit of their own, and empty ones)
        templates, moves = _build_moves(base, tables, draws)
        want = moves[a.claim(plan_keys_host(apply_moves_host(templates, moves, tables.db.n_algo)))]
        t2, got = b.claim_moves(base, tables, draws)
        assert np.array_equal(got, want) and np.array_equal(t2.codes, templates.codes) and np.array_equal(t2.hdr, templates.hdr)
        assert len(a) == len(b) and not a.unseen(b._small.keys()).any()
        seen, first = set(), []
        for m in moves.tolist():
            first.append(tuple(m) not in seen)
            seen.add(tuple(m))
        assert np.array_equal(_build_moves(base, tables, draws, [])[1], moves[first])


@pytest.mark.parametrize("limit", [10, 65536])
def test_key_set_behaves_like_a_set(limit):
    import copy
    rng = np.random.default_rng(3)
    vk, seen = VisitedKeys(), set()
    vk.SMALL_LIMIT = limit
    for step in range(12):
        keys = rng.integers(0, [1, 40, 5000, 1 << 63][step % 4], size=(3000, 2), dtype=np.uint64)   # (the zero key, many repeats, ...)
        want, here = [], set()
        for k in map(tuple, keys.tolist()):
            want.append(k not in seen and k not in here)
            here.add(k)
        assert vk.unseen(keys).tolist() == want and len(vk) == len(seen)
        assert vk.claim(keys).tolist() == want
        seen |= here
        assert len(vk) == len(seen) and not vk.unseen(keys).any()
    assert len(copy.deepcopy(vk)) == len(vk) and not copy.deepcopy(vk).unseen(keys).any()
    assert vk.unseen(np.zeros((0, 2), dtype=np.uint64)).tolist() == []


def test_threads_may_share_a_visited_set():
    """Every key is claimed once, whichever thread comes first (and copies are whole)."""
    import copy
    from concurrent.futures import ThreadPoolExecutor
    w = WORKLOADS["gpt_wide_stages"]
    tables = synth.make_tables(w)
    base = synth.make_plans(w, tables, n_plans=1, seed_offset=50)
    vk = VisitedKeys()
    vk.SMALL_LIMIT = 3000

    def work(seed):
        rng = np.random.default_rng(seed)
        mine = []
        for step in range(15):
            keys = rng.integers(0, 60_000, size=(4000, 1), dtype=np.uint64).repeat(2, axis=1)
            vk.unseen(keys)
            mine.append(keys[vk.claim(keys)])
            draws = _draw_moves(2000, int(base.hdr[0, 0] & 0xff), tables, rng, 8)
            templates, moves = vk.claim_moves(base, tables, draws)
            mine.append(plan_keys_host(apply_moves_host(templates, moves, tables.db.n_algo)))
            if step % 5 == 0:
                copied = copy.deepcopy(vk)
                assert not copied.unseen(mine[0]).any() and len(copied) <= len(vk)
        return np.concatenate(mine)
    with ThreadPoolExecutor(8) as pool:
        claimed = np.concatenate(list(pool.map(work, range(8))))
    assert len(np.unique(claimed, axis=0)) == len(claimed) == len(vk)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["gpt3_1_3b", "t5_770m", "wresnet_1b", "gpt_wide_stages"])
def test_a_step_picks_what_its_parts_pick(name):
    from superscaler_amd.evaluator import PlanEvaluator
    from superscaler_amd.neighbours import _draws_struct
    w = WORKLOADS[name]
    tables = synth.make_tables(w)
    ev = PlanEvaluator(tables)
    a, b = VisitedKeys(), VisitedKeys()
    for p in range(6):
        base = synth.make_plans(w, tables, n_plans=8, seed_offset=50).slice(p % 4, p % 4 + 1)
        draws = _draw_moves([3000, 200, 1][p % 3], int(base.hdr[0, 0] & 0xff), tables, np.random.default_rng(p), 8)
        for keep in (None, a):
            templates, moves = _build_moves(base, tables, draws, []) if keep is None else a.claim_moves(base, tables, draws)
            got = ev.search_step(base, _draws_struct(draws), () if keep is None else b.handles())
            want = None
            if len(moves):
                it, pk, fe, _ = ev.score(ev.apply_moves(templates, moves))
                idx, val = ev.read_topk(ev.topk_packed(it, fe, 1), 1)
                if len(idx):
                    want = (apply_moves_host(templates, moves[idx[:1]], tables.db.n_algo), float(val[0]), float(pk[int(idx[0])].item()))
            assert (got is None) == (want is None) and len(a) == len(b)
            if got is not None:
                assert got[1:] == want[1:] and np.array_equal(got[0].codes, want[0].codes) and np.array_equal(got[0].hdr, want[0].hdr)
    ev.close()
