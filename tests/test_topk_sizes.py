"""ace_topk where its form changes: one workgroup or two launches, entries per lane, stretches of 4,096 / 8,192 / 16,384
entries, the many-launch form -- against a stable sort."""
import numpy as np
import pytest

from superscaler_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("distinct", [3, 1000, 1 << 40])
def test_every_form_equals_a_stable_sort(distinct):
    import torch
    from superscaler_amd.evaluator import PlanEvaluator
    ev = PlanEvaluator(synth.make_tables(synth.WORKLOADS["gpt3_1_3b"]))
    rng = np.random.default_rng(distinct)
    for n in (1, 1024, 4096, 4097, 8192, 8193, 16384, 16385, 65536, 262144, 262145, 524289, (1 << 20) + 7):
        t = rng.integers(0, distinct, n).astype(np.float64)
        f = (rng.random(n) < 0.8).astype(np.uint8)
        order = np.flatnonzero(f)[np.argsort(t[f > 0], kind="stable")]
        dt, df = torch.from_numpy(t).cuda(), torch.from_numpy(f).cuda()
        for k in (1, 63, 64, 128, 255, 256, 257):
            print(f"[case] n={n} k={k} distinct={distinct}", flush=True)
            idx, val, cnt = ev.topk(dt, df, k)
            c = int(cnt.item())
            assert c == min(k, len(order)) and np.array_equal(idx.cpu().numpy()[:c], order[:c]) and np.array_equal(val.cpu().numpy()[:c], t[order[:c]])
            assert (idx[c:] == -1).all() and torch.isinf(val[c:]).all()
    ev.close()


@pytest.mark.parametrize("n", [161, 4096, 5000, 16384, 16385, 65536, 262145, (1 << 20) + 7])
def test_bounded_selection_equals_a_stable_sort(n):
    """Inputs on which the bound of the short form's selection is close, loose or none: random, sorted either way, the best entries
    side by side, keys that differ in their low bits alone, few feasible entries."""
    import torch
    from superscaler_amd.evaluator import PlanEvaluator
    ev = PlanEvaluator(synth.make_tables(synth.WORKLOADS["gpt3_1_3b"]))
    rng = np.random.default_rng(n)
    t = rng.lognormal(3.0, 1.0, n)
    side_by_side = 100.0 + t
    side_by_side[n // 2:n // 2 + 150] = rng.random(min(150, n - n // 2))
    low_bits = (np.float64(3.0).view(np.uint64) + rng.integers(0, 1 << 20, n).astype(np.uint64)).view(np.float64)
    every = np.ones(n, dtype=np.uint8)
    few = np.zeros(n, dtype=np.uint8)
    few[rng.choice(n, 100, replace=False)] = 1
    for name, times, f in (("random", t, (rng.random(n) < 0.8).astype(np.uint8)), ("ascending", np.sort(t), every), ("descending", -np.sort(-t), every),
                           ("side by side", side_by_side, every), ("low bits", low_bits, every), ("few", t, few), ("negative", -t, every)):
        order = np.flatnonzero(f)[np.argsort(times[f > 0], kind="stable")]
        dt, df = torch.from_numpy(np.ascontiguousarray(times)).cuda(), torch.from_numpy(f).cuda()
        for k in (1, 3, 7, 10, 64, 101, 160, 161):
            print(f"[case] {name} n={n} k={k}", flush=True)
            idx, val, cnt = ev.topk(dt, df, k)
            c = int(cnt.item())
            assert c == min(k, len(order)) and np.array_equal(idx.cpu().numpy()[:c], order[:c]) and np.array_equal(val.cpu().numpy()[:c], times[order[:c]])
            assert (idx[c:] == -1).all() and torch.isinf(val[c:]).all()
    ev.close()
