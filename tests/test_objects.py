"""The native walk over plan objects (superscaler_amd/csrc/ace_objects.cpp) against the Python code it stands in for: the same
arrays and lists for a search's plans, the same arrays and errors for everything it leaves to that code."""
import collections
import copy

import numpy as np
import pytest

from superscaler_amd import synth
from superscaler_amd.evaluator import load_objects
from superscaler_amd.plan import PlanBatch
from tests.helpers import emu_score, odd_workloads
from tests.test_recompute_kernel import cost_model
from tests.test_small_batches import WORKLOADS


def by_python(configs, tables, intra=False):
    P, N = len(configs), tables.graph.num_ops
    codes, hdr = np.empty((P, N), dtype=np.uint8), np.empty((P, 4), dtype=np.uint32)
    for p, c in enumerate(configs):
        PlanBatch._encode_config(p, c, tables, intra, codes[p], hdr[p])
    return codes, hdr


@pytest.mark.parametrize("name", ["gpt3_13b", "t5_770m", "wresnet_1b", "gpt3_175b", "gpt_1tp_1mbs", "gpt_wide_stages", "resnet_16gpus"])
def test_encode_and_fill_equal_the_python_code(name):
    w = WORKLOADS[name]
    cm = cost_model(w)
    batch = synth.make_plans(w, cm.tables, n_plans=12, seed_offset=2)
    configs = [batch.to_config(p, cm.tables) for p in range(12)]
    for intra in (False, True):
        native, (codes, hdr) = PlanBatch.from_configs(configs, cm.tables, intra), by_python(configs, cm.tables, intra)
        assert np.array_equal(native.codes, codes) and np.array_equal(native.hdr, hdr) and np.array_equal(codes, batch.codes)
    rec = emu_score(cm.tables, batch, breakdown=True)[4]
    s = cm.settings
    for p, c in enumerate(configs):
        other = copy.deepcopy(c)
        assert load_objects().fill(c, rec[p], s.memory_limit, s.memory_main_params, s.memory_optimizer, s.consider_reserved_space) is True
        other.stages = tuple(other.stages)              # (left to the Python code)
        assert load_objects().fill(other, rec[p], s.memory_limit, s.memory_main_params, s.memory_optimizer, s.consider_reserved_space) is False
        cm._fill_breakdown(other, rec[p])
        other.stages = list(other.stages)
        assert c == other and c.time_list and all(type(x) is float for x in c.time_list + c.memory_list + c.efficient_time_list)


def test_other_plan_objects_and_errors_take_the_python_code():
    w = odd_workloads()[2]
    tables = synth.make_tables(w)
    batch = synth.make_plans(w, tables, n_plans=6, seed_offset=1)
    good = [batch.to_config(p, tables) for p in range(6)]
    odd = copy.deepcopy(good)
    odd[1].stages[0].tp_size = tuple(odd[1].stages[0].tp_size)                 # not a list
    odd[3].stages[-1].algo = [np.int64(a) for a in odd[3].stages[-1].algo]      # not ints
    odd[4].stages[0].recompute_ops = [2 * r for r in odd[4].stages[0].recompute_ops]   # only 1 means recomputed
    got = PlanBatch.from_configs(odd, tables)
    want = PlanBatch.from_configs(good, tables)
    n = len(good[4].stages[0].ops)
    want.codes[4, :n] &= 0xF7
    assert np.array_equal(got.codes, want.codes) and np.array_equal(got.hdr, want.hdr)

    def change(**kw):
        c = copy.deepcopy(good[2])
        for k, v in kw.items():
            setattr(c if hasattr(c, k) else c.stages[0], k, v(getattr(c if hasattr(c, k) else c.stages[0], k)))
        return c
    bad = [(KeyError, change(micro_bs=lambda m: 3)), (ValueError, change(num_stages=lambda n: 17)), (ValueError, change(ops=lambda o: [])),
           (ValueError, change(tp_size=lambda t: [3] * len(t))), (ValueError, change(algo=lambda a: [9] * len(a))),
           (ValueError, change(ops=lambda o: o[:-1], tp_size=lambda t: t[:-1])), ((KeyError, ValueError), change(dp_size=lambda d: d[:1] + [2 * x for x in d[1:]])),
           (AttributeError, object())]
    for error, c in bad:
        with pytest.raises(error):
            PlanBatch.from_configs([good[0], c], tables)


def test_a_list_of_plans_is_filled_like_each_of_them():
    w = odd_workloads()[2]
    cm = cost_model(w)
    batch = synth.make_plans(w, cm.tables, n_plans=9, seed_offset=4)
    rec = emu_score(cm.tables, batch, breakdown=True)[4]
    one, all_ = ([batch.to_config(p, cm.tables) for p in range(9)] for _ in range(2))
    for p in (0, 4, 5, 8):
        one[p].stages = all_[p].stages = tuple(one[p].stages)        # (left to the Python code)
    for p, c in enumerate(one):
        cm._fill_breakdown(c, rec[p])
    cm._fill_all(all_, rec)
    assert one == all_ and all(c.time_list for c in all_)
    cm._fill_all([], rec[:0])


def test_plans_come_in_any_collection():
    w = odd_workloads()[2]
    cm = cost_model(w)
    batch = synth.make_plans(w, cm.tables, n_plans=5, seed_offset=4)
    configs = [batch.to_config(p, cm.tables) for p in range(5)]
    configs[2].stages[0].tp_size = tuple(configs[2].stages[0].tp_size)      # (left to the Python code)
    configs[3].stages = tuple(configs[3].stages)
    rec = emu_score(cm.tables, batch, breakdown=True)[4]
    for some in (dict(enumerate(configs)).values(), collections.deque(configs)):
        got = PlanBatch.from_configs(some, cm.tables)
        assert np.array_equal(got.codes, batch.codes) and np.array_equal(got.hdr, batch.hdr)
        cm._fill_all(some, rec)
        assert all(c.time_list for c in configs)
        for c in configs:
            c.time_list = []


class Changing:
    """A plan object (or stage) whose attribute `when` runs `what` each time it is read; `log` gets every read, and "gone" when the
    object is."""

    def __init__(self, of, when, what, log):
        self.__dict__["_in"] = (dict(vars(of)), when, what, log)

    def __getattr__(self, name):
        attributes, when, what, log = self.__dict__["_in"]
        log.append(name)
        if name == when:
            what()
        return attributes[name]

    def __setattr__(self, name, value):
        self.__dict__["_in"][3].append(name)

    def __del__(self):
        self.__dict__["_in"][3].append("gone")


READ_OF_STAGE = {"encode": ["ops", "tp_size", "dp_size", "algo", "recompute_ops"], "fill": ["num_gpus", "num_stages_behind", "recompute_ops"]}


@pytest.mark.parametrize("call", ["encode", "fill"])
@pytest.mark.parametrize("when", [0, 1, 2])
def test_objects_that_attribute_reads_drop_are_held(call, when):
    w = odd_workloads()[2]
    cm = cost_model(w)
    t, s = cm.tables, cm.settings
    batch = synth.make_plans(w, t, n_plans=40, seed_offset=4)
    rec = emu_score(t, batch, breakdown=True)[4]
    codes, hdr = np.empty((2, t.graph.num_ops), dtype=np.uint8), np.empty((2, 4), dtype=np.uint32)

    def run(configs):
        if call == "encode":
            return load_objects().encode(configs, 0, t.graph.num_ops, t.db.n_algo, s.num_gpus_per_node, False, *t.encode_luts, codes, hdr)
        return load_objects().fill_all(configs, rec[:2], 0, s.memory_limit, s.memory_main_params, s.memory_optimizer, True)
    p = next(p for p in range(40) if (batch.hdr[p, 0] & 0xff) > 2)
    # a stage that its own list drops: every attribute is read before it is gone, and the plan is left (its stages are others now)
    c, log = batch.to_config(p, t), []
    stages = c.stages
    read = READ_OF_STAGE[call]
    stages[0] = Changing(stages[0], read[when], stages.clear, log)
    assert run([c]) == 0
    assert log == read + ["gone"]
    # ... its last stage: nothing is left to refuse
    c, log = batch.to_config(p, t), []
    stages = c.stages
    stages[-1] = Changing(stages[-1], read[when], stages.clear, log)
    assert run([c]) == 1
    assert log == read + ["gone"]
    # a plan that the list of plans drops, and the plans behind it
    name = ["num_stages", "micro_bs", "stages"][when]
    log, configs = [], []
    configs[:] = [Changing(batch.to_config(p, t), name, configs.clear, log), batch.to_config(p, t)]
    assert run(configs) == 1
    assert log[-1] == "gone" and log.count("gone") == 1 and len(log) > 3
