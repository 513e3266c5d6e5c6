"""check_recompute in one launch (superscaler_amd/csrc/ace_recompute.h) where its division of the work changes: workgroups of one wavefront
(what LDS leaves room for where every op has a type of its own), stages of more segments and of more types than a wavefront has lanes."""
import ctypes
import dataclasses

import numpy as np
import pytest

from superscaler_amd import synth
from superscaler_amd.recompute import update_recompute_arrays
from tests.helpers import emu_lib
from tests.test_recompute_kernel import cost_model, emu_recompute, limits
from tests.test_small_batches import WORKLOADS

#: 96 layers in one stage, a segment each; 134 types in one or two stages
LONG = {"gpt3_1_3b": dict(num_layers=96, pp_choices=[1]), "wresnet_1b": dict(pp_choices=[1, 2])}


def models(name, emu=True):
    w = dataclasses.replace(WORKLOADS[name], **LONG.get(name, {}))
    cm = cost_model(w, emu=emu)
    return cm, synth.make_plans(w, cm.tables, n_plans=12, seed_offset=4)


@pytest.mark.parametrize("lds", [0, 160 * 1024])
@pytest.mark.parametrize("name", ["gpt3_1_3b", "wresnet_1b", "gpt_16ops", "t5_1layer"])
def test_one_and_two_wavefronts_on_the_cpu(name, lds):
    cm, batch = models(name)
    room = ctypes.c_uint32.in_dll(emu_lib(), "ace_emu_rc_lds")
    before, room.value = room.value, lds
    try:
        for limit in limits(cm, batch):
            cm.settings.memory_limit = limit
            codes, flags = emu_recompute(cm, batch)
            assert not flags.any() and np.array_equal(codes, update_recompute_arrays(cm, batch).codes)
    finally:
        room.value = before


@pytest.mark.parametrize("name", ["gpt3_1_3b", "wresnet_1b", "gpt_16ops"])
def test_arguments_that_say_no_groups_and_no_wavefronts(name):
    """A launch whose arguments leave both as they come, with LDS for as much as that needs: room for a group per op, one wavefront."""
    cm, batch = models(name)
    said = ctypes.c_int32.in_dll(emu_lib(), "ace_emu_rc_set")
    said.value = 0
    try:
        for limit in limits(cm, batch):
            cm.settings.memory_limit = limit
            codes, flags = emu_recompute(cm, batch)
            assert not flags.any() and np.array_equal(codes, update_recompute_arrays(cm, batch).codes)
    finally:
        said.value = 1


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(LONG))
def test_long_stages_on_the_gpu(name):
    (cm, batch), (ref, _) = models(name, emu=False), models(name)
    for limit in limits(ref, batch):
        print(f"[case] {name} limit={limit}", flush=True)
        cm.settings.memory_limit = ref.settings.memory_limit = limit
        assert np.array_equal(cm.update_recompute_arrays(batch).codes, update_recompute_arrays(ref, batch).codes)


def many_types(emu=True):
    """3,974 ops, each of a type of its own: LDS has room for one wavefront's groups."""
    w = dataclasses.replace(WORKLOADS["wresnet_1b"], resnet_blocks=(3, 4, 486, 3), mbs_list=[1], gpus_per_node=1, num_gpus=4, pp_choices=[2, 4])
    cm = cost_model(w, emu=emu)
    assert len(set(cm.tables.graph.type_of_pos)) == cm.tables.graph.num_ops == 3974
    return cm, synth.make_plans(w, cm.tables, n_plans=9, seed_offset=4)


def test_so_many_types_take_one_wavefront():
    lib = emu_lib()
    assert lib.ace_emu_rc_waves(3974, 3974) == 1 and lib.ace_emu_rc_waves(3974, 40) == 2 and lib.ace_emu_rc_waves(134, 134) == 2
    cm, batch = many_types()
    for limit in limits(cm, batch):
        cm.settings.memory_limit = limit
        codes, flags = emu_recompute(cm, batch)
        assert not flags.any() and np.array_equal(codes, update_recompute_arrays(cm, batch).codes)


@pytest.mark.gpu
def test_one_wavefront_on_the_gpu():
    assert emu_lib().ace_emu_rc_waves(3974, 3974) == 1
    (cm, batch), (ref, _) = many_types(emu=False), many_types()
    chosen = 0
    for limit in limits(ref, batch):
        print(f"[case] 3974 types limit={limit}", flush=True)
        cm.settings.memory_limit = ref.settings.memory_limit = limit
        got = cm.update_recompute_arrays(batch).codes
        assert np.array_equal(got, update_recompute_arrays(ref, batch).codes)
        chosen += int((got & 8).any())
    assert chosen and cm.evaluator._rc_ready     # (the kernel took them)
