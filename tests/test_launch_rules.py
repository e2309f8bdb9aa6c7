"""The host's launch rules (pippin_amd/csrc/launch_rules.hpp), without a device."""
import ctypes as C

import numpy as np
import pytest

from oracle import mjcf
from tests.emu.pyemu import EmuSim, _p, lib
from tests.scenes import COUPLED_SLIDERS

GRID, SPLIT = 0, 3


@pytest.mark.parametrize("kib,packed,asked,want", [
    (4, False, None, (4, GRID)), (16, False, None, (4, GRID)), (17, False, None, (2, GRID)),
    (33, False, None, (1, GRID)), (4, True, None, (1, SPLIT)), (33, True, None, (1, SPLIT)),
    # a number of envs per wavefront that is asked for, with or without room
    (4, False, b"2", (2, GRID)), (4, True, b"4", (4, GRID)), (4, True, b"1", (1, GRID)),
    (40, False, b"4", (4, GRID)), (41, False, b"4", (1, GRID)), (41, True, b"4", (1, SPLIT)),
    # and values that are not taken: the shape is as if nothing had been asked for
    (4, False, b"3", (4, GRID)), (4, True, b"3", (1, SPLIT)), (4, True, b"", (1, SPLIT)), (4, True, b"no", (1, SPLIT)),
    (4, True, b"-4", (1, SPLIT)), (4, True, b"0", (1, SPLIT)),
])
def test_the_shape_a_sim_starts_with(kib, packed, asked, want):
    k, sched = C.c_int(-1), C.c_int(-1)
    lib().emu_start_shape(kib * 1024, packed, 160 * 1024, asked, C.byref(k), C.byref(sched))
    assert (k.value, sched.value) == want


@pytest.mark.parametrize("envs", [1, 7, 1023, 1024, 1025, 5120, 8192, 16384])
@pytest.mark.parametrize("per_cu,cus", [(20, 256), (4, 256), (8, 64)])
def test_the_general_sweeps_fill_the_device(envs, per_cu, cus):
    """Every env of a batch may be left to them: a wavefront each, as far as the device holds them."""
    assert lib().emu_general_sweep_blocks(envs, per_cu, cus) == min(envs, per_cu * cus)


# candidates: grid, stealing and buckets of one kernel, the same of another, the split step
@pytest.mark.parametrize("times,want", [
    # the lowest median, wherever it is
    ([[9, 9, 9], [8, 8, 8], [9, 9, 9], [7, 7, 7], [6, 6, 6], [7, 7, 7], [8, 8, 8]], 4),
    ([[9, 9, 9], [8, 8, 8], [9, 9, 9], [7, 7, 7], [7, 7, 7], [7, 7, 7], [1, 1, 1]], 6),
    # buckets 3 % slower in every launch: told apart, so not taken
    ([[1.00, 1.01, 0.99], [2, 2, 2], [1.03, 1.04, 1.02], [2, 2, 2], [2, 2, 2], [2, 2, 2], [2, 2, 2]], 0),
    # buckets with a launch as fast: not told apart
    ([[1.00, 1.03, 0.99], [2, 2, 2], [1.02, 1.00, 1.04], [2, 2, 2], [2, 2, 2], [2, 2, 2], [2, 2, 2]], 2),
    # one slow launch of the other does not make buckets that are slower in every launch its equal
    ([[1.00, 5.00, 1.01], [2, 2, 2], [1.20, 1.21, 1.20], [2, 2, 2], [2, 2, 2], [2, 2, 2], [2, 2, 2]], 0),
    # only of the same kernel, and not instead of the split step
    ([[1.00, 1.00, 1.00], [2, 2, 2], [3, 3, 3], [2, 2, 2], [2, 2, 2], [0.9, 1.1, 1.1], [2, 2, 2]], 0),
    ([[2, 2, 2], [2, 2, 2], [0.9, 1.1, 1.1], [2, 2, 2], [2, 2, 2], [2, 2, 2], [1.00, 1.00, 1.00]], 6),
    # not timed
    ([[-1, -1, -1], [-1, -1, -1], [-1, -1, -1], [2, 2, 2], [-1] * 3, [-1] * 3, [-1] * 3], 3),
    ([[-1] * 3] * 7, -1),
])
def test_autotuning_keeps_what_its_trials_show(times, want):
    ms = np.array(times, dtype=np.float64)
    prefer = np.array([2, 2, 2, 5, 5, 5, -1], dtype=np.int32)
    assert lib().emu_tune_choice(_p(ms), _p(prefer), *ms.shape) == want


def test_trials_are_timed_alike():
    """One clock for every candidate of an autotuning; a grid launch outside of it stamps itself."""
    by_dispatch = lib().emu_timed_by_dispatch
    assert {by_dispatch(1, 1, grid) for grid in (0, 1)} == {0}
    assert by_dispatch(1, 0, 1) == 1
    assert {by_dispatch(0, trial, grid) for trial in (0, 1) for grid in (0, 1)} == {0}
    assert by_dispatch(1, 0, 0) == 0


@pytest.mark.parametrize("nblock,kib,envs,want", [
    (1, 10, 1, 1), (1, 10, 1024, 1), (1, 10, 1025, 2), (1, 10, 2048, 2), (1, 10, 2049, 4), (1, 10, 4096, 4),
    (1, 10, 16384, 4), (1, 33, 16384, 1), (1, 17, 4096, 2), (6, 10, 1, 1), (6, 10, 4096, 1), (2, 4, 16384, 1),
])
def test_envs_per_wavefront_of_the_learned_warm_start(nblock, kib, envs, want):
    """Under the split PGS step's shape by the range; else what the shape says."""
    rule = lib().emu_learned_envs_per_wave
    assert rule(1, 1, nblock, kib * 1024, 256, envs) == want
    for k in (1, 2, 4):
        assert rule(k, 0, nblock, kib * 1024, 256, envs) == k


_HINGES = ('<mujoco><compiler angle="radian"/><default><geom contype="0" conaffinity="0"/></default><worldbody>'
           '<body pos="0 0 1"><joint name="a" type="hinge" axis="0 1 0" {a}/><geom type="sphere" size=".1" pos=".2 0 0"/>'
           '<body pos=".4 0 0"><joint name="b" type="hinge" axis="0 1 0" {b}/><geom type="sphere" size=".1" pos=".2 0 0"/>'
           '</body></body><body pos="0 1 1"><joint name="c" type="hinge" axis="0 1 0" {c}/>'
           '<geom type="sphere" size=".1" pos=".2 0 0"/></body></worldbody>{eq}</mujoco>')
_LIM = 'limited="true" range="-1 1"'


@pytest.mark.parametrize("name,want", [("cartpole.xml", 0), ("pendulum.xml", 0), ("arm3d.xml", 0), ("box_drop.xml", 1), ("ant.xml", 1)])
def test_rows_of_the_assets_that_can_meet(assets, name, want):
    assert lib().emu_rows_can_meet(EmuSim(mjcf.load_file(assets / name), 1).h) == want


@pytest.mark.parametrize("a,b,c,eq,want", [
    ("", "", "", "", 0), (_LIM, "", "", "", 0), (_LIM, "", _LIM, "", 0), (_LIM, _LIM, "", "", 1),
    ("", "", "", "ab", 0), ("", "", "", "ac", 0), (_LIM, "", "", "ab", 1), ("", "", _LIM, "ab", 0), ("", "", _LIM, "ac", 1),
])
def test_limits_and_equalities_that_can_meet(a, b, c, eq, want):
    """More than one row on a dof block: a and b are one, c another."""
    eq = f'<equality><joint joint1="{eq[0]}" joint2="{eq[1]}"/></equality>' if eq else ""
    assert lib().emu_rows_can_meet(EmuSim(mjcf.load_string(_HINGES.format(a=a, b=b, c=c, eq=eq)), 1).h) == want
    assert lib().emu_rows_can_meet(EmuSim(mjcf.load_string(COUPLED_SLIDERS), 1).h) == 1
