"""The split PGS step with packed rows (kbody.hpp pgs_prepare_packed, pgs_sweeps_rows) on
the host emulation, against the oracle and against the general path, bit for bit."""
import numpy as np
import pytest

from oracle import mjcf
from oracle.pyoracle import OracleSim
from pippin_amd.workloads import arm_gripper_xml, random_pile_xml
from tests.emu.pyemu import EmuSim
from tests.scenes import COUPLED_SLIDERS, MULTIBODY_SCENES


def _model(name, assets):
    if name == "ant":
        arr = mjcf.load_file(assets / "ant.xml")  # one block of 14 dofs, limits
    elif name == "arm":
        arr = mjcf.load_string(arm_gripper_xml(3))  # blocks of 9 and 6 dofs, an equality, a tendon
    elif name == "sliders":
        arr = mjcf.load_string(COUPLED_SLIDERS)  # blocks of 1 dof, an equality across two
    elif name.startswith("seed"):
        arr = mjcf.load_string(random_pile_xml(int(name[4:])))  # blocks of 6 dofs
    else:
        xml = MULTIBODY_SCENES[name]
        arr = mjcf.load_file(assets / "box_drop.xml") if xml is None else mjcf.load_string(xml)
    return {**arr, "solver_kind": 1}


# capacities: every row packed; none; envs on either side of it
@pytest.mark.parametrize("cap", [1 << 20, 1, 900])
@pytest.mark.parametrize("name", ["ant", "arm", "sliders", "seed3", "seed11", "seed29", *sorted(MULTIBODY_SCENES)])
def test_split_step_equals_the_oracle(assets, name, cap):
    arr = _model(name, assets)
    n, steps = 3, 120
    o, e = OracleSim(arr, n), EmuSim(arr, n)
    rng = np.random.default_rng(5)
    packed = 0
    for t in range(steps):
        if int(arr["nu"]):
            c = rng.uniform(-1, 1, (n, int(arr["nu"]))) * (0.3 if name == "arm" else 1.0)
            for s in (o, e):
                s.set("ctrl", 0, n, c)
        o.step(0, n, 1)
        packed += e.step_split(0, n, 1, cap)
        assert np.array_equal(o.ncon(), e.ncon()), t
        assert np.array_equal(o.get("qpos"), e.get("qpos")), t
    assert np.array_equal(o.get("qvel"), e.get("qvel"))
    assert o.ncon().sum() > 0
    if cap == 1:
        assert packed == 0
    if cap == 1 << 20:
        assert packed > 0


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 1e200, 1e308])
@pytest.mark.parametrize("name,dof", [("seed29", 0), ("seed29", 8), ("seed29", 35), ("ant", 2), ("ant", 13), ("arm", 0),
                                      ("arm", 14), ("sliders", 1)])
def test_velocities_that_are_not_finite_spread_as_in_the_general_path(assets, value, name, dof):
    """A row's zeros outside its blocks still carry 0 * inf = NaN to the other blocks."""
    arr = _model(name, assets)
    n = 2
    a, b = EmuSim(arr, n), EmuSim(arr, n)
    for s in (a, b):
        s.step(0, n, 90)
    v = a.get("qvel")
    v[0, dof] = value
    for s in (a, b):
        s.set("qvel", 0, n, v)
    for _ in range(3):
        a.step(0, n, 1)
        b.step_split(0, n, 1)
        assert np.array_equal(a.get("qpos"), b.get("qpos"), equal_nan=True)
        assert np.array_equal(a.get("qvel"), b.get("qvel"), equal_nan=True)
