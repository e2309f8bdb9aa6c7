"""Branches of the step body that depend on a model's sizes, on the host emulation
against the oracle, bit for bit."""
import numpy as np
import pytest

from oracle import mjcf
from oracle.pyoracle import OracleSim
from tests.emu.pyemu import EmuSim
from tests.scenes import FEW_BODIES, few_bodies_xml


def _sliders(n, gap, integrator="Euler"):
    """n boxes on vertical slides over a plane: nv = n; with gap 0 they all overlap."""
    bodies = "".join(
        f'<body pos="{gap * i + 0.003 * i} {0.002 * i} {0.095 + 0.001 * i}"><joint type="slide" axis="0 0 1" damping="0.5"/>'
        f'<geom type="box" size="0.1 {0.1 + 0.001 * i} 0.1" mass="{1 + 0.1 * i}"/></body>' for i in range(n))
    return mjcf.load_string(f'<mujoco><option timestep="0.002" integrator="{integrator}"/><worldbody>'
                            f'<geom type="plane" size="5 5 0.1"/>{bodies}</worldbody></mujoco>')


# rows of one or two dofs: contact frames formed in place (no room beside the vectors), or kept
@pytest.mark.parametrize("solver", [0, 1])
@pytest.mark.parametrize("nv", [1, 2, 3])
@pytest.mark.parametrize("integrator", ["Euler", "implicitfast"])
def test_contact_rows_of_few_dofs(nv, solver, integrator):
    arr = {**_sliders(nv, 0.5, integrator), "solver_kind": solver}
    o, e = OracleSim(arr, 2), EmuSim(arr, 2)
    for t in range(40):
        for s in (o, e):
            s.step(0, 2, 1)
        assert np.array_equal(o.ncon(), e.ncon()), t
        assert np.array_equal(o.get("qpos"), e.get("qpos")), t
    assert o.ncon().min() >= 4 * nv


# more contacts than the list over the geom rotations holds (18 a geom), and fewer
@pytest.mark.parametrize("n", [4, 15])
def test_contact_copy_past_its_list(n):
    arr = _sliders(n, 0.0)
    o, e = OracleSim(arr, 1), EmuSim(arr, 1)
    for t in range(3):
        for s in (o, e):
            s.step(0, 1, 1)
        assert np.array_equal(o.ncon(), e.ncon()), t
        assert np.array_equal(o.get("qpos"), e.get("qpos")), t
    assert (o.ncon()[0] > 18 * int(arr["ngeom"])) == (n == 15), o.ncon()


@pytest.mark.parametrize("name", FEW_BODIES)
def test_islands_of_few_bodies(name):
    arr = mjcf.load_string(few_bodies_xml(name))
    o, e = OracleSim(arr, 2), EmuSim(arr, 2)
    q = o.get("qpos")
    q[1, ::7] += 0.001 * np.arange(q.shape[1] // 7)
    for s in (o, e):
        s.set("qpos", 0, 2, q)
    for t in range(80):
        for s in (o, e):
            s.step(0, 2, 1)
        assert np.array_equal(o.ncon(), e.ncon()), t
        assert np.array_equal(o.solver_iterations(), e.solver_iterations()), t
        assert np.array_equal(o.get("qpos"), e.get("qpos")), t
    assert o.ncon().min() >= len(name.split())
