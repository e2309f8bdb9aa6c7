"""Branches of the step body that depend on a model's sizes, on the host emulation
against the oracle, bit for bit."""
import numpy as np
import pytest

from oracle import mjcf
from oracle.pyoracle import OracleSim
from pippin_amd.workloads import arm_gripper_xml, random_pile_xml
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


# an env on one 16-lane row (several envs per wavefront), or on the four of a wavefront of its own
@pytest.mark.parametrize("rows", [1, 4])
@pytest.mark.parametrize("name", FEW_BODIES)
def test_islands_of_few_bodies(name, rows):
    arr = mjcf.load_string(few_bodies_xml(name))
    o, e = OracleSim(arr, 2), EmuSim(arr, 2, rows)
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


@pytest.mark.parametrize("integrator", [0, 1])
@pytest.mark.parametrize("name", ["seed0", "seed3", "seed11", "seed29", "seed41", "arm", "ant", "pressed"])
def test_an_env_with_a_wavefront_of_its_own(assets, monkeypatch, name, integrator):
    """Blocks factored and islands solved side by side on four 16-lane rows, and
    constraint rows in the LDS past the layout, with the LDS full of NaN before a step."""
    monkeypatch.setenv("EMU_POISON_LDS", "1")
    if name.startswith("seed"):
        arr = mjcf.load_string(random_pile_xml(int(name[4:])))
    elif name == "arm":
        arr = mjcf.load_string(arm_gripper_xml(3))
    else:
        arr = mjcf.load_file(assets / "ant.xml")
    arr = {**arr, "integrator": integrator}
    n = 3
    o, e = OracleSim(arr, n), EmuSim(arr, n, rows=4)
    rng = np.random.default_rng(1)
    if name == "pressed":
        q = o.get("qpos")
        q[:, 2] = rng.uniform(0.05, 0.2, n)
        q[:, 7:] += rng.uniform(-0.8, 0.8, (n, 8))
        for s in (o, e):
            s.set("qpos", 0, n, q)
    rows = 0
    for t in range(25 if name in ("ant", "pressed") else 130):
        if int(arr["nu"]):
            c = rng.uniform(-0.3, 0.3, (n, int(arr["nu"])))
            for s in (o, e):
                s.set("ctrl", 0, n, c)
        for s in (o, e):
            s.step(0, n, 1)
        it, nr, _ = o.step_stats()
        rows = max(rows, int(nr.max()))
        assert np.array_equal(o.ncon(), e.ncon()), t
        assert np.array_equal(it, e.solver_iterations()), t
        assert np.array_equal(o.get("qpos"), e.get("qpos")), t
    assert np.array_equal(o.get("qvel"), e.get("qvel"))
    if name in ("pressed", "arm", "seed29"):
        assert rows > 32  # past the row block
