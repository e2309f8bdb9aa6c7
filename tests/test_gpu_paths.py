"""Host paths of get and set, and the split PGS step's launches (needs a GPU)."""
import sys

import numpy as np
import pytest

from oracle import mjcf
from oracle.pyoracle import OracleSim
from pippin_amd.physics import HipError, HipPhysics
from pippin_amd.workloads import arm_gripper_xml, random_pile_xml
from tests.scenes import COUPLED_SLIDERS

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("shared", [False, True])
def test_get_and_set_on_both_sides_of_the_staging(assets, shared):
    """Set calls of up to 256 KiB (2184 Ants' qpos) go through pinned staging,
    which several calls in a row fill, and get calls below 17 KiB (145 Ants);
    more is copied directly, as is every call after a device pointer to state
    was handed out."""
    n = 2300
    say("staging, shared", shared)
    arr = mjcf.load_file(assets / "ant.xml")
    g = HipPhysics(arr, n)
    if shared:
        assert g.state_ptr("qpos")
    rng = np.random.default_rng(3)
    want = g.get("qpos").copy()
    # one env, a block and a ragged end, the largest staged, the smallest direct,
    # and staged calls that do not fit beside each other
    for b, e in [(0, 1), (17, 120), (2299, 2300), (0, 2184), (5, 2190), (0, 1500), (300, 1800), (100, 101), (0, 2300),
                 (900, 2300)]:
        x = rng.normal(size=(e - b, 15))
        g.set("qpos", b, e, x)
        want[b:e] = x
        x[:] = np.nan  # the caller's array is free again when the call returns
    assert np.array_equal(g.get("qpos"), want)
    for b, e in [(0, 1), (2299, 2300), (0, 145), (0, 146), (7, 152), (0, 2184), (0, 2185), (116, 2300)]:
        assert np.array_equal(g.get("qpos", b, e), want[b:e]), (b, e)
    g.close()


@pytest.mark.parametrize("n", [1, 2300])
def test_get_and_set_refuse_a_null_buffer(assets, n):
    """Through the staging as on the direct path: an error code, and nothing is changed."""
    g = HipPhysics(mjcf.load_file(assets / "ant.xml"), n)
    before = g.get("qpos")
    for fn in (g.L.pippin_hip_get, g.L.pippin_hip_set):
        assert fn(g.h, 0, 0, n, None, n * g.nq) != 0
        assert fn(g.h, 0, 0, 0, None, 0) == 0  # no envs: nothing to copy
    assert np.array_equal(g.get("qpos"), before)


def pgs_model(name, assets):
    if name == "arm":
        arr = mjcf.load_string(arm_gripper_xml(3))
    elif name == "pile":
        arr = mjcf.load_string(random_pile_xml(29))
    elif name == "sliders":
        arr = mjcf.load_string(COUPLED_SLIDERS)
    else:
        arr = mjcf.load_file(assets / "ant.xml")
    return {**arr, "solver_kind": 1}


@pytest.mark.parametrize("n", [1, 5, 130])
@pytest.mark.parametrize("name", ["ant", "pressed", "arm", "pile", "sliders"])
def test_split_pgs_step_equals_the_oracle(assets, name, n):
    """The shape that PGS models start with, by the instances of the packed
    sweeps: one dof block with limits (16 entries, no equality); Ants pressed
    into the floor, some with more rows than the packed sweeps hold; two blocks
    with an equality and a tendon (16, equalities); blocks of six dofs (12);
    blocks of one dof with an equality across two (12, equalities)."""
    arr = pgs_model(name, assets)
    o, g = OracleSim(arr, n), HipPhysics(arr, n)
    say("split PGS", name, n, g.launch_shape())
    assert g.launch_shape()[2] == "pgs_split"
    rng = np.random.default_rng(1)
    q = o.get("qpos")
    if name == "pressed":
        q[:, 2] = rng.uniform(0.05, 0.35, n)
        q[:, 7:] += rng.uniform(-0.8, 0.8, (n, 8))
    elif name == "ant":
        q += 0.01 * rng.normal(size=q.shape)
    for s in (o, g):
        s.set("qpos", 0, n, q)
    nu = int(arr["nu"])
    rows = 0
    for t in range(20):
        if nu:
            c = rng.uniform(-0.3, 0.3, (n, nu))
            for s in (o, g):
                s.set("ctrl", 0, n, c)
        # uneven ranges, one and several steps a call
        for s in (o, g):
            s.step(0, (n + 1) // 2, 1)
            s.step(0, n, 3)
        rows = max(rows, int(o.step_stats()[1].max()))
        assert np.array_equal(o.ncon(), g.ncon()), t
        assert np.array_equal(o.get("qpos"), g.get("qpos")), t
        assert np.array_equal(o.get("qvel"), g.get("qvel")), t
    say("  rows up to", rows)
    g.close()


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 1e160, 1e200, 1e308])
@pytest.mark.parametrize("name,dofs", [("pile", (0, 8, 35)), ("ant", (2, 13)), ("arm", (0, 14)), ("sliders", (1,))])
def test_packed_sweeps_hand_over_what_is_not_finite(assets, name, dofs, value):
    """A velocity that is not finite before the sweeps, or that overflows at
    some row of one: the packed sweeps leave the env to the general form from
    that row on. Equal to the fused step bit for bit, also for the envs that
    share a wavefront and stay finite."""
    arr = pgs_model(name, assets)
    n, before, after = 10, 90, 3
    say("not finite", name, value)
    split, fused, calm = HipPhysics(arr, n), HipPhysics(arr, n), HipPhysics(arr, n)
    assert split.launch_shape()[2] == "pgs_split"
    fused.set_launch_shape(1, 0, "grid")
    sims = (split, fused, calm)
    rng = np.random.default_rng(6)
    q = split.get("qpos")
    if name == "pile":
        q[:, ::7] += rng.normal(0.0, 0.004, q[:, ::7].shape)
    for s in sims:
        s.set("qpos", 0, n, q)
        s.step(0, n, before)
    hit = [1 + 3 * i for i in range(len(dofs))]  # envs 1, 4, 7: each shares its wavefront with finite ones
    v = split.get("qvel")
    for e, d in zip(hit, dofs):
        v[e, d] = value
    for s in (split, fused):
        s.set("qvel", 0, n, v)
    for _ in range(after):
        for s in sims:
            s.step(0, n, 1)
        for f in ("qpos", "qvel", "qacc"):
            assert np.array_equal(split.get(f), fused.get(f), equal_nan=True), f
        for a, b in zip(split.get_history(), fused.get_history()):
            a, b = ((x if x.dtype.names is None else x["pos"]) for x in (a, b))
            assert np.array_equal(a, b, equal_nan=True)
    rest = [e for e in range(n) if e not in hit]
    assert np.isfinite(split.get("qpos")[rest]).all()
    assert np.array_equal(split.get("qpos")[rest], calm.get("qpos")[rest])
    for s in sims:
        s.close()


@pytest.mark.parametrize("steps", [1, 3])
def test_split_pgs_step_reports_an_env_that_cannot_be_stepped(assets, steps):
    """A contact capacity that a step of some call exceeds: that call fails, the
    env keeps its state and reports again, the others go on."""
    arr = {**mjcf.load_file(assets / "box_drop.xml"), "solver_kind": 1}
    n = 5
    g = HipPhysics(arr, n, max_contacts=2)  # a box resting on the plane makes 4
    assert g.launch_shape()[2] == "pgs_split"
    q = g.get("qpos")
    q[1:, [2, 9, 16]] += 5.0  # env 0's bodies land first
    g.set("qpos", 0, n, q)
    with pytest.raises(HipError, match=r"capacity exceeded \(env 0\)"):
        for _ in range(200):
            g.step(0, n, steps)
    frozen = g.get("qpos")
    g.step(1, n, steps)
    after = g.get("qpos")
    assert np.array_equal(after[0], frozen[0]) and not (after[1:] == frozen[1:]).all(axis=1).any()
    with pytest.raises(HipError, match="capacity"):
        g.step(0, 1, steps)
    assert np.array_equal(g.get("qpos")[0], frozen[0])
    g.reset([0])
    g.step(0, 1, steps)
    assert not np.array_equal(g.get("qpos")[0], frozen[0])
    g.close()


@pytest.mark.parametrize("asked,want", [("3", (1, 0, "pgs_split")), ("", (1, 0, "pgs_split")), ("2", (2, 0, "grid"))])
def test_envs_per_wavefront_from_the_environment(assets, monkeypatch, asked, want):
    """A value that is not taken leaves a PGS model with the split step."""
    monkeypatch.setenv("PIPPIN_HIP_ENVS_PER_WG", asked)
    g = HipPhysics({**mjcf.load_file(assets / "ant.xml"), "solver_kind": 1}, 2)
    assert g.launch_shape() == want
    g.close()


def test_learned_pgs_step_is_the_same_for_every_number_of_envs_per_wavefront(assets):
    """The split step's shape leaves the number to the range: 4 for these 2053
    Ants (a ragged last wavefront), 1 for the ranges that fit the device."""
    n = 2053
    arr = {**mjcf.load_file(assets / "ant.xml"), "solver_kind": 1}
    rng = np.random.default_rng(2)
    runs = []
    for shape in (None, (1, 0, "grid"), (2, 0, "grid"), (4, 0, "grid")):
        say("learned PGS", shape)
        g = HipPhysics(arr, n)
        if shape:
            g.set_launch_shape(*shape)
        if not runs:
            q = g.get("qpos")
            q[:, 2] = rng.uniform(0.3, 0.6, n)
            c = rng.uniform(-1, 1, (n, 8))
        g.set("qpos", 0, n, q)
        g.set("ctrl", 0, n, c)
        g.mlp_init(hidden=32, seed=5)
        g.mlp_mode(3)
        for b, e, k in [(0, n, 20), (7, 900, 3), (0, n, 2)]:
            g.step(b, e, k)
        runs.append([g.get("qpos"), g.get("qvel"), g.ncon(), g.solver_iterations()])
        g.close()
    assert runs[0][2].sum() > n
    for r in runs[1:]:
        for a, b in zip(runs[0], r):
            assert np.array_equal(a, b)


def test_pgs_models_whose_rows_cannot_meet_start_fused(assets):
    """One launch for all steps; masks that parameters open later bring the
    split step, a shape that was set stays."""
    arr = {**mjcf.load_file(assets / "cartpole.xml"), "solver_kind": 1}
    g = HipPhysics(arr, 2)
    assert g.launch_shape() == (4, 0, "grid")
    g.close()
    xml = (assets / "box_drop.xml").read_text().replace("<worldbody>",
                                                        '<default><geom contype="0" conaffinity="0"/></default><worldbody>', 1)
    arr = {**mjcf.load_string(xml), "solver_kind": 1}
    assert not np.any(arr["geom_contype"])
    g, fixed, o = HipPhysics(arr, 3), HipPhysics(arr, 3), OracleSim(arr, 3)
    first = g.launch_shape()
    assert first[2] == "grid"
    fixed.set_launch_shape(2, 0, "grid")
    for s in (g, fixed, o):
        s.step(0, 3, 2)
        for gi in range(int(arr["ngeom"])):
            s.set_param("geom_contype", gi, 0, 3, [0.0, 0.0, 0.0])
    assert g.launch_shape() == first
    for s in (g, fixed, o):
        for gi in range(int(arr["ngeom"])):
            s.set_param("geom_contype", gi, 1, 2, [1.0])
            s.set_param("geom_conaffinity", gi, 1, 2, [1.0])
    assert g.launch_shape() == (1, 0, "pgs_split") and fixed.launch_shape() == (2, 0, "grid")
    for _ in range(60):
        for s in (g, fixed, o):
            s.step(0, 3, 2)
        assert np.array_equal(g.get("qpos"), o.get("qpos"))
        assert np.array_equal(fixed.get("qpos"), o.get("qpos"))
    assert o.ncon()[1] > 0
    for s in (g, fixed):
        s.close()
