"""The work a program has this library do, as cases that can be timed and compared.

A case names a workload (a model, its solver, how the program calls the library) and its
sizes. Four ways to call it:

  host     buffers in host memory, as a backend behind the `Physics` trait is driven: set the
           controls, step, get positions and velocities;
  step     state, controls and results resident on the GPU, as a training or planning loop holds
           them: put the envs back to the state the plan starts from, set one action, step it;
  rollout  the same with a sequence of controls, one per physics step, and qpos after each of them;
  poses    geom poses for a renderer on the GPU, for new positions on every call.

All arithmetic is float64 (poses are rounded to float32). Workloads on the GPU start each pass
from the same state, so that a pass is the same work whenever it is run.
"""
import os
import tempfile

import numpy as np
import torch

from pippin_amd.physics import HipPhysics, load_model
from pippin_amd.workloads import arm_env_params, arm_gripper_xml, random_pile_xml, tabletop_tumble

ASSETS = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pippin_amd", "assets")

# FP64 operations (+ - * / sqrt pow sin cos, one each) per physics step of one env, counted by the
# host engine's op-counting build over 32 envs once the bodies are in contact; the arm's without
# per-env draws, the tumble's taken from the piles'.
OPS = {
    ("cartpole", "newton"): 2.75e3,
    ("arm3d", "newton"): 6.33e3,
    ("ant", "newton"): 2.25e4, ("ant", "pgs"): 2.57e4,
    ("pile", "newton"): 5.29e4, ("pile", "pgs"): 2.06e5,
    ("pile_general", "newton"): 5.32e4, ("pile_general", "pgs"): 1.74e5,
    ("tumble", "newton"): 5.3e4, ("tumble", "pgs"): 1.8e5,
    ("arm", "newton"): 7.32e4,
}


def listed():
    return [
        # one env driven from the host, one physics step per control: an interactive session
        dict(name="cartpole_host_1", model="cartpole", solver="newton", call="host", envs=1, steps=1, tune=False),
        # an evaluation batch of odd size behind the trait, four substeps per action
        dict(name="ant_host_37", model="ant", solver="newton", call="host", envs=37, steps=4, tune=False),
        # the contact-free benchmark arm: hinges, a ball joint, a slide; implicit actuator terms
        dict(name="arm3d_rollout_1024", model="arm3d", solver="newton", call="rollout", envs=1024, steps=50, tune=False),
        # the rollout benchmark's batch: joint limits and ground contacts, a new control every step
        dict(name="ant_rollout_1024", model="ant", solver="newton", call="rollout", envs=1024, steps=25, tune=False),
        # the training loop: one action of four substeps over a large batch
        dict(name="ant_step_16384", model="ant", solver="newton", call="step", envs=16384, steps=4, tune=True),
        # the same model under the other solver
        dict(name="ant_pgs_step_4096", model="ant", solver="pgs", call="step", envs=4096, steps=4, tune=True),
        # tabletop piles of six free bodies, both solvers
        dict(name="pile_step_8192", model="pile", solver="newton", call="step", envs=8192, steps=4, tune=True),
        dict(name="pile_pgs_step_8192", model="pile", solver="pgs", call="step", envs=8192, steps=4, tune=True),
        # a ragged batch of piles whose cylinders meet every body (GJK/EPA narrow phase)
        dict(name="pile_general_step_1003", model="pile_general", solver="newton", call="step", envs=1003, steps=4,
             tune=False),
        # per-env object sets with hull wedges, every env with parameters of its own
        dict(name="tumble_step_768", model="tumble", solver="newton", call="step", envs=768, steps=4, tune=False),
        # a 7-DoF arm with a gripper and a cube on a table, per-env masses, sizes and frictions
        dict(name="arm_rollout_1024", model="arm", solver="newton", call="rollout", envs=1024, steps=10, tune=True),
        # poses of every geom for a renderer
        dict(name="ant_poses_8192", model="ant", solver="newton", call="poses", envs=8192, steps=1, tune=False),
    ]


def draw(rng):
    kind = rng.choice(["cartpole", "arm3d", "ant", "ant", "ant", "pile", "pile", "pile_general", "tumble", "arm"])
    solver = "newton" if kind in ("cartpole", "arm3d", "arm") else rng.choice(["newton", "pgs"])

    def envs(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    if kind in ("cartpole", "arm3d"):
        call = rng.choice(["host", "rollout", "step"])
        n, steps = envs(1, 8192), rng.randint(1, 20)
    elif kind == "ant":
        call = rng.choice(["host", "rollout", "step", "step", "poses"])
        n, steps = envs(1, 16384), rng.randint(1, 4)
    elif kind == "arm":
        call, n, steps = "rollout", envs(1, 1024), rng.randint(1, 8)
    elif kind == "tumble":
        call, n, steps = "step", envs(1, 512), rng.randint(1, 4)
    else:
        call, n, steps = "step", envs(1, 4096), rng.randint(1, 4)
    if call == "host":
        n = min(n, 4096)
    return dict(model=kind, solver=solver, call=call, envs=n, steps=1 if call == "poses" else steps,
                tune=call in ("step", "rollout") and rng.random() < 0.5)


# ---------------------------------------------------------------- models and starting states
_models = {}


def _arrays(kind):
    """The compiled model, read once per process."""
    if kind not in _models:
        if kind in ("cartpole", "arm3d", "ant"):
            _models[kind] = load_model(os.path.join(ASSETS, kind + ".xml"))
        elif kind in ("pile", "pile_general"):
            # six bodies; 19 and 11 contacts per env once they have dropped
            _models[kind] = load_model(random_pile_xml(29 if kind == "pile" else 18, kind == "pile_general"), is_xml=True)
        elif kind == "arm":
            _models[kind] = load_model(arm_gripper_xml(0), is_xml=True)
    return _models[kind]


def _shape_cache():
    """Where a program keeps its tuned launch shapes: a file of this process."""
    return os.path.join(tempfile.gettempdir(), "launch_shapes_%d" % os.getpid())


class _DeviceField:
    """The sim's own device buffer of a field, as torch.as_tensor takes it; the tensor keeps the sim alive."""

    def __init__(self, sim, field):
        self.sim = sim
        self.__cuda_array_interface__ = dict(shape=(sim.n, sim.width(field)), typestr="<f8", version=2,
                                             data=(sim.state_ptr(field), False))


class _DevicePoses:
    def __init__(self, sim, address):
        self.sim = sim
        self.__cuda_array_interface__ = dict(shape=(sim.n, sim.ngeom, 12), typestr="<f4", version=2,
                                             data=(address, False))


def _rng(seed):
    return np.random.default_rng(seed)


def _start_qpos(kind, qpos0, n, rng):
    """Positions an episode starts from."""
    q = np.tile(qpos0, (n, 1))
    if kind == "ant":
        q += rng.normal(0.0, 0.01, q.shape)
        q[:, 3:7] /= np.linalg.norm(q[:, 3:7], axis=1, keepdims=True)
    elif kind in ("pile", "pile_general"):
        for b in range(q.shape[1] // 7):
            q[:, 7 * b:7 * b + 2] += rng.normal(0.0, 0.005, (n, 2))
    elif kind == "cartpole":
        q += rng.normal(0.0, 0.1, q.shape)
    elif kind == "arm3d":
        q[:, :4] += rng.normal(0.0, 0.3, (n, 4))
        q[:, 8] += rng.normal(0.0, 0.05, n)
    return q


def _new_sim(kind, solver, n, rng):
    """A sim whose envs have their parameters and stand at the start of an episode."""
    if kind == "tumble":
        plan = tabletop_tumble(n, int(rng.integers(1 << 30)))
        if kind not in _models:
            _models[kind] = load_model(plan.xml, is_xml=True)
        # of the candidate pairs' many contacts an env meets a few dozen
        sim = HipPhysics(_models[kind], n, solver=solver, max_contacts=96)
        plan.apply(sim)
        return sim
    arrays = _arrays(kind)
    sim = HipPhysics(arrays, n, solver=solver)
    if kind == "arm":
        params, qpos0 = arm_env_params(arrays, n, int(rng.integers(1 << 30)))
        for name, gid, values in params:
            sim.set_param(name, gid, 0, n, np.ascontiguousarray(values))
        sim.set_param("qpos0", 0, 0, n, np.ascontiguousarray(qpos0))
        sim.reset(np.arange(n))
    else:
        sim.set("qpos", 0, n, _start_qpos(kind, np.asarray(arrays["qpos0"]), n, rng))
        if kind == "arm3d":
            sim.set("qvel", 0, n, rng.normal(0.0, 0.5, (n, sim.nv)))
        elif kind == "cartpole":
            sim.set("qvel", 0, n, rng.normal(0.0, 0.3, (n, sim.nv)))
    return sim


# untimed physics steps from the start of the episode to the state a pass works on: the ant walks,
# the objects have dropped onto each other
_BEFORE = {"cartpole": 0, "arm3d": 0, "ant": 240, "pile": 120, "pile_general": 120, "tumble": 200, "arm": 40}


def _controls(kind, nu, shape, gen):
    scale = {"ant": 1.0, "cartpole": 1.0, "arm3d": 0.5, "arm": 0.6}.get(kind, 1.0)
    c = (torch.rand((*shape, nu), generator=gen, dtype=torch.float64, device=gen.device) * 2 - 1) * scale
    if kind == "arm":
        c[..., -1] *= 0.05  # the gripper's opening in metres
    return c


def _pre_roll(sim, kind, steps, tune, gen):
    """Step to the state the case works on; the launch shape is tuned on the way, as a long run does."""
    n, nu = sim.n, sim.nu
    left = _BEFORE[kind]

    def chunk(k):
        if nu:
            c = _controls(kind, nu, (n,), gen)
            torch.cuda.current_stream().synchronize()
            sim.set_device("ctrl", 0, n, c.data_ptr())
        sim.step(0, n, k)

    while left > 0:
        k = min(10, left)
        chunk(k)
        left -= k
    if tune:
        sim.autotune(rounds=2, cache_path=_shape_cache())
        for _ in range(200):
            if not sim.autotune_pending():
                break
            chunk(min(steps, 4))


def prepare(case, seed):
    kind, call, n, steps = case["model"], case["call"], case["envs"], case["steps"]
    rng = _rng(seed)
    sim = _new_sim(kind, case["solver"], n, rng)
    if call == "host":
        # host-driven sessions start with the episode; a bank of actions stands for a policy's output
        return dict(call=call, sim=sim, steps=steps, at=0, ctrl=_host_controls(kind, sim.nu, n, rng))
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    if call == "poses":
        poses = [torch.as_tensor(_start_qpos(kind, np.asarray(_arrays(kind)["qpos0"]), n, rng), device="cuda")
                 for _ in range(2)]
        stream = torch.cuda.ExternalStream(sim.L.pippin_hip_stream(sim.h))
        qpos = torch.as_tensor(_DeviceField(sim, "qpos"), device="cuda")
        torch.cuda.synchronize()
        return dict(call=call, sim=sim, at=0, poses=poses, stream=stream, qpos=qpos)
    _pre_roll(sim, kind, steps, case["tune"], gen)
    st = dict(call=call, sim=sim, steps=steps)
    st["stream"] = torch.cuda.ExternalStream(sim.L.pippin_hip_stream(sim.h))
    st["qpos"] = torch.as_tensor(_DeviceField(sim, "qpos"), device="cuda")
    st["qvel"] = torch.as_tensor(_DeviceField(sim, "qvel"), device="cuda")
    st["qpos_start"], st["qvel_start"] = st["qpos"].clone(), st["qvel"].clone()
    if call == "rollout":
        st["ctrl"] = _controls(kind, sim.nu, (n, steps), gen)
        st["out"] = torch.empty((n, steps, sim.nq), dtype=torch.float64, device="cuda")
    elif sim.nu:
        st["ctrl"] = _controls(kind, sim.nu, (n,), gen)
    torch.cuda.synchronize()
    return st


def _host_controls(kind, nu, n, rng):
    return rng.uniform(-1.0, 1.0, (16, n, nu)) * (0.5 if kind == "arm3d" else 1.0)


def run(st):
    sim, call = st["sim"], st["call"]
    if call == "host":
        sim.set("ctrl", 0, sim.n, st["ctrl"][st["at"] % len(st["ctrl"])])
        st["at"] += 1
        sim.step(0, sim.n, st["steps"])
        return {"qpos": sim.get("qpos"), "qvel": sim.get("qvel")}
    if call == "poses":
        with torch.cuda.stream(st["stream"]):
            st["qpos"].copy_(st["poses"][st["at"] % 2])
        st["at"] += 1
        geoms, _ = sim.poses_device()
        return {"geoms": torch.as_tensor(_DevicePoses(sim, geoms), device="cuda")}
    with torch.cuda.stream(st["stream"]):
        st["qpos"].copy_(st["qpos_start"])
    sim.set_device("qvel", 0, sim.n, st["qvel_start"].data_ptr())
    if call == "rollout":
        sim.rollout_device(st["ctrl"].data_ptr(), st["out"].data_ptr(), st["steps"])
        return {"qpos": st["out"], "qvel": st["qvel"]}
    if "ctrl" in st:
        sim.set_device("ctrl", 0, sim.n, st["ctrl"].data_ptr())
    sim.step(0, sim.n, st["steps"])
    return {"qpos": st["qpos"], "qvel": st["qvel"]}


# ---------------------------------------------------------------- work, tolerance, reference values
_SIZES = {"cartpole": (3, 3, 2, 4), "arm3d": (9, 8, 4, 6), "ant": (15, 14, 8, 14), "pile": (42, 36, 0, 7),
          "pile_general": (42, 36, 0, 7), "tumble": (42, 36, 0, 31), "arm": (16, 15, 8, 13)}  # nq, nv, nu, ngeom


def work(case):
    nq, nv, nu, ng = _SIZES[case["model"]]
    n, steps = case["envs"], case["steps"]
    if case["call"] == "poses":
        # positions in, 12 float32 values per geom out; a rotation and a translation per geom and joint
        return {"bytes": n * (8 * nq + 48 * ng), "flops": n * 150.0 * ng}
    # positions, velocities and the warm start in and out, controls in, rolled-out positions out
    per_env = 8 * (2 * (nq + 2 * nv) + nu)
    if case["call"] == "rollout":
        per_env += 8 * steps * (nq + nu) - 8 * nu
    return {"bytes": n * per_env, "flops": n * steps * OPS[case["model"], case["solver"]]}


def tolerance(case):
    """float64 throughout. Sums in another order move the pile's positions by about 1e-15 in one step
    and 2e-13 after 200 (row-by-row Hessian against the matrix cores'). Contacts that come and go
    amplify that over the steps of a pass, above all in single velocities, and the solvers stop by a
    rule (Newton's gradient, PGS's largest change of a sweep) that another rounding can meet one
    iteration earlier or later."""
    if case["call"] == "poses":
        return {"rel": 2e-7, "max": 1e-6}  # float32 results
    if case["model"] in ("cartpole", "arm3d"):
        return {"rel": 1e-12, "max": 1e-10}
    return {"rel": 1e-9, "max": 1e-6}


def exact(case, seed):
    """The cart with its two poles in closed form (no contacts: a step is one linear solve) and the
    geom poses by forward kinematics. The workloads with contacts and the ball joint have no such
    value: what a step computes there is the solver's own iteration."""
    if case["call"] == "poses" and case["model"] == "ant":
        return _exact_poses(case, seed)
    if case["model"] == "cartpole" and case["call"] in ("host", "rollout", "step"):
        return _exact_cartpole(case, seed)
    return None


def _exact_cartpole(case, seed):
    a = _arrays("cartpole")
    n, steps, call = case["envs"], case["steps"], case["call"]
    rng = _rng(seed)
    q = _start_qpos("cartpole", np.asarray(a["qpos0"]), n, rng)
    v = rng.normal(0.0, 0.3, (n, 3))
    if call == "host":
        ctrl = np.repeat(_host_controls("cartpole", 2, n, rng)[0][:, None], steps, axis=1)
    else:
        if case["tune"] and case["solver"]:
            return None  # the tuning trials step the envs first, as many times as there are shapes
        gen = torch.Generator(device="cuda").manual_seed(int(seed))
        if call == "rollout":
            ctrl = _controls("cartpole", 2, (n, steps), gen).cpu().numpy()
        else:
            ctrl = np.repeat(_controls("cartpole", 2, (n,), gen).cpu().numpy()[:, None], steps, axis=1)
    out = []
    for t in range(steps):
        q, v = _cartpole_step(a, q, v, ctrl[:, t])
        out.append(q)
    return {"qpos": np.stack(out, axis=1) if call == "rollout" else q, "qvel": v}


def _cartpole_step(a, q, v, u):
    """One semi-implicit Euler step of the slide and the two hinges about y, planar (x, z)."""
    mass, ipos = np.asarray(a["body_mass"]), np.asarray(a["body_ipos"]).reshape(-1, 3)
    iyy = np.asarray(a["body_inertia"]).reshape(-1, 3, 3)[:, 1, 1]
    arm, damp = np.asarray(a["dof_armature"]), np.asarray(a["dof_damping"])
    q0, h = np.asarray(a["qpos0"]), float(a["timestep"])
    g = float(np.asarray(a["gravity"])[2])
    n = len(q)
    link = np.asarray(a["body_pos"]).reshape(-1, 3)[3]  # the second pole's hinge in the first pole
    th = np.cumsum(np.stack([np.zeros(n), q[:, 1] - q0[1], q[:, 2] - q0[2]], axis=1), axis=1)
    om = np.cumsum(np.stack([np.zeros(n), v[:, 1], v[:, 2]], axis=1), axis=1)

    def arm_of(r, i):  # body vector r at angle th_i, and its derivative by that angle (rotation about +y)
        c, s = np.cos(th[:, i]), np.sin(th[:, i])
        return np.stack([c * r[0] + s * r[2], -s * r[0] + c * r[2]], axis=1)

    def turned(w):  # d/dtheta of a vector that turns about +y
        return np.stack([w[:, 1], -w[:, 0]], axis=1)

    M, bias = np.zeros((n, 3, 3)), np.zeros((n, 3))
    for b in range(3):  # cart, first pole, second pole
        r = arm_of(ipos[b + 1], b)
        J = np.zeros((n, 2, 3))
        J[:, 0, 0] = 1.0
        acc = np.zeros((n, 2))  # acceleration at zero joint accelerations
        if b >= 1:
            first = r if b == 1 else arm_of(link, 1)
            J[:, :, 1] += turned(first)
            acc -= first * om[:, 1:2] ** 2
        if b == 2:
            J[:, :, 1] += turned(r)
            J[:, :, 2] += turned(r)
            acc -= r * om[:, 2:3] ** 2
        w = np.array([0.0, float(b >= 1), float(b >= 2)])
        M += mass[b + 1] * np.einsum("nak,nal->nkl", J, J) + iyy[b + 1] * np.outer(w, w)
        acc[:, 1] -= g
        bias += mass[b + 1] * np.einsum("nak,na->nk", J, acc)
    M += np.diag(arm)
    lo, hi = np.asarray(a["actuator_ctrlrange"]).reshape(-1, 2).T
    lim = np.asarray(a["actuator_ctrllimited"]) != 0
    u = np.where(lim, np.clip(u, lo, hi), u)
    gear, gain = np.asarray(a["actuator_gear"]), np.asarray(a["actuator_gain"])
    bia = np.asarray(a["actuator_bias"]).reshape(-1, 3)
    f = -damp * v - bias
    for i, k in enumerate((0, 2)):  # the motor on the slide, the position actuator on the second hinge
        f[:, k] += gear[i] * (gain[i] * u[:, i] + bia[i, 0] + bia[i, 1] * gear[i] * q[:, k]
                              + bia[i, 2] * gear[i] * v[:, k])
    qacc = np.linalg.solve(M + h * np.diag(damp), f[:, :, None])[:, :, 0]
    v = v + h * qacc
    return q + h * v, v


def _mat(q):
    q = q / np.linalg.norm(q, axis=-1, keepdims=True)
    w, x, y, z = np.moveaxis(q, -1, 0)
    return np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                     2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                     2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], axis=-1).reshape(*w.shape, 3, 3)


def _turn(axis, angle):
    half = 0.5 * angle[:, None]
    return _mat(np.concatenate([np.cos(half), np.sin(half) * axis], axis=1))


def _exact_poses(case, seed):
    a, n = _arrays("ant"), case["envs"]
    q0, rng = np.asarray(a["qpos0"]), _rng(seed)
    _start_qpos("ant", q0, n, rng)  # where the sim starts
    q = _start_qpos("ant", q0, n, rng)  # the first set that prepare() draws for the passes
    three = lambda k: np.asarray(a[k]).reshape(-1, 3)  # noqa: E731
    pos, rot = [np.zeros((n, 3))], [np.tile(np.eye(3), (n, 1, 1))]
    for b in range(1, int(a["nbody"])):
        p = int(a["body_parent"][b])
        x = pos[p] + rot[p] @ three("body_pos")[b]
        r = rot[p] @ _mat(np.asarray(a["body_quat"]).reshape(-1, 4)[b])
        for j in range(int(a["body_jntadr"][b]), int(a["body_jntadr"][b]) + int(a["body_jntnum"][b])):
            k = int(a["jnt_qposadr"][j])
            if int(a["jnt_type"][j]) == 0:  # free
                x, r = q[:, k:k + 3], _mat(q[:, k + 3:k + 7])
            else:  # hinge
                anchor = x + r @ three("jnt_pos")[j]
                r = r @ _turn(np.tile(three("jnt_axis")[j], (n, 1)), q[:, k] - q0[k])
                x = anchor - r @ three("jnt_pos")[j]
        pos.append(x)
        rot.append(r)
    out = np.zeros((n, int(a["ngeom"]), 12))
    for g in range(int(a["ngeom"])):
        b = int(a["geom_body"][g])
        out[:, g, :3] = pos[b] + rot[b] @ three("geom_pos")[g]
        out[:, g, 3:] = (rot[b] @ _mat(np.asarray(a["geom_quat"]).reshape(-1, 4)[g])).reshape(n, 9)
    return {"geoms": out}
