"""What this library is used for, as measurable cases.

A case is one call sequence of a program that uses the library: a batch of
worlds loaded, stepped and read back (the reference's own batch benchmark times
exactly that), a host-driven environment step, an on-device policy rollout with
or without its histories read back, and a PPO iteration (batch upload and
update). Models, world counts, step counts and widths are the repository's own
workloads (phyz_amd/workloads.py, bench.py); `draw` varies them.

    listed()            the cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) inputs and the handle a program keeps
    run(state)          one pass through the public entry points
    work(case)          bytes and operations a pass cannot do without
    tolerance(case)     how far another correct implementation may be off
    exact(case, seed)   the pass in plain torch, 64 bits
"""
import dataclasses
import math

import numpy as np
import torch

from phyz_amd import workloads as W
from phyz_amd.sim import BatchSim, from_control_loop, from_workload
from phyz_amd.train import AdamCfg, KlMode, NetDims, PpoUpdateCfg, SampleBatch, TrainPipeline

# Workload index of each model (phyz_amd/workloads.py) and the operations of
# one world-step (tests/golden/flops_per_world_step.json).
MODELS = {"double_pendulum": (1, 71), "chain7": (2, 1899), "ant": (3, 3503), "humanoid": (4, 8643),
          "hand": (5, 5065), "ant_terrain_impulse": (6, 17770), "mjcf_ant": (7, 5899),
          "mjcf_humanoid": (8, 8713), "mjcf_shadow_hand": (9, 8509)}


def listed():
    return [
        # A planner's inner loop on the README model: a few candidate states
        # rolled a short horizon. Call and transfer latency is all there is.
        {"name": "pendulum_plan", "kind": "span", "model": "double_pendulum", "dtype": "f64", "worlds": 96, "steps": 25},
        # The headline span: the 7-link chain, 65536 worlds, 20 steps.
        {"name": "chain_short", "kind": "span", "model": "chain7", "dtype": "f32", "worlds": 65536, "steps": 20},
        # The chain in double precision over a long span (system identification).
        {"name": "chain_long_f64", "kind": "span", "model": "chain7", "dtype": "f64", "worlds": 65536, "steps": 1000},
        # An odd, half-filled batch on one GPU of several (a share of a larger job).
        {"name": "chain_odd", "kind": "span", "model": "chain7", "dtype": "f32", "worlds": 12345, "steps": 200},
        # The quadruped at its benchmark batch, with contact.
        {"name": "ant_large", "kind": "span", "model": "ant", "dtype": "f32", "worlds": 131072, "steps": 100},
        # Humanoid-scale tree with contact.
        {"name": "humanoid", "kind": "span", "model": "humanoid", "dtype": "f32", "worlds": 32768, "steps": 100},
        # Dexterous hand under PD targets, double precision.
        {"name": "hand_f64", "kind": "span", "model": "hand", "dtype": "f64", "worlds": 16384, "steps": 200},
        # Rough terrain with the impulse solver.
        {"name": "terrain", "kind": "span", "model": "ant_terrain_impulse", "dtype": "f32", "worlds": 32768, "steps": 20},
        # A host-driven environment step: new servo targets, a few physics
        # steps, states and contact rows back to the learner on the host.
        {"name": "env_step", "kind": "env", "dtype": "f32", "worlds": 8192, "every": 5},
        # Evaluating a policy on the device at 250 Hz: the whole rollout, then final states.
        {"name": "policy_eval", "kind": "rollout", "dtype": "f32", "worlds": 131072, "hidden": 256, "control": 25,
         "every": 2, "history": False},
        # A collector's iteration: rollout, then every history row to the host.
        {"name": "collect", "kind": "rollout", "dtype": "f32", "worlds": 4096, "hidden": 256, "control": 20, "every": 5,
         "history": True},
        # A learner's iteration: the batch uploaded, four epochs of updates.
        {"name": "ppo", "kind": "ppo", "rows": 131072, "actor_in": 55, "critic_in": 67, "hidden": 64, "act": 22,
         "minibatch": 4096, "epochs": 4},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["span", "span", "span", "span", "env", "rollout", "rollout", "ppo"])
    if kind == "span":
        model = rng.choice(list(MODELS))
        both = model in ("chain7", "humanoid", "mjcf_humanoid", "mjcf_shadow_hand")
        dtype = rng.choice(["f32", "f64"]) if both else "f64" if model in ("double_pendulum", "hand") else "f32"
        # No more than the listed cases of the model's size: worlds first, then
        # steps within a budget of world-steps x operations.
        worlds = _log(rng, 64, {"double_pendulum": 65536, "chain7": 131072, "ant": 131072,
                                "mjcf_ant": 131072}.get(model, 32768))
        most = min(1000, int(1.0e11 / (worlds * MODELS[model][1])))
        if dtype == "f32":  # the tolerances are stated for these spans: rounding grows with the steps
            most = min(most, {"chain7": 200, "ant_terrain_impulse": 20}.get(model, 100))
        return {"kind": "span", "model": model, "dtype": dtype, "worlds": worlds, "steps": _log(rng, 1, max(2, most))}
    if kind == "env":
        return {"kind": "env", "dtype": "f32", "worlds": _log(rng, 16, 65536), "every": rng.randint(1, 10)}
    if kind == "rollout":
        history = rng.random() < 0.5
        worlds = _log(rng, 64, 8192 if history else 131072)
        return {"kind": "rollout", "dtype": "f32", "worlds": worlds, "hidden": rng.choice([64, 256]),
                "control": rng.randint(1, 20), "every": rng.randint(1, 5), "history": history}
    hidden = rng.choice([64, 64, 256])
    rows = _log(rng, 512, 131072)
    act = rng.randint(1, 32)
    return {"kind": "ppo", "rows": rows, "actor_in": rng.randint(8, 80), "critic_in": rng.randint(8, 80), "hidden": hidden,
            "act": act, "minibatch": min(rows, _log(rng, 128, 8192 if hidden == 64 else 2048)) if rows <= 32768
            else _log(rng, 2048, 8192), "epochs": rng.randint(1, 3)}


# ── inputs ───────────────────────────────────────────────────────────────────
def _single(case, *arrays):
    """The values as the case's precision holds them (inputs a program in that
    precision has), carried in f64 rows as the entry points take them."""
    if case.get("dtype") == "f64":
        return [np.ascontiguousarray(a, dtype=np.float64) for a in arrays]
    return [np.ascontiguousarray(np.asarray(a, dtype=np.float32).astype(np.float64)) for a in arrays]


def _workload(case, seed):
    w = W.config(MODELS[case["model"]][0])
    noise = None if w.noise is None else dataclasses.replace(w.noise, seed=(w.noise.seed + 7919 * seed) & (2**63 - 1))
    return dataclasses.replace(w, nworld=case["worlds"], nsteps=case["steps"], noise=noise, init_seed=seed + 1000)


def _span_inputs(case, seed):
    w = _workload(case, seed)
    q, v, ctrl, targets = w.initial_state(case["worlds"])
    if w.impulse_sweeps > 0:
        q[:, 5] *= 0.8  # feet on or near the ground: the solver at work from the first step
    q, v, ctrl = _single(case, q, v, ctrl)
    return w, q, v, ctrl, None if targets is None else _single(case, targets)[0]


def _loop(case, seed):
    """The ant under its PD servos and policy; initial poses and targets from the seed."""
    cl = W.control_loop(case.get("hidden", 64))
    n = case["worlds"]
    rng = np.random.default_rng(seed + 2000)
    base = dataclasses.replace(cl.base, nworld=n, init_seed=seed + 1000)
    history = case.get("control", 1)
    cl = dataclasses.replace(cl, base=base, spec=dataclasses.replace(cl.spec, history_steps=history),
                             weights=_single(case, cl.weights * rng.uniform(0.9, 1.1, cl.weights.size))[0],
                             std=_single(case, cl.std)[0], seed=seed + 77)
    q, v, ctrl, _ = base.initial_state(n)
    if case.get("history", True):
        q[:, 5] = rng.uniform(0.3, 0.7, size=n)  # a collector's worlds: most feet touch or nearly touch
    q, v = _single(case, q, v)
    targets, = _single(case, cl.base_targets(n) + rng.uniform(-0.3, 0.3, size=(n, 8)))
    return cl, q, v, targets


def _ppo_inputs(case, seed):
    rng = np.random.default_rng(seed + 3000)
    n, ai, ci, h, act = case["rows"], case["actor_in"], case["critic_in"], case["hidden"], case["act"]
    f = lambda *s: rng.standard_normal(size=s, dtype=np.float32)  # noqa: E731

    def net(i, o):
        return np.concatenate([rng.normal(size=h * i) / math.sqrt(i), np.zeros(h), rng.normal(size=h * h) / math.sqrt(h),
                               np.zeros(h), 0.1 * rng.normal(size=o * h) / math.sqrt(h), np.zeros(o)])
    a0 = np.concatenate([net(ai, act), np.full(act, -0.7)])
    c0 = net(ci, 1)
    batch = SampleBatch(f(n, ai), f(n, ci), 0.5 * f(n, act), np.float32(-0.5 * act) + 0.4 * f(n), f(n), 2.0 * f(n))
    # The behaviour policy's log-probs: the sampled actions scored under a
    # policy near the current one, so that ratios lie around 1.
    act_z = batch.act / np.float32(math.exp(-0.7))
    batch.logp_old = (-0.5 * act_z.astype(np.float64) ** 2 + 0.7 - 0.5 * math.log(2 * math.pi)).sum(axis=1).astype(np.float32)
    orders = [rng.permutation(n).astype(np.uint32) for _ in range(case["epochs"])]
    cfg = PpoUpdateCfg(0.2, 0.003, 6.0, case["minibatch"], case["epochs"], float("inf"), float(act), KlMode.MINIBATCH)
    return a0, c0, batch, orders, cfg


# ── the passes ───────────────────────────────────────────────────────────────
def prepare(case, seed):
    kind = case["kind"]
    if kind == "span":
        w, q, v, ctrl, targets = _span_inputs(case, seed)
        sim = from_workload(w, case["dtype"], nworld=case["worlds"])
        sim.compile()
        return {"kind": kind, "case": case, "sim": sim, "q": q, "v": v, "ctrl": ctrl, "targets": targets,
                "contact": w.contact is not None}
    if kind == "env":
        cl, q, v, targets = _loop(case, seed)
        c = cl.base.contact
        sim = BatchSim(cl.base.model, case["worlds"], case["dtype"])
        sim.enable_ground_contact(c.ground_height, c.stiffness, c.damping, c.friction)
        sim.enable_pd_control(cl.pd)
        sim.load_states(q, v)
        sim.compile()
        return {"kind": kind, "case": case, "sim": sim, "targets": targets}
    if kind == "rollout":
        cl, q, v, _ = _loop(case, seed)
        sim = from_control_loop(cl, case["dtype"], nworld=case["worlds"])
        sim.compile()
        return {"kind": kind, "case": case, "sim": sim, "q": q, "v": v, "seed": cl.seed}
    a0, c0, batch, orders, cfg = _ppo_inputs(case, seed)
    pipe = TrainPipeline(NetDims(case["actor_in"], case["hidden"], case["act"]),
                         NetDims(case["critic_in"], case["hidden"], 1), case["rows"], case["minibatch"])
    pipe.set_adam(AdamCfg(), AdamCfg())
    return {"kind": kind, "case": case, "pipe": pipe, "a0": a0, "c0": c0, "batch": batch, "orders": orders, "cfg": cfg}


def run(state):
    case, kind = state["case"], state["kind"]
    if kind == "span":
        sim = state["sim"]
        if state["targets"] is not None:
            sim.set_position_targets(state["targets"])
        sim.load_states(state["q"], state["v"], state["ctrl"])
        sim.step_many(case["steps"])
        q, v = sim.readback_states()
        return {"q": q, "v": v}
    if kind == "env":
        sim = state["sim"]
        sim.set_position_targets(state["targets"])
        sim.step_many(case["every"])
        q, v = sim.readback_states()
        return {"q": q, "v": v, "contacts": sim.readback_contacts()}
    if kind == "rollout":
        sim, n = state["sim"], case["control"]
        sim.load_states(state["q"], state["v"])
        sim.seed_policy(state["seed"])
        sim.rollout(0, n, case["every"], record_states=case["history"])
        if not case["history"]:
            q, v = sim.readback_states()
            return {"q": q, "v": v, "targets": sim.readback_targets()}
        obs, out = sim.readback_policy_history(0, n)
        q, v = sim.readback_state_history(0, n)
        return {"obs": obs, "out": out, "q": q, "v": v}
    pipe = state["pipe"]
    pipe.set_actor_params(state["a0"])
    pipe.set_critic_params(state["c0"])
    pipe.upload_batch(case["rows"], state["batch"])
    stats = pipe.update(state["orders"], state["cfg"])
    return {"actor": pipe.actor_params(), "critic": pipe.critic_params(), "policy_loss": stats.policy_loss,
            "value_loss": stats.value_loss, "kl": stats.kl}


def work(case):
    """Bytes: the host rows in and out, 8 bytes a value as the entry points take
    them (4 in a PPO batch). Operations: the frozen count per world-step, the
    MLP's multiply-adds, and forward plus backward of the update."""
    kind = case["kind"]
    if kind == "span":
        w = _workload(case, 0)
        nq, nv, nc = w.model.nq, w.model.nv, w.model.nctrl()
        npd = 0 if w.pd is None else len(w.pd)
        n = case["worlds"]
        return {"bytes": 8.0 * n * (2 * nq + 2 * nv + nc + npd), "flops": float(n) * case["steps"] * MODELS[case["model"]][1]}
    if kind == "env":
        n = case["worlds"]
        return {"bytes": 8.0 * n * (8 + 28 + 9 * 8), "flops": float(n) * case["every"] * 3503}
    if kind == "rollout":
        n, c, h = case["worlds"], case["control"], case["hidden"]
        back = c * (29 + 9 + 28) if case["history"] else 28 + 8
        return {"bytes": 8.0 * n * (28 + back), "flops": float(n) * c * (case["every"] * 3503 + 2 * (29 * h + h * h + 8 * h))}
    n, h = case["rows"], case["hidden"]
    f = 0.0
    for i, o in ((case["actor_in"], case["act"]), (case["critic_in"], 1)):
        f += 2.0 * n * (2 * (i * h + h * h + h * o) + o * h + h * h)
    params = 2 * h * h + h * (case["actor_in"] + case["critic_in"] + case["act"] + 1)
    return {"bytes": 4.0 * n * (case["actor_in"] + case["critic_in"] + case["act"] + 3 + case["epochs"]) + 32.0 * params,
            "flops": f * case["epochs"]}


def tolerance(case):
    """About four times what the same pass shows when its inputs (or the policy's
    weights) move by one rounding, over three seeds: (rel, max) measured
      f64 spans     chain 1000 steps 1.2e-10, 6e-8; contact-free trees 200 steps 1e-15, 7e-14
      f32 chain     3.6e-7, 9e-6 (200 steps; 7e-6 rel against 64 bits)
      f32 contact   humanoid 8e-5, 6e-2 (100 steps), terrain 6e-6, 3e-3 (20 steps): a foot that
                    touches one step earlier in a few worlds moves those worlds by far more
      env           1.2e-6, 8e-5 in 5 steps without such a foot; stated as the f32 contact spans
      rollouts      2.2e-4, 0.22 (feet touching down during the rollout)
      ppo           4e-8; 6e-4, 3e-3 where one row lies on the clip boundary and its gradient
                    switches on or off
    """
    kind = case["kind"]
    if kind == "ppo":
        return {"rel": 2.5e-3, "max": 0.012}
    if kind == "rollout":
        return {"rel": 1e-3, "max": 0.9}
    if case["dtype"] == "f64":
        return {"rel": 5e-10, "max": 2.4e-7}
    if case["model"] == "chain7":
        return {"rel": 2.8e-5, "max": 2e-3}
    return {"rel": 4e-4, "max": 0.3}


# ── 64-bit answers in plain torch ────────────────────────────────────────────
# Body-frame spatial vectors [angular, linear] with a leading world axis, the
# articulated-body recursion with dense 6 x 6 matrices.
def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _t(a):
    return torch.as_tensor(np.asarray(a, dtype=np.float64), device=_dev())


def _skew(v):
    z = torch.zeros_like(v[..., 0])
    return torch.stack([torch.stack([z, -v[..., 2], v[..., 1]], -1), torch.stack([v[..., 2], z, -v[..., 0]], -1),
                        torch.stack([-v[..., 1], v[..., 0], z], -1)], -2)


def _cross(a, b):
    a, b = torch.broadcast_tensors(a, b)
    return torch.linalg.cross(a, b)


def _mv(m, v):
    return (m * v.unsqueeze(-2)).sum(-1)


def _mtv(m, v):
    return (m * v.unsqueeze(-1)).sum(-2)


def _dot(a, b):
    return (a * b).sum(-1)


def _quat_exp(w):
    a = w.norm(dim=-1, keepdim=True)
    f = torch.where(a < 2.3e-16, torch.full_like(a, 0.5), torch.sin(0.5 * a) / a.clamp_min(1e-300))
    return torch.cat([torch.cos(0.5 * a), w * f], -1)


def _quat_mul(a, b):
    w, u, x, y = a[..., :1], a[..., 1:], b[..., :1], b[..., 1:]
    return torch.cat([w * x - _dot(u, y).unsqueeze(-1), w * y + x * u + _cross(u, y)], -1)


def _quat_log(q):
    u = q[..., 1:]
    n = u.norm(dim=-1, keepdim=True)
    return torch.where(n < 2.3e-16, 2.0 * u, u * (2.0 * torch.atan2(n, q[..., :1]) / n.clamp_min(1e-300)))


def _quat_mat(q):
    s = _skew(q[..., 1:])
    return torch.eye(3, dtype=q.dtype, device=q.device) + 2.0 * q[..., :1].unsqueeze(-1) * s + 2.0 * (s @ s)


class _Stream:
    """Per-world xorshift64 seeded by SplitMix64 of (seed, world)."""

    def __init__(self, seed, n):
        with np.errstate(over="ignore"):
            z = np.uint64(seed) + np.uint64(0x9E3779B97F4A7C15) * np.arange(1, n + 1, dtype=np.uint64)
            z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
            z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
            z = z ^ (z >> np.uint64(31))
        z[z == 0] = 1
        self.s = torch.as_tensor(z.view(np.int64).copy(), device=_dev())

    def uniform(self):
        x = self.s
        x = x ^ (x << 13)
        x = x ^ ((x >> 7) & ((1 << 57) - 1))
        x = x ^ (x << 17)
        self.s = x
        return ((x >> 11) & ((1 << 53) - 1)).double() * 2.0**-53

    def normal(self):
        u1, u2 = self.uniform(), self.uniform()
        return torch.sqrt(-2.0 * torch.log(u1.clamp_min(1e-300))) * torch.cos(2.0 * math.pi * u2)


class _Bodies:
    """The model's numbers and one world batch's dynamics."""

    def __init__(self, w, pd=None):
        m = w.model
        self.m, self.w, self.nb, self.dt = m, w, m.nbodies, float(m.dt)
        self.pd = pd
        self.I, self.Ic_inv = [], []
        for b in m.bodies:
            c, mass = np.asarray(b.inertia.com, float), float(b.inertia.mass)
            cx = np.array([[0, -c[2], c[1]], [c[2], 0, -c[0]], [-c[1], c[0], 0]])
            S = np.zeros((6, 6))
            S[:3, :3] = b.inertia.inertia + mass * cx @ cx.T
            S[:3, 3:], S[3:, :3], S[3:, 3:] = mass * cx, mass * cx.T, mass * np.eye(3)
            self.I.append(_t(S))
            J = np.asarray(b.inertia.inertia, float)
            self.Ic_inv.append(_t(np.linalg.inv(J) if abs(np.linalg.det(J)) >= 1e-20 else np.zeros((3, 3))))
        self.gains = None if w.contact is None else w.contact_gains()

    def kinematics(self, q, v):
        """Per body: E (parent -> body rotation), r (origin in the parent), spatial velocity, world rotation and origin."""
        self.E, self.r, self.vel, self.S, self.R, self.P, self.vj = [], [], [], [], [], [], []
        n = q.shape[0]
        eye = torch.eye(3, dtype=torch.float64, device=q.device)
        for i, b in enumerate(self.m.bodies):
            j, o = b.joint, self.m.q_offsets[i]
            nd = j.ndof()
            pos = torch.zeros(n, 3, dtype=torch.float64, device=q.device)
            if j.jtype == W.REVOLUTE:
                K = _skew(_t(j.axis))
                a = q[:, o, None, None]
                E = eye - K * torch.sin(a) + (K @ K) * (1.0 - torch.cos(a))
                S = torch.cat([_t(j.axis), torch.zeros(3, dtype=torch.float64, device=q.device)])[None]
            elif j.jtype == W.FREE:
                E = _quat_mat(_quat_exp(q[:, o:o + 3])).transpose(-1, -2)
                pos = q[:, o + 3:o + 6]
                S = torch.eye(6, dtype=torch.float64, device=q.device)
            elif j.jtype == W.FIXED:
                E, S = eye.expand(n, 3, 3), torch.zeros(0, 6, dtype=torch.float64, device=q.device)
            elif j.jtype == W.PRISMATIC:
                E, S = eye.expand(n, 3, 3), torch.cat([torch.zeros(3, dtype=torch.float64, device=q.device), _t(j.axis)])[None]
                pos = q[:, o:o + 1] * _t(j.axis)
            else:
                raise ValueError("joint type")
            rot, at = _t(j.parent_to_joint.rot), _t(j.parent_to_joint.pos)
            r = at + pos @ rot
            E = E @ rot
            vj = v[:, o:o + nd] @ S if nd else torch.zeros(n, 6, dtype=torch.float64, device=q.device)
            p = b.parent
            if p < 0:
                vel, R, P = vj, E.transpose(-1, -2), r
            else:
                vel = self.motion(E, r, self.vel[p]) + vj
                R = self.R[p] @ E.transpose(-1, -2)
                P = self.P[p] + _mv(self.R[p], r)
            for name, x in (("E", E), ("r", r), ("vel", vel), ("S", S), ("R", R), ("P", P), ("vj", vj)):
                getattr(self, name).append(x)

    @staticmethod
    def motion(E, r, x):
        return torch.cat([_mv(E, x[:, :3]), _mv(E, x[:, 3:] - _cross(r, x[:, :3]))], -1)

    @staticmethod
    def force_up(E, r, f):
        lin = _mtv(E, f[:, 3:])
        return torch.cat([_mtv(E, f[:, :3]) + _cross(r, lin), lin], -1)

    @staticmethod
    def motion_matrix(E, r):
        X = torch.zeros(E.shape[0], 6, 6, dtype=torch.float64, device=E.device)
        X[:, :3, :3], X[:, 3:, 3:] = E, E
        X[:, 3:, :3] = -E @ _skew(r)
        return X

    def forces(self, q, v, ctrl):
        m = self.m
        if m.actuators:
            f = torch.zeros_like(v)
            for a, act in enumerate(m.actuators):
                o = m.q_offsets[act.joint_idx]
                c = ctrl[:, a]
                if act.ctrl_range is not None:
                    c = c.clamp(min(act.ctrl_range), max(act.ctrl_range))
                x = act.gear * (act.gain * c + act.bias_q * q[:, o] + act.bias_v * v[:, o])
                if act.force_range is not None:
                    x = x.clamp(min(act.force_range), max(act.force_range))
                f[:, o] += x
        else:
            f = ctrl.clone()
        for i, b in enumerate(m.bodies):
            j, o = b.joint, m.q_offsets[i]
            for k in range(j.ndof()):
                f[:, o + k] -= j.damping * v[:, o + k]
            if j.ndof() == 1:
                f[:, o] -= j.stiffness * (q[:, o] - j.spring_ref)
                if j.limits is not None:
                    lo, hi = j.limits
                    for sign, depth in ((1.0, lo - q[:, o]), (-1.0, q[:, o] - hi)):
                        push = sign * (j.limit_stiffness * depth + j.limit_damping * (-sign * v[:, o]).clamp_min(0.0))
                        f[:, o] += torch.where(depth > 0.0, push, torch.zeros_like(push))
                if j.friction_loss > 0.0:
                    f[:, o] -= j.friction_loss * torch.tanh(v[:, o] / 1e-3)
        return f

    @staticmethod
    def inverse(D):
        """Inverse of symmetric positive definite n x n blocks, Gauss-Jordan."""
        n = D.shape[-1]
        A = torch.cat([D, torch.eye(n, dtype=D.dtype, device=D.device).expand_as(D)], -1).clone()
        for k in range(n):
            A[:, k] = A[:, k] / A[:, k, k:k + 1].clone()
            f = A[:, :, k:k + 1].clone()
            f[:, k] = 0.0
            A = A - f * A[:, k:k + 1]
        return A[:, :, n:]

    def solve(self, q, v, ctrl, ext):
        """qdd, keeping the factorisation for `respond`."""
        m, nb = self.m, self.nb
        f = self.forces(q, v, ctrl)
        IA = [self.I[i].expand(q.shape[0], 6, 6).clone() for i in range(nb)]
        pA, c = [], []
        for i in range(nb):
            w, l = self.vel[i][:, :3], self.vel[i][:, 3:]
            jw, jl = self.vj[i][:, :3], self.vj[i][:, 3:]
            c.append(torch.cat([_cross(w, jw), _cross(w, jl) + _cross(l, jw)], -1) if m.bodies[i].parent >= 0
                     else torch.zeros_like(self.vel[i]))
            h = self.vel[i] @ self.I[i]
            p = torch.cat([_cross(w, h[:, :3]) + _cross(l, h[:, 3:]), _cross(w, h[:, 3:])], -1)
            pA.append(p if ext is None else p - ext[i])
        self.U, self.Dinv = [None] * nb, [None] * nb
        u = [None] * nb
        for i in reversed(range(nb)):
            b = m.bodies[i]
            j, o, nd = b.joint, m.q_offsets[i], b.joint.ndof()
            S = self.S[i]
            Ia, pa = IA[i], pA[i]
            if nd:
                U = Ia @ S.T
                D = S @ U + (j.armature + self.dt * j.damping) * torch.eye(nd, dtype=q.dtype, device=q.device)
                Dinv = 1.0 / D if nd == 1 else self.inverse(D)
                u[i] = f[:, o:o + nd] - pa @ S.T
                self.U[i], self.Dinv[i] = U, Dinv
                if b.parent >= 0:
                    Ia = Ia - U @ Dinv @ U.transpose(-1, -2)
                    pa = pa + _mv(Ia, c[i]) + _mv(U @ Dinv, u[i])
            elif b.parent >= 0:
                pa = pa + _mv(Ia, c[i])
            if b.parent >= 0:
                X = self.motion_matrix(self.E[i], self.r[i])
                IA[b.parent] = IA[b.parent] + X.transpose(-1, -2) @ Ia @ X
                pA[b.parent] = pA[b.parent] + self.force_up(self.E[i], self.r[i], pa)
        g = torch.cat([torch.zeros(3, dtype=q.dtype, device=q.device), -_t(m.gravity)]).expand(q.shape[0], 6)
        return self._down(u, c, g, q)

    def _down(self, u, c, root, like):
        qdd, acc = torch.zeros_like(like), []
        for i in range(self.nb):
            b = self.m.bodies[i]
            o, nd = self.m.q_offsets[i], b.joint.ndof()
            a = self.motion(self.E[i], self.r[i], acc[b.parent] if b.parent >= 0 else root)
            if c is not None:
                a = a + c[i]
            if nd:
                x = _mv(self.Dinv[i], u[i] - _mtv(self.U[i], a))
                qdd[:, o:o + nd] = x
                a = a + x @ self.S[i]
            acc.append(a)
        return qdd

    def respond(self, dext, like):
        """Change of qdd for a change of the external forces."""
        p = [-x for x in dext]
        u = [None] * self.nb
        for i in reversed(range(self.nb)):
            b = self.m.bodies[i]
            pa = p[i]
            if b.joint.ndof():
                u[i] = -(pa @ self.S[i].T)
                if b.parent >= 0:
                    pa = pa + _mv(self.U[i] @ self.Dinv[i], u[i])
            if b.parent >= 0:
                p[b.parent] = p[b.parent] + self.force_up(self.E[i], self.r[i], pa)
        return self._down(u, None, torch.zeros(like.shape[0], 6, dtype=like.dtype, device=like.device), like)

    # ── contact ──
    def eff_mass(self, i, at, d):
        b = self.m.bodies[i]
        a = _cross(at - _t(b.inertia.com), d)
        return 1.0 / (1.0 / b.inertia.mass + _dot(a, a @ self.Ic_inv[i]).clamp_min(0.0))

    def points(self, i, z):
        """Contact points of body i's shape, body frame."""
        g = self.m.bodies[i].geometry
        rot, pos = _t(g.origin.rot), _t(g.origin.pos)
        n = z @ rot.T
        if g.kind == W_SPHERE:
            s = [-g.params[0] * n]
        elif g.kind == W_CAPSULE:
            end = torch.zeros_like(n)
            end[:, 2] = -0.5 * g.params[1] * torch.sign(n[:, 2])
            s = [end - g.params[0] * n]
        elif g.kind == W_BOX:
            s = [_t([g.params[k] * (1.0 if c >> k & 1 else -1.0) for k in range(3)]).expand_as(n) for c in range(8)]
        else:
            raise ValueError("shape")
        return [pos + x @ rot for x in s]

    def terrain(self, x, y):
        h = self.w.heightfield
        if h is None:
            z = torch.zeros_like(x)
            return z + self.w.contact.ground_height, torch.stack([z, z, z + 1.0], -1)
        nodes = _t(np.asarray(h.heights, dtype=np.float32)).reshape(h.ny, h.nx) + h.origin[2]

        def cell(p, o, n):
            u = ((p - o) / h.cell).clamp(0.0, n - 1.0)
            k = u.floor().long().clamp(0, n - 2)
            return k, u - k, (p >= o) & (p <= o + (n - 1) * h.cell)
        ix, tx, inx = cell(x, h.origin[0], h.nx)
        iy, ty, iny = cell(y, h.origin[1], h.ny)
        h00, h10, h01, h11 = nodes[iy, ix], nodes[iy, ix + 1], nodes[iy + 1, ix], nodes[iy + 1, ix + 1]
        z = (h00 * (1 - tx) + h10 * tx) * (1 - ty) + (h01 * (1 - tx) + h11 * tx) * ty
        gx = torch.where(inx, ((h10 - h00) * (1 - ty) + (h11 - h01) * ty) / h.cell, torch.zeros_like(x))
        gy = torch.where(iny, ((h01 - h00) * (1 - tx) + (h11 - h10) * tx) / h.cell, torch.zeros_like(x))
        nrm = torch.stack([-gx, -gy, torch.ones_like(gx)], -1)
        return z, nrm / nrm.norm(dim=-1, keepdim=True)

    def penalty(self):
        """External forces of the bounded spring-damper law, and the readback rows."""
        mu, dt = self.w.contact.friction, self.dt
        n = self.vel[0].shape[0]
        zero = torch.zeros(n, dtype=torch.float64, device=self.vel[0].device)
        ext, rows = [], []
        for i, b in enumerate(self.m.bodies):
            e, row = torch.zeros_like(self.vel[i]), torch.zeros(n, 8, dtype=torch.float64, device=zero.device)
            if b.geometry is not None and b.geometry.kind != 0:
                k, d = self.gains[i]
                scale = 0.25 if b.geometry.kind == W_BOX else 1.0
                R = self.R[i]
                for at in self.points(i, R[:, 2]):
                    world = self.P[i] + _mv(R, at)
                    hgt, nw = self.terrain(world[:, 0], world[:, 1])
                    pen = nw[:, 2] * (hgt - world[:, 2])
                    on = pen > 0.0
                    nb = _mtv(R, nw)
                    vp = self.vel[i][:, 3:] + _cross(self.vel[i][:, :3], at)
                    vn = _dot(vp, nb)
                    mn = self.eff_mass(i, at, nb)
                    fn = ((4.0 * mn / dt**2).clamp_max(scale * k) * pen - (mn / dt).clamp_max(scale * d) * vn).clamp_min(0.0)
                    vt = vp - nb * vn[:, None]
                    sp = vt.norm(dim=-1)
                    t = vt / sp.clamp_min(1e-300)[:, None]
                    ft = torch.minimum(mu * fn * (sp / 1e-3).clamp_max(1.0), self.eff_mass(i, at, t) / dt * sp)
                    fb = nb * fn[:, None] - torch.where((sp > 1e-6)[:, None], t * ft[:, None], torch.zeros_like(t))
                    fb = torch.where(on[:, None], fb, torch.zeros_like(fb))
                    e = e + torch.cat([_cross(at, fb), fb], -1)
                    deeper = on & (pen > row[:, 1])
                    row[:, 0] = torch.where(on, torch.ones_like(zero), row[:, 0])
                    row[:, 1] = torch.where(deeper, pen, row[:, 1])
                    for c, x in enumerate((world[:, 0], world[:, 1], hgt)):
                        row[:, 2 + c] = torch.where(deeper, x, row[:, 2 + c])
                    row[:, 5:] = row[:, 5:] + _mv(R, fb)
            ext.append(e)
            rows.append(row)
        return ext, torch.stack(rows, 1)

    def impulse(self, q, v, ctrl, carried):
        """The velocity-level solve: a leading solve at the carried forces, then
        the sweeps, each at the free velocity v + dt qdd."""
        w, dt, mu = self.w, self.dt, self.w.contact.friction
        qdd = self.solve(q, v, ctrl, carried["ext"])
        pts = {}
        for i, b in enumerate(self.m.bodies):
            if b.geometry is None or b.geometry.kind == 0:
                continue
            R = self.R[i]
            at, = self.points(i, R[:, 2])
            world = self.P[i] + _mv(R, at)
            hgt, nw = self.terrain(world[:, 0], world[:, 1])
            pen = nw[:, 2] * (hgt - world[:, 2])
            nb = _mtv(R, nw)
            axis = torch.where((nb[:, :1].abs() > 0.9), _t([0.0, 1.0, 0.0]), _t([1.0, 0.0, 0.0]))
            tu = _cross(nb, axis)
            tu = tu / tu.norm(dim=-1, keepdim=True)
            tw = _cross(nb, tu)
            x = (pen.abs() / 0.001).clamp(0.0, 1.0)
            imp = 0.9 + 0.05 * torch.where(x <= 0.5, x * x / 0.5, 1.0 - (1.0 - x) ** 2 / 0.5)
            bias = torch.where(pen > 0.0, imp * w.impulse_erp() * pen / dt, torch.zeros_like(pen))
            pts[i] = (at, nb, tu, tw, self.eff_mass(i, at, nb).clamp_min(1e-9), self.eff_mass(i, at, tu).clamp_min(1e-9),
                      self.eff_mass(i, at, tw).clamp_min(1e-9), bias, pen > -0.001)
        ext = [x.clone() for x in carried["ext"]]
        for _ in range(w.impulse_sweeps):
            vf = v + dt * qdd
            vel = []
            for i, b in enumerate(self.m.bodies):
                o, nd = self.m.q_offsets[i], b.joint.ndof()
                vj = vf[:, o:o + nd] @ self.S[i]
                vel.append(vj if b.parent < 0 else self.motion(self.E[i], self.r[i], vel[b.parent]) + vj)
            new = [torch.zeros_like(x) for x in ext]
            for i, (at, nb, tu, tw, mn, cu, cw, bias, on) in pts.items():
                s = carried["imp"][i]
                vp = vel[i][:, 3:] + _cross(vel[i][:, :3], at)
                fn = ((bias - _dot(vp, nb)) * mn + s[:, 0]).clamp_min(0.0)
                fu, fw = s[:, 1] - _dot(vp, tu) * cu, s[:, 2] - _dot(vp, tw) * cw
                size = torch.sqrt(fu * fu + fw * fw)
                cut = torch.where(size > mu * fn, mu * fn / size.clamp_min(1e-300), torch.ones_like(size))
                s = torch.stack([fn, fu * cut, fw * cut], -1)
                s = torch.where(on[:, None], s, torch.zeros_like(s))
                carried["imp"][i] = s
                fb = (nb * s[:, :1] + tu * s[:, 1:2] + tw * s[:, 2:]) / dt
                new[i] = torch.cat([_cross(at, fb), fb], -1)
            qdd = qdd + self.respond([a - b for a, b in zip(new, ext)], q)
            ext = new
        carried["ext"] = ext
        return qdd

    def integrate(self, q, v, qdd):
        v = v + self.dt * qdd
        q = q.clone()
        for i, b in enumerate(self.m.bodies):
            o, nd = self.m.q_offsets[i], b.joint.ndof()
            if nd == 1:
                q[:, o] += self.dt * v[:, o]
            elif nd == 6:
                cur = _quat_exp(q[:, o:o + 3])
                q[:, o + 3:o + 6] += self.dt * _mv(_quat_mat(cur), v[:, o + 3:o + 6])
                q[:, o:o + 3] = _quat_log(_quat_mul(cur, _quat_exp(v[:, o:o + 3] * self.dt)))
        return q, v

    def steps(self, q, v, ctrl, targets, stream, n):
        w, rows = self.w, None
        imp = w.contact is not None and w.impulse_sweeps > 0
        carried = None
        for _ in range(n):
            if stream is not None:
                ctrl = ctrl.clone()
                nz = w.noise
                if nz.dist == W.NOISE_UNIFORM:
                    for k in nz.dofs:
                        ctrl[:, k] = nz.a + (nz.b - nz.a) * stream.uniform()
                else:
                    for k in range(0, len(nz.dofs), 2):
                        u1, u2 = stream.uniform(), stream.uniform()
                        r = torch.sqrt(-2.0 * torch.log1p(-u1))
                        ctrl[:, nz.dofs[k]] = nz.a + nz.b * r * torch.cos(2.0 * math.pi * u2)
                        if k + 1 < len(nz.dofs):
                            ctrl[:, nz.dofs[k + 1]] = nz.a + nz.b * r * torch.sin(2.0 * math.pi * u2)
            if self.pd is not None:
                ctrl = ctrl.clone()
                for k, d in enumerate(self.pd):
                    x = d.kp * (targets[:, k] - q[:, d.q_index]) - d.kd * v[:, d.v_index]
                    ctrl[:, d.v_index] = x.clamp(-d.max_force, d.max_force)
            self.kinematics(q, v)
            if imp:
                if carried is None:
                    carried = {"ext": [torch.zeros_like(x) for x in self.vel],
                               "imp": {i: torch.zeros(q.shape[0], 3, dtype=q.dtype, device=q.device) for i in range(self.nb)}}
                qdd = self.impulse(q, v, ctrl, carried)
            else:
                ext = None
                if w.contact is not None:
                    ext, rows = self.penalty()
                qdd = self.solve(q, v, ctrl, ext)
            q, v = self.integrate(q, v, qdd)
        return q, v, rows


W_SPHERE, W_BOX, W_CAPSULE = 1, 2, 3


def _observe(bodies, spec, q, v):
    """The observation row of each world."""
    m = bodies.m
    bodies.kinematics(q, v)
    R, P = bodies.R, bodies.P
    out = []
    for op in spec.obs:
        name = type(op).__name__
        if name == "QMinus":
            out.append(q[:, op.i] - op.c)
        elif name == "V":
            out.append(v[:, op.i])
        elif name == "BodyPitch":
            out.append(torch.atan2(-R[op.body][:, 2, 0], R[op.body][:, 2, 2]))
        elif name == "BodyRoll":
            out.append(torch.atan2(R[op.body][:, 2, 1], R[op.body][:, 2, 2]))
        elif name == "BodyYawError":
            e = op.cmd - torch.atan2(R[op.body][:, 1, 0], R[op.body][:, 0, 0])
            out.append(e - 2 * math.pi * torch.round(e / (2 * math.pi)))
        elif name == "BodyPosZ":
            out.append(P[op.body][:, 2])
        elif name == "BodyPos":
            out.append(P[op.body][:, op.axis])
        elif name == "ComOverSupport":
            mass = [b.inertia.mass for b in m.bodies]
            com = sum((P[i] + _mv(R[i], _t(b.inertia.com).expand_as(P[i]))) * mass[i] for i, b in enumerate(m.bodies)) / sum(mass)
            tgt = sum(P[b] + _mv(R[b], _t(o).expand_as(P[b])) for b, o in op.support) / len(op.support)
            e = com - tgt
            yaw = torch.atan2(R[op.heading_body][:, 1, 0], R[op.heading_body][:, 0, 0])
            s, c = torch.sin(yaw), torch.cos(yaw)
            out.append((c * e[:, 0] + s * e[:, 1], -s * e[:, 0] + c * e[:, 1], e[:, 2])[op.axis])
        else:
            raise ValueError(name)
    return torch.stack(out, -1)


def _mlp(flat, i, h, o, x):
    sizes = [h * i, h, h * h, h, o * h, o]
    W1, b1, W2, b2, W3, b3 = torch.split(flat[:sum(sizes)], sizes)
    h1 = torch.tanh(x @ W1.reshape(h, i).T + b1)
    h2 = torch.tanh(h1 @ W2.reshape(h, h).T + b2)
    return h1, h2, h2 @ W3.reshape(o, h).T + b3, W2.reshape(h, h), W3.reshape(o, h)


def _backward(x, h1, h2, W2, W3, d):
    d2 = (d @ W3) * (1.0 - h2 * h2)
    d1 = (d2 @ W2) * (1.0 - h1 * h1)
    return torch.cat([(d1.T @ x).reshape(-1), d1.sum(0), (d2.T @ h1).reshape(-1), d2.sum(0), (d.T @ h2).reshape(-1), d.sum(0)])


def _exact_ppo(case, seed):
    a0, c0, batch, orders, cfg = _ppo_inputs(case, seed)
    ai, ci, h, na = case["actor_in"], case["critic_in"], case["hidden"], case["act"]
    x = {k: _t(getattr(batch, k)) for k in ("obs_a", "obs_c", "act", "logp_old", "adv", "ret")}
    nets = [_t(a0), _t(c0)]
    mom = [(torch.zeros_like(p), torch.zeros_like(p)) for p in nets]
    off = a0.size - na
    ploss = vloss = kl = 0.0
    steps = 0
    for order in orders:
        order = torch.as_tensor(order.astype(np.int64), device=_dev())
        for at in range(0, order.numel(), cfg.minibatch):
            r = order[at:at + cfg.minibatch]
            nb = r.numel()
            xa, xc = x["obs_a"][r], x["obs_c"][r]
            h1, h2, mean, W2, W3 = _mlp(nets[0], ai, h, na, xa)
            sd = torch.exp(nets[0][off:])
            z = (x["act"][r] - mean) / sd
            logp = (-0.5 * z * z - torch.log(sd) - 0.5 * math.log(2 * math.pi)).sum(1)
            lr = logp - x["logp_old"][r]
            ratio = torch.exp(lr)
            adv = x["adv"][r]
            free, cut = ratio * adv, ratio.clamp(1 - cfg.clip, 1 + cfg.clip) * adv
            coef = torch.where(free <= cut + 1e-12, -adv * ratio / nb, torch.zeros_like(adv))[:, None]
            ga = torch.cat([_backward(xa, h1, h2, W2, W3, coef * z / sd), (coef * (z * z - 1.0)).sum(0) - cfg.entropy_coef])
            h1, h2, val, W2, W3 = _mlp(nets[1], ci, h, 1, xc)
            err = val[:, 0] - x["ret"][r]
            gc = _backward(xc, h1, h2, W2, W3, (2.0 * err.clamp(-cfg.vdelta, cfg.vdelta) / nb)[:, None])
            steps += 1
            for k, g in enumerate((ga, gc)):
                m1, m2 = mom[k]
                m1 = 0.9 * m1 + (1.0 - 0.9) * g
                m2 = 0.999 * m2 + (1.0 - 0.999) * g * g
                mom[k] = (m1, m2)
                nets[k] = nets[k] - 3e-4 * (m1 / (1.0 - 0.9**steps)) / (torch.sqrt(m2 / (1.0 - 0.999**steps)) + 1e-8)
            ploss = ploss - torch.minimum(free, cut).sum() / nb
            vloss = vloss + (err * err).sum() / nb
            kl = kl + (ratio - 1.0 - lr).sum() / nb / cfg.kl_scale
    return {"actor": nets[0], "critic": nets[1], "policy_loss": float(ploss / steps), "value_loss": float(vloss / steps),
            "kl": float(kl / steps)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "ppo":
        return _exact_ppo(case, seed)
    if kind == "span":
        # About 10 us for each of the ~55 torch operations per body and step.
        nb = W.config(MODELS[case["model"]][0]).model.nbodies
        if case["steps"] * nb * (30.0 if case["model"] == "ant_terrain_impulse" else 1.0) * max(1.0, case["worlds"] / 16384) > 25000:
            return None
        w, q, v, ctrl, targets = _span_inputs(case, seed)
        stream = None if w.noise is None else _Stream(w.noise.seed, case["worlds"])
        q, v, _ = _Bodies(w, w.pd).steps(_t(q), _t(v), _t(ctrl), None if targets is None else _t(targets), stream, case["steps"])
        return {"q": q, "v": v}
    if kind == "env":
        cl, q, v, targets = _loop(case, seed)
        q, v, rows = _Bodies(cl.base, cl.pd).steps(_t(q), _t(v), torch.zeros_like(_t(v)), _t(targets), None, case["every"])
        return {"q": q, "v": v, "contacts": rows}
    cl, q, v, _ = _loop(case, seed)
    n, spec = case["worlds"], cl.spec
    bodies = _Bodies(cl.base, cl.pd)
    q, v, ctrl = _t(q), _t(v), torch.zeros_like(_t(v))
    base, std, weights = _t(cl.base_targets(n)), _t(cl.std), _t(cl.weights)
    stream = _Stream(cl.seed, n)
    z = torch.zeros(n, spec.n_out(), dtype=torch.float64, device=q.device)
    keep = math.sqrt(1.0 - spec.noise_rho**2)
    hist = {"obs": [], "out": [], "q": [], "v": []}
    for _ in range(case["control"]):
        obs = _observe(bodies, spec, q, v)
        obs = torch.stack([obs[:, i] + s * stream.normal() for i, s in enumerate(spec.input_noise)], -1)
        mean = _mlp(weights, spec.n_in(), spec.hidden, spec.n_out(), obs)[2]
        z = torch.stack([spec.noise_rho * z[:, k] + keep * stream.normal() for k in range(spec.n_out())], -1)
        act = mean + std * z
        logp = (-0.5 * z * z - torch.log(std) - 0.5 * math.log(2 * math.pi)).sum(1)
        targets = base + act.clamp(-spec.act_clamp, spec.act_clamp)
        q, v, _ = bodies.steps(q, v, ctrl, targets, None, case["every"])
        if case["history"]:
            for k, x in (("obs", obs), ("out", torch.cat([act, logp[:, None]], -1)), ("q", q), ("v", v)):
                hist[k].append(x)
    if case["history"]:
        return {k: torch.stack(x) for k, x in hist.items()}
    return {"q": q, "v": v, "targets": targets}
