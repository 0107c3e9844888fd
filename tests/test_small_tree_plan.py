"""Trees of fewer than 14 bodies over several waves in small f32 launches
(plan_partition): the plan by size, and on the device the partitioned kernel
against the lane-per-world kernel of the same launch."""
import numpy as np
import pytest

from phyz_amd import workloads as W
from phyz_amd.sim import BatchSim, from_workload
from tests.models import deck_and_feet, legged, random_tree


@pytest.mark.parametrize("index,nworld,prec,block", [
    (3, 1, "f32", 256),       # ant: a leg per wave
    (3, 49152, "f32", 256),   # three workgroups per CU
    (3, 49153, "f32", 64),
    (3, 4096, "f64", 64),     # f64 keeps one lane per world
    (7, 32768, "f32", 256),   # MJCF ant
    (7, 65536, "f32", 64),
    (6, 4096, "f32", 64),     # impulse contact needs the whole tree in one lane
    (2, 4096, "f32", 64),     # a chain has no subtrees
])
def test_plan_by_size(index, nworld, prec, block, monkeypatch):
    monkeypatch.delenv("PHZ_PARTITION", raising=False)
    s = from_workload(W.config(index), prec, nworld=nworld, device=-1)
    s.compile()
    info = s.kernel_info()
    assert info["block"] == block
    if block == 256:
        assert info["vgpr"] + max(info["agpr"], 0) <= 256 and info["scratch_bytes"] == 0


def _tree_sim(name, nworld, device=0):
    """A legged tree or three free bodies on the ground, or the ant under PD servos."""
    if name == "ant_pd":
        cl = W.control_loop()
        c = cl.base.contact
        sim = BatchSim(cl.base.model, nworld, "f32", device=device)
        sim.enable_ground_contact(c.ground_height, c.stiffness, c.damping, c.friction)
        sim.enable_pd_control(cl.pd)
        return cl.base.model, sim
    model = deck_and_feet() if name == "deck" else random_tree(1) if name == "mixed" else legged(*name)
    sim = BatchSim(model, nworld, "f32", device=device)
    if name != "mixed":
        sim.enable_ground_contact(0.0, 2e4, 200.0, 0.8)
    return model, sim


# Blocks at one workgroup per CU, at most two, at most three, and beyond: the
# third workgroup only where the plan's registers and gain pay for it.
@pytest.mark.parametrize("name,blocks", [
    ((2, 2), (128, 128, 64, 64)),
    ((3, 2), (128, 128, 64, 64)),    # 423 us as one lane per world, 441 partitioned
    ((5, 2), (256, 256, 64, 64)),    # 632 / 739: two waves carry a leg, one carries two
    ((6, 2), (256, 256, 256, 64)),
    ((4, 3), (256, 256, 256, 64)),
    ((3, 3), (128, 128, 64, 64)),    # above 256 registers: two workgroups of two waves fill a CU's SIMDs
    ("deck", (128, 128, 128, 64)),   # no trunk: independent bodies
    ("mixed", (256, 256, 64, 64)),   # 841 / 1167
    ("ant_pd", (256, 256, 256, 64)),
])
def test_third_workgroup_per_cu_only_where_it_pays(name, blocks, monkeypatch):
    monkeypatch.delenv("PHZ_PARTITION", raising=False)
    got = []
    for n in (16384, 32768, 49152, 49153):
        _, sim = _tree_sim(name, n, device=-1)
        sim.compile()
        got.append(sim.kernel_info()["block"])
    assert tuple(got) == blocks


@pytest.mark.gpu
@pytest.mark.parametrize("name,nworld,tol_v", [((2, 2), 65, 4e-4), ((3, 2), 16385, 4e-4), ((5, 2), 129, 4e-4), ((3, 3), 70, 4e-4),
                                               ("deck", 100, 4e-4), ("mixed", 77, 1e-5), ("ant_pd", 49151, 4e-4)])
def test_other_trees_match_lane_per_world(name, nworld, tol_v, monkeypatch):
    """As above on two, three and five legs, on a forest, on mixed joints
    without contact and under PD servos; a repeat and a span cut into launches
    give the same bits."""
    got = []
    for plan in (None, "0"):
        if plan is None:
            monkeypatch.delenv("PHZ_PARTITION", raising=False)
        else:
            monkeypatch.setenv("PHZ_PARTITION", plan)
        model, sim = _tree_sim(name, nworld)
        rng = np.random.default_rng(5)
        q, v = (0.05 * rng.normal(size=(nworld, model.nq)).astype(np.float32).astype(np.float64) for _ in range(2))
        if name != "mixed":
            q[:, 5] += 0.45
        assert (sim.kernel_info()["block"] == 64) == (plan == "0")
        spans = []
        for cut in ((40,), (40,), (1, 16, 23)):
            if name == "ant_pd":
                sim.set_position_targets(np.tile([0.0, 0.5] * 4, (nworld, 1)))
            sim.load_states(q, v)
            for n in cut:
                sim.step_many(n)
            spans.append(sim.readback_states() + (sim.readback_controls(),))
        for other in spans[1:]:
            for x, y in zip(spans[0], other):
                assert np.array_equal(x, y)
        got.append(spans[0])
        sim.close()
    a, b = got
    for x, y, tol in ((a[0], b[0], 1e-5), (a[1], b[1], tol_v)):
        gap = np.linalg.norm(x - y) / np.linalg.norm(y)
        print(f"{name} {nworld}: {gap:.2e}", flush=True)
        assert np.isfinite(x).all() and gap <= tol


@pytest.mark.gpu
@pytest.mark.parametrize("index,nworld", [(3, 1), (3, 65), (3, 16385), (7, 64), (7, 4099)])
def test_small_tree_matches_lane_per_world(index, nworld, monkeypatch):
    """40 steps from the workload's states lowered onto the ground: the same
    random stream, states and contact rows of the two plans within the f32
    rounding the steps amplify (two kernels of one plan differ as much: 1.3e-7
    in q and 5.4e-7 in v over 100 steps for one rounding of the input, 4e-4
    where a foot touches one step apart), a repeat the same bits, and a span
    cut into launches the same bits."""
    w = W.config(index)
    q, v, c, _ = w.initial_state(nworld)
    if index == 3:
        q[:, 5] -= 0.2
    got = []
    for plan in (None, "0"):
        if plan is None:
            monkeypatch.delenv("PHZ_PARTITION", raising=False)
        else:
            monkeypatch.setenv("PHZ_PARTITION", plan)
        sim = from_workload(w, "f32", nworld=nworld)
        assert sim.kernel_info()["block"] == (64 if plan else 256)
        spans = []
        for cut in ((40,), (40,), (1, 16, 23)):
            sim.load_states(q, v, c)
            for n in cut:
                sim.step_many(n)
            spans.append(sim.readback_states() + (sim.readback_contacts(), sim.readback_rng(), sim.readback_controls()))
        for other in spans[1:]:
            for x, y in zip(spans[0], other):
                assert np.array_equal(x, y)
        got.append(spans[0])
        sim.close()
    a, b = got
    assert np.array_equal(a[3], b[3]) and np.array_equal(a[4], b[4])
    for x, y, tol in ((a[0], b[0], 1e-5), (a[1], b[1], 4e-4)):
        assert np.isfinite(x).all() and np.linalg.norm(x - y) <= tol * np.linalg.norm(y)
    assert (a[2][..., 0] != b[2][..., 0]).mean() < 1e-3
