"""Trees of fewer than 14 bodies over several waves in small f32 launches
(plan_partition): the plan by size, and on the device the partitioned kernel
against the lane-per-world kernel of the same launch."""
import numpy as np
import pytest

from phyz_amd import workloads as W
from phyz_amd.sim import from_workload


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
