"""State rows between host arrays and the device layout, through the C ABI.

Loads and readbacks pass through pinned slots of whole 64-world tiles (at most
128 K values each, four in turn) and a tile kernel of 64 columns. Sizes here sit at
their edges: one world, a partial tile, more chunks than slots, rows wider than
a column tile, and values that a conversion can get wrong. An f32 sim must give
back each value rounded once, whatever the host thread's subnormal mode.
"""
import numpy as np
import pytest
import torch

from phyz_amd import workloads as W
from phyz_amd.sim import BatchSim, from_control_loop, from_workload

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.ascontiguousarray(a, dtype=np.float64).view(np.uint64)


def _rounded(a, prec):
    return a if prec == "f64" else a.astype(np.float32).astype(np.float64)


# chain7 rows are 7 wide: a slot holds 9344 worlds of q and v, 6208 with ctrl;
# 100001 worlds are more chunks than slots.
@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 6209, 9345, 12345, 100001])
def test_rows_come_back_as_loaded(n, prec):
    sim = from_workload(W.config(2), prec, nworld=n)
    rng = np.random.default_rng(n)
    q, v, c = (rng.normal(size=(n, 7)) * 10.0 ** rng.integers(-30, 30, size=(n, 7)) for _ in range(3))
    for a in (q, v, c):
        a[0, :6] = [1e-40, -0.0, np.inf, -np.inf, 1e-46, 3.4028235677973366e38]
    for _ in range(2):  # the second load reuses slots that the first one's kernels read
        sim.load_states(q, v, c)
        torch.set_flush_denormal(True)
        try:
            sim.load_states(v, q, c)
            got = (*sim.readback_states(), sim.readback_controls())
        finally:
            torch.set_flush_denormal(False)
        with np.errstate(over="ignore"):
            want = [_rounded(a, prec) for a in (v, q, c)]
        for g, w in zip(got, want):
            assert np.array_equal(_bits(g), _bits(w))
    sim.load_states(q, v)
    assert not sim.readback_controls().any()
    sim.close()


@pytest.mark.parametrize("prec", ["f32", "f64"])
def test_wide_rows(prec):
    """Impulse rows are 48 values per body: seven column tiles of an ant's."""
    n = 1000
    sim = from_workload(W.config(6), prec, nworld=n)
    nb = sim.nb
    rng = np.random.default_rng(3)
    cs = rng.normal(size=(n, nb, 56))
    ext = rng.normal(size=(n, nb, 6))
    sim.load_contact_state(cs, ext)
    cs2, ext2 = sim.readback_contact_state()
    assert np.array_equal(_bits(cs2[..., 8:]), _bits(_rounded(cs[..., 8:], prec)))
    assert np.array_equal(_bits(ext2), _bits(_rounded(ext, prec)))
    sim.close()


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("n", [65, 300])
def test_rows_of_many_column_tiles(n, prec):
    """A 22-body tree's impulses are 1056 values a world, 16.5 column tiles, and
    a full slot holds one or two tiles of worlds; 300 worlds take several."""
    w = W.config(4)
    sim = BatchSim(w.model, n, prec)
    sim.enable_contact_impulse(w.contact.ground_height, w.contact.friction, w.contact_gains(), None, None)
    rng = np.random.default_rng(n)
    cs = rng.normal(size=(n, sim.nb, 56))
    ext = rng.normal(size=(n, sim.nb, 6))
    sim.load_contact_state(cs, ext)
    cs2, ext2 = sim.readback_contact_state()
    assert np.array_equal(_bits(cs2[..., 8:]), _bits(_rounded(cs[..., 8:], prec)))
    assert np.array_equal(_bits(ext2), _bits(_rounded(ext, prec)))
    sim.close()


def test_history_ranges_match_single_rows():
    """A range of history rows is one pipelined readback: the same bits as row by row."""
    cl = W.control_loop()
    n = 3001
    sim = from_control_loop(cl, "f32", nworld=n)
    q, v, _, _ = cl.base.initial_state(n)
    sim.load_states(q, v)
    k = min(7, cl.spec.history_steps)
    sim.rollout(0, k, 2, record_states=True)
    obs, out = sim.readback_policy_history(0, k)
    hq, hv = sim.readback_state_history(0, k)
    for j in range(k):
        o1, u1 = sim.readback_policy_history(j, j + 1)
        q1, v1 = sim.readback_state_history(j, j + 1)
        for a, b in ((obs, o1), (out, u1), (hq, q1), (hv, v1)):
            assert np.array_equal(_bits(a[j]), _bits(b[0]))
    qf, vf = sim.readback_states()
    assert np.array_equal(_bits(hq[-1]), _bits(qf)) and np.array_equal(_bits(hv[-1]), _bits(vf))
    assert np.isfinite(obs).all() and np.abs(obs[1] - obs[0]).max() > 0
    sim.close()
