"""The policy kernel's layers 2 and 3 in bf16 pieces, and its workgroup-per-tile
form for small launches (phz_control.h, tanh_layer_split and policy_team).

- The split layers' error against the MLP in 64 bits is no larger than the f32
  MFMA's on the same weights and inputs. Weights with one value that a bf16
  piece cannot hold (1e-40) take the f32 kernel and change nothing else by more
  than 1e-40; infinite weights take it too.
- The three forms give the same bits, at ragged widths, two output blocks, wide
  inputs, partial tiles and a single world.
"""
import dataclasses

import numpy as np
import pytest

from phyz_amd import workloads as W
from phyz_amd.policy import QMinus
from phyz_amd.sim import from_control_loop

pytestmark = pytest.mark.gpu


def _sim(hidden, n, extra=0, noise=0.0):
    cl = W.control_loop(hidden)
    obs = list(cl.spec.obs) + [QMinus(6 + k % 8, 0.1 * k) for k in range(extra)]
    spec = dataclasses.replace(cl.spec, obs=obs, input_noise=[noise] * len(obs), history_steps=3)
    cl = dataclasses.replace(cl, spec=spec, weights=np.zeros(spec.n_weights()))
    sim = from_control_loop(cl, "f32", nworld=n)
    q, v, _, _ = cl.base.initial_state(n)
    sim.load_states(q, v)
    return cl, sim


def _weights(spec, seed, scale):
    i, h, o = spec.n_in(), spec.hidden, spec.n_out()
    rng = np.random.default_rng(seed)
    parts = [rng.normal(size=(h, i)) / np.sqrt(i), 0.1 * rng.normal(size=h), rng.normal(size=(h, h)) / np.sqrt(h),
             0.1 * rng.normal(size=h), rng.normal(size=(o, h)) / np.sqrt(h), 0.1 * rng.normal(size=o)]
    return [(scale * p).astype(np.float32).astype(np.float64) for p in parts]


def _flat(parts):
    return np.concatenate([p.ravel() for p in parts])


def _errors(hidden, w):
    """Relative error of the means against 64 bits in f32 layers (one weight of
    1e-40 added, which changes no sum) and in split ones."""
    err = {}
    for form in ("f32", "split"):
        _, sim = _sim(hidden, 4000)
        parts = [a.copy() for a in w]
        if form == "f32":
            parts[2][0, 0] = 1e-40
        sim.set_policy_weights(_flat(parts))
        sim.set_policy_std(np.full(8, 1e-30))  # the action is the mean
        sim.run_policy(0)
        obs, out = sim.readback_policy_history(0, 1)
        h = np.tanh(np.tanh(obs[0] @ parts[0].T + parts[1]) @ parts[2].T + parts[3])
        want = h @ parts[4].T + parts[5]
        err[form] = np.linalg.norm(out[0][:, :8] - want) / np.linalg.norm(want)
        sim.close()
    return err


@pytest.mark.parametrize("hidden,scale", [(32, 1.0), (48, 0.2), (100, 3.0), (256, 1.0), (256, 0.05)])
@pytest.mark.parametrize("seed", [5, 6])
def test_split_error_is_not_larger(hidden, scale, seed):
    err = _errors(hidden, _weights(W.control_loop(hidden).spec, seed, scale))
    print(f"hidden {hidden} scale {scale} seed {seed}: {err}", flush=True)
    assert err["split"] <= err["f32"]


@pytest.mark.parametrize("kind", ["random signs", "one sign", "equal activations"])
@pytest.mark.parametrize("hidden", [32, 64, 256])
def test_dropped_products_at_their_largest(hidden, kind):
    """Weights of 0x3f807fc0 (pieces 1, 2^-8, -2^-17) times powers of two: the
    products that the split leaves out are then up to 2^-24 of the whole and,
    with activations of the same kind, all of one sign. In sums of one sign
    they add at most 2^-24 of the sum per layer to what the roundings leave, so
    2 x 2^-24 over the two layers (tanh does not enlarge the first's); sums of
    mixed signs do not line up and stay below the f32 layers' error."""
    worst = float(np.uint32(0x3F807FC0).view(np.float32))
    w = _weights(W.control_loop(hidden).spec, 1, 1.0)
    rng = np.random.default_rng(2)
    for k in (2, 4):
        sign = np.sign(rng.normal(size=w[k].shape)) if kind == "random signs" else 1.0
        w[k] = worst * sign * 2.0 ** rng.integers(-7, -3, size=w[k].shape)
    if kind != "random signs":
        w[3], w[5] = 0.0 * w[3], 0.0 * w[5]
    if kind == "equal activations":
        w[0], w[1] = 0.0 * w[0], np.full(hidden, float(np.float32(np.arctanh(worst / 2))))
    err = _errors(hidden, w)
    print(f"hidden {hidden} {kind}: {err}", flush=True)
    assert err["split"] <= err["f32"] + (0.0 if kind == "random signs" else 2 * 2.0 ** -24)


@pytest.mark.parametrize("hidden,n,extra", [(32, 1, 0), (40, 50, 3), (64, 4000, 40), (256, 33, 0), (256, 4097, 4),
                                             (256, 70, 99)])
def test_team_same_bits(hidden, n, extra, monkeypatch):
    outs = []
    for team in ("0", "1", "2"):
        monkeypatch.setenv("PHZ_POLICY_TEAM", team)
        cl, sim = _sim(hidden, n, extra, 0.02)
        sim.set_policy_weights(_flat(_weights(cl.spec, 6, 1.0)))
        sim.seed_policy(9)
        assert sim.control_kernel_info("policy")["block"] == {"0": 64, "1": 256, "2": 512}[team]
        sim.rollout(0, 3, 2, False)
        outs.append(sim.readback_policy_history(0, 3) + (sim.readback_targets(),) + sim.readback_states())
    for x, y, z in zip(*outs):
        assert np.isfinite(x).all() and np.array_equal(x, y) and np.array_equal(x, z)


@pytest.mark.parametrize("hidden,n", [(112, 65601), (144, 65601), (176, 49200), (200, 32801), (240, 32801)])
def test_parked_two_wave_build_same_bits(hidden, n, monkeypatch):
    """One wave more than the SIMDs, so that the build for two waves per SIMD
    runs, with 2 to 13 tiles of layer 1 parked in LDS: the same bits as the
    one-wave build and as 32-world tiles."""
    outs = []
    for env in ({}, {"PHZ_TWO_WAVES": "0"}, {"PHZ_POLICY_TEAM": "2"}):
        for key in ("PHZ_TWO_WAVES", "PHZ_POLICY_TEAM"):
            monkeypatch.delenv(key, raising=False)
        for key, value in env.items():
            monkeypatch.setenv(key, value)
        cl, sim = _sim(hidden, n, 0, 0.02)
        sim.set_policy_weights(_flat(_weights(cl.spec, 8, 1.0)))
        sim.seed_policy(9)
        info = sim.control_kernel_info("policy")
        assert (info["block"] == 64) == ("PHZ_POLICY_TEAM" not in env)
        if info["block"] == 64:
            assert (info["vgpr"] + max(info["agpr"], 0) <= 256) == (not env), info
        sim.run_policy(0)
        outs.append(sim.readback_policy_history(0, 1) + (sim.readback_targets(),))
        sim.close()
    for x, y, z in zip(*outs):
        assert np.isfinite(x).all() and np.array_equal(x, y) and np.array_equal(x, z)


def test_weights_out_of_range_take_f32_and_back():
    cl, sim = _sim(64, 100)
    w = _weights(cl.spec, 7, 1.0)
    sim.set_policy_std(np.full(8, 1e-30))
    got = []
    for k, first in enumerate((w[2][0, 0], np.inf, w[2][0, 0])):
        w[2][0, 0] = first
        sim.set_policy_weights(_flat(w))
        sim.run_policy(k)
        obs, out = sim.readback_policy_history(k, k + 1)
        h = np.tanh(np.tanh(obs[0] @ w[0].T + w[1]) @ w[2].T + w[3])
        got.append(out[0][:, :8])
        assert np.abs(got[-1] - (h @ w[4].T + w[5])).max() < 1e-5
    assert np.array_equal(got[0], got[2])
