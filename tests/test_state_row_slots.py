"""Sizes of the pinned slots that state rows pass through (phz_sim::slot_bytes).

A sim's calls move rows of different widths. Slots sized by each call's own
width differ by a few pages, and a later call that outgrows them waits for the
queued span, frees them and pins new ones; so one size serves them all."""
import pytest

from phyz_amd import _lib
from phyz_amd import workloads as W
from phyz_amd.sim import from_workload

KB = 1024


def _bytes(sim, width, f64):
    return _lib.load().phz_staging_bytes(sim._h, width, 1 if f64 else 0)


# The ant: 42 values a world up, 28 down, 72 contact values; the chain 21 and 14.
@pytest.mark.parametrize("index,prec,nworld", [
    (3, "f32", 131072), (3, "f32", 4096), (3, "f32", 300), (3, "f32", 1),
    (2, "f64", 65536), (2, "f64", 6272), (2, "f64", 96), (2, "f32", 65536), (5, "f64", 16384), (4, "f32", 32768),
])
def test_no_call_outgrows_the_first(index, prec, nworld):
    sim = from_workload(W.config(index), prec, nworld=nworld, device=-1)
    f64 = prec == "f64"
    first = _bytes(sim, 0, f64)
    widths = [2 * sim.nq + sim.nctrl, 2 * sim.nq, sim.nq, 1] + ([8 * sim.nb] if W.config(index).contact else [])
    assert [_bytes(sim, w, f64) for w in widths] == [first] * len(widths)
    # At most the state: four slots of 128 K values, and little for few worlds.
    assert first <= 4 * 128 * KB * (8 if f64 else 4)
    assert first <= 4 * max(4 * KB, 2 * (-(-nworld // 64) * 64 * max(widths) * (8 if f64 else 4) + 5 * KB))


def test_wide_rows_take_a_tile():
    """A tile of 64 worlds that exceeds the slot's values is the slot's size;
    a width in between rounds up to no more than the full size."""
    sim = from_workload(W.config(6), "f32", nworld=1000, device=-1)
    assert _bytes(sim, 4096, True) >= 4 * 64 * 4096 * 8
    assert _bytes(sim, 54 * sim.nb, False) <= 4 * 128 * KB * 4
    assert _bytes(from_workload(W.config(2), "f32", nworld=0, device=-1), 14, False) == 0
