"""Which form of the policy kernel a launch takes (phz_sim::team_columns), on
both sides of each line, from a host-only sim: one wave per tile (block 64),
four waves per 16-world tile or eight per 32-world tile."""
import dataclasses

import numpy as np
import pytest

from phyz_amd import workloads as W
from phyz_amd.policy import QMinus
from phyz_amd.sim import from_control_loop


def _form(n_in, hidden, n_out, n):
    cl = W.control_loop(hidden)
    obs = list(cl.spec.obs)[:n_in] + [QMinus(6 + k % 8, 0.0) for k in range(n_in - 29)]
    spec = dataclasses.replace(cl.spec, obs=obs, input_noise=[0.01] * n_in, act_slots=[k % 8 for k in range(n_out)],
                               history_steps=1)
    cl = dataclasses.replace(cl, spec=spec, weights=np.zeros(spec.n_weights()), std=np.full(n_out, 0.2))
    sim = from_control_loop(cl, "f32", nworld=n, device=-1)
    sim.compile()
    i = sim.control_kernel_info("policy")
    return {(64, i["worlds_per_block"]): 0, (256, 16): 1, (512, 32): 2}[i["block"], i["worlds_per_block"]]


@pytest.mark.parametrize("shape,forms", [
    ((29, 16, 8), (0, 0, 0, 0, 0, 0, 0, 0)),     # below 32 neurons: f32 layers, one wave per tile
    ((29, 32, 8), (1, 1, 2, 2, 1, 1, 0, 0)),
    ((29, 64, 8), (1, 1, 2, 2, 1, 1, 1, 0)),
    ((128, 32, 32), (1, 1, 2, 2, 1, 1, 0, 0)),
    ((29, 128, 8), (1, 1, 2, 2, 1, 1, 1, 0)),
    ((29, 129, 8), (1, 1, 2, 2, 2, 0, 0, 0)),
    ((29, 256, 8), (1, 1, 2, 2, 2, 0, 0, 0)),
    ((128, 256, 8), (1, 1, 2, 2, 2, 0, 0, 0)),   # 30.0 us at 4096 in 16-world tiles, 31.8 in 32-world ones
    ((60, 256, 32), (1, 1, 2, 2, 2, 0, 0, 0)),
    ((128, 256, 32), (2, 2, 2, 2, 2, 0, 0, 0)),  # 32 worlds a block at every size (36.5 us at 4096 in 16, 38.0)
])
def test_form_by_size(shape, forms, monkeypatch):
    monkeypatch.delenv("PHZ_POLICY_TEAM", raising=False)
    assert tuple(_form(*shape, n) for n in (1, 4096, 4097, 8192, 16384, 20480, 24576, 24577)) == forms
