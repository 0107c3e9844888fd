"""A recorded rollout's snapshots and FK readout: the next control step's
observation pass stores a control step's final state and only the last one is
copied; only the last control step's FK readout is stored. Both equal the
calls issued one by one, bit for bit, also for a single control step, for
control steps without physics and for spans recorded in the middle of a
history."""
import numpy as np
import pytest

from tests.test_gpu_policy import ant_policy_setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first,n,every,record", [(0, 1, 3, True), (1, 2, 0, True), (0, 4, 2, True), (1, 3, 1, False)])
def test_rollout_records_as_single_calls(first, n, every, record):
    outs = []
    for manual in (True, False):
        m, sim, spec, *_ = ant_policy_setup(32, 70, history=4)
        sim.enable_state_history(4)
        if manual:
            for c in range(first, first + n):
                sim.run_policy(c)
                sim.step_many(every)
                if record:
                    sim.record_state(c)
        else:
            sim.rollout(first, n, every, record)
        outs.append(sim.readback_state_history(0, 4) + (sim.readback_kinematics(),) + sim.readback_states())
    for x, y in zip(*outs):
        assert np.array_equal(x, y)
