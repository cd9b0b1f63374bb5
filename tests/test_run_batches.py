"""LBM.run queues its steps in calls of at most STEPS_PER_CALL: an interrupt or an error between
two calls leaves t at the steps that were queued, and nothing more is queued (no GPU: the
library is a stand-in that records the calls)."""
import types

import pytest

from fluidx3d_amd import lbm as module
from fluidx3d_amd.lbm import LBM


def stand_in(fail_at=None, error=KeyboardInterrupt):
    calls = []

    def fx_lbm_run(h, fi, rho, u, flags, t, steps, *rest):
        if len(calls) == fail_at:
            raise error
        calls.append((t, steps))
        return 0

    lbm = LBM.__new__(LBM)
    field = types.SimpleNamespace(device=1)
    lib = types.SimpleNamespace(fx_lbm_run=fx_lbm_run)
    lbm.ctx = types.SimpleNamespace(lib=lib, h=1, sync=lambda: calls.append("sync"))
    lbm.rho = lbm.u = lbm.flags = field
    lbm.F = lbm.porosity = None
    lbm.fi, lbm.fx, lbm.fy, lbm.fz, lbm.extensions = 1, 0.0, 0.0, 0.0, 0
    lbm.initialized, lbm.t = True, 5
    return lbm, calls


@pytest.mark.parametrize("steps", [0, -3, 1, 999, 1000, 1001, 2500])
def test_calls_cover_the_steps(steps):
    lbm, calls = stand_in()
    lbm.run(steps)
    assert calls.pop() == "sync" and lbm.t == 5 + max(steps, 0)
    t = 5
    for start, n in calls:
        assert start == t and 0 < n <= module.STEPS_PER_CALL
        t += n
    assert t == lbm.t and all(n % 4 == 0 for _, n in calls[:-1])


def test_interrupt_between_calls():
    lbm, calls = stand_in(fail_at=2)
    with pytest.raises(KeyboardInterrupt):
        lbm.run(1_000_000)
    assert lbm.t == 5 + 2 * module.STEPS_PER_CALL and len(calls) == 2
