"""Lattices that are stepped in turn on one device share its last-level cache.  A single step of a
lattice whose DDFs the others drove out takes the launch for DDFs from HBM; with the
others idle, for runs of several steps and for programs that look at the fields after every
step the launch for cached DDFs stays.  The bits do not depend on it."""
import numpy as np
import pytest

from tests import scenes
from tests.test_gpu_parity import compare_state, setup_pair

pytestmark = pytest.mark.gpu


def cached(lbm):
    from fluidx3d_amd import _abi
    return bool(lbm.ctx.launches().step_form & _abi.FX_FORM_CACHED)


@pytest.mark.parametrize("q,collision,storage,size", [(19, "SRT", "FP16S", (128, 9, 7)), (19, "TRT", "FP16C", (256, 5, 4)), (27, "SRT", "FP32", (64, 9, 7)),
                                                      (19, "SRT", "FP32", (32, 12, 10))])
def test_single_steps_beside_other_lattices(oracle, crowd, q, collision, storage, size):
    rho, u, flags = scenes.random_scene(*size, seed=3)
    lbm, ref = setup_pair(oracle, *size, 0.05, q, collision, storage, (), rho, u, flags)
    try:
        lbm.initialize()
        ref.initialize()

        def expect(want, steps=1):
            lbm.run(steps)
            ref.step(steps)
            assert cached(lbm) == want
            compare_state(lbm, ref, oracle, storage, f"t={lbm.t}")

        expect(True)                     # alone since it was created
        for _ in range(3):
            crowd.lbm.run(1)
            expect(False)
        expect(True)                     # again alone
        crowd.lbm.run(1)
        expect(True, 2)                  # in the cache from the first step to the second
        crowd.lbm.run(1)
        expect(False)
        lbm.update_fields()
        for _ in range(2):               # a program that looks at the fields after every step
            crowd.lbm.run(1)
            expect(True)
            lbm.update_fields()
        ref.update_fields()
        lbm.u.read_from_device()
        assert np.array_equal(lbm.u.host, ref.u)
    finally:
        lbm.close()


def test_rows_off_half_lines_keep_the_cached_launch(crowd):
    import fluidx3d_amd as fx
    lbm = fx.LBM(150, 9, 7, 0.05)
    try:
        lbm.initialize()
        crowd.run(lbm, cached=True)
    finally:
        lbm.close()


def test_split_lattice():
    """Two domains of 155 MiB on one device, stepped in turn."""
    from fluidx3d_amd.domains import DomainLBM
    many = DomainLBM(128, 128, 256, 1, 1, 2, 0.05)
    try:
        many.run(2)
        assert [cached(L) for L in many.domains] == [False, False]
    finally:
        many.close()


def test_other_lattices_that_are_idle_or_small_do_not_count(crowd):
    import fluidx3d_amd as fx
    a, b = fx.LBM(64, 32, 32, 0.05), fx.LBM(64, 32, 32, 0.05)
    try:
        for _ in range(3):               # the crowd exists, and is not stepped
            a.run(1)
            b.run(1)
            assert cached(a) and cached(b)
    finally:
        a.close()
        b.close()
