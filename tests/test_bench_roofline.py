"""The bytes behind bench.py's roofline figures come from the launches that the library
counted (fx_ctx_launches), one pass over the DDFs each, whatever the rule that chose them."""
import pytest

import bench


def test_bytes_of_the_launches():
    # 3 batches of 20 steps over 1e6 cells, 1 ms each: 20, 10 and (4 in pairs of launches, rest single) 11 launches
    for launches, per_batch in ((60, 20), (30, 10), (33, 11)):
        r = bench.rate_summary(10 ** 6, 153, [1.0, 1.0, 1.0], 20, launches)
        assert r["achieved_GBps"] == pytest.approx(153e6 * per_batch / 1e-3 * 1e-9)
        assert r["steps_per_launch"] == pytest.approx(20 / per_batch)
        assert r["mlups"] == pytest.approx(20e6 / 1e-3 * 1e-6)


# two steps per launch pay at 96^3, not at 48^3; 6 steps: two launches of two and two of one
@pytest.mark.gpu
@pytest.mark.parametrize("size,storage,steps,per_launch", [(96, "FP32", 8, 2.0), (96, "FP32", 6, 1.5), (96, "FP32", 3, 1.0), (48, "FP32", 8, 1.0),
                                                           (96, "FP16S", 8, 1.0)])
def test_steps_per_launch(size, storage, steps, per_launch):
    import fluidx3d_amd as fx
    r = bench.gpu_mode(fx, size, storage, steps, 4, 3, 3)
    assert r["steps_per_launch"] == per_launch and r["finite"]
    moved = fx.bandwidth_bytes_per_cell(fx.make_config(8, 8, 8, 1.0, 19, "SRT", storage)) * size ** 3
    assert r["achieved_GBps"] == pytest.approx(moved / (r["ms_per_step"] * per_launch * 1e-3) * 1e-9)
