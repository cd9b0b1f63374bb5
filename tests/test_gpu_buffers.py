"""Box transfers of a field between device and host (fx_buf_read_box / fx_buf_write_box
through Field.read_from_device_1d/2d/3d and write_to_device_1d/2d/3d): the elements
moved are exactly those the reference's row loops move (Memory<T>, src/opencl.hpp:532-607:
per component and row, offset min(i*N+n, N*d), length min(x1-x0, N*d-offset)), and no
other element of the host array or the device buffer changes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Nx, Ny, Nz = 12, 7, 5
N = Nx * Ny * Nz


def reference_mask(d, nx, ny, x0, x1, y0, y1, z0, z1, dimension):
    """Elements the reference's loops copy, as a boolean mask over the N*d elements."""
    mask = np.zeros(N * d, bool)
    end = N * d
    comps = range(d) if dimension < 0 else [dimension]
    for z in range(z0, z1):
        for y in range(y0, y1):
            n = x0 + (y + z * ny) * nx
            for i in comps:
                off = min(i * N + n, end)
                length = min(x1 - x0, end - off)
                mask[off:off + length] = True
    return mask


# (form, box, dimension): 1-D (x0, x1), 2-D (x0, x1, y0, y1, Nx, Ny), 3-D (x0, x1, y0, y1, z0, z1, Nx, Ny, Nz)
CASES = [
    ("3d", (2, 9, 1, 6, 1, 4, Nx, Ny, Nz), -1),
    ("3d", (2, 9, 1, 6, 1, 4, Nx, Ny, Nz), 1),
    ("3d", (0, Nx, 0, Ny, 0, Nz, Nx, Ny, Nz), 2),    # one whole component
    ("3d", (11, 12, 6, 7, 4, 5, Nx, Ny, Nz), -1),    # last cell only
    ("3d", (3, 3, 0, Ny, 0, Nz, Nx, Ny, Nz), -1),    # empty rows
    ("3d", (5, 9, 2, 2, 0, Nz, Nx, Ny, Nz), -1),     # no rows
    ("3d", (0, 10, 0, 5, 0, 3, 4, 6, 3), -1),        # rows wider than the pitch overlap
    ("2d", (1, 11, 3, 30, Nx, Ny * Nz), -1),         # 2-D view of the 3-D field
    ("2d", (0, 12, 30, 36, Nx, Ny * Nz), 0),         # rows past component 0 run into component 1
    ("1d", (17, 301, ), -1),
    ("1d", (N - 20, N + 35), -1),                    # last component cut at the end of the buffer
    ("1d", (N - 20, N + 35), 2),
    ("1d", (0, 4 * N), -1),                          # every row cut
]


def transfer(field, form, box, dimension, write):
    fn = getattr(field, ("write_to_device_" if write else "read_from_device_") + form)
    fn(*box, dimension=dimension)


def expand(form, box):
    if form == "1d":
        x0, x1 = box
        return N, 1, x0, x1, 0, 1, 0, 1
    if form == "2d":
        x0, x1, y0, y1, nx, ny = box
        return nx, ny, x0, x1, y0, y1, 0, 1
    x0, x1, y0, y1, z0, z1, nx, ny, _ = box
    return nx, ny, x0, x1, y0, y1, z0, z1


@pytest.mark.parametrize("name,dtype", [("u", np.float32), ("flags", np.uint8)])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_box_read_and_write_move_the_reference_elements(name, dtype, case):
    import fluidx3d_amd as fx
    form, box, dimension = CASES[case]
    lbm = fx.LBM(Nx, Ny, Nz, 0.1)
    try:
        field = getattr(lbm, name)
        d = field.dims
        if dimension >= d:
            pytest.skip("component beyond the field")
        nx, ny, x0, x1, y0, y1, z0, z1 = expand(form, box)
        mask = reference_mask(d, nx, ny, x0, x1, y0, y1, z0, z1, dimension)
        rng = np.random.default_rng(case)
        on_device = rng.integers(1, 250, N * d).astype(dtype)
        on_host = rng.integers(1, 250, N * d).astype(dtype)
        # read: host elements in the box take the device values, the rest keep theirs
        field.host[:] = on_device
        field.write_to_device()
        field.host[:] = on_host
        transfer(field, form, box, dimension, write=False)
        assert np.array_equal(field.host, np.where(mask, on_device, on_host))
        # write: device elements in the box take the host values, the rest keep theirs
        field.host[:] = on_host
        transfer(field, form, box, dimension, write=True)
        field.host[:] = 0
        field.read_from_device()
        assert np.array_equal(field.host, np.where(mask, on_host, on_device))
    finally:
        lbm.close()


def test_box_argument_errors():
    import fluidx3d_amd as fx
    lbm = fx.LBM(Nx, Ny, Nz, 0.1)
    try:
        with pytest.raises(fx.FxError):
            lbm.u.read_from_device_1d(5, 4)                            # x1 < x0
        with pytest.raises(fx.FxError):
            lbm.u.read_from_device_3d(0, 4, 3, 2, 0, 1, Nx, Ny, Nz)   # y1 < y0
        with pytest.raises(fx.FxError):
            lbm.flags.write_to_device_1d(0, 4, dimension=1)            # flags has one component
        with pytest.raises(fx.FxError):
            lbm.u.read_from_device_2d(0, 4, 0, 2, 0, 2)                # Nx = 0
    finally:
        lbm.close()


def test_failed_allocation_is_reported_once():
    """An allocation that cannot be had is an FX_ERR_MEMORY of that call only; the next step
    neither fails nor reports it."""
    import fluidx3d_amd as fx
    from fluidx3d_amd import _abi
    lbm = fx.LBM(Nx, Ny, Nz, 0.05)
    try:
        lbm.run(1)
        with pytest.raises(_abi.FxError) as e:
            lbm.ctx.alloc(1 << 42)
        assert e.value.code == _abi.FX_ERR_MEMORY
        lbm.run(1)
        assert lbm.t == 2
    finally:
        lbm.close()
