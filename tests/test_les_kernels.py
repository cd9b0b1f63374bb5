"""The kernel subsets with SUBGRID and MOVING_BOUNDARIES against the oracle, bit for bit: on
slabs in the caches, and, where another lattice crowds the cache, with two cells per lane for
the D3Q19 16-bit formats on rows of whole waves (256 cells) and one cell per lane through buffer
instructions on rows of half a wave (64)."""
import itertools

import numpy as np
import pytest

from tests import scenes
from tests.test_gpu_parity import compare_state, setup_pair, step

SETS = {"subgrid": ("EQUILIBRIUM_BOUNDARIES", "SUBGRID"), "moving": ("MOVING_BOUNDARIES",),
        "moving_subgrid": ("EQUILIBRIUM_BOUNDARIES", "FORCE_FIELD", "MOVING_BOUNDARIES", "SUBGRID")}


@pytest.mark.gpu
@pytest.mark.parametrize("size,crowded", [((256, 5, 4), False), ((64, 5, 4), False), ((150, 6, 5), False), ((256, 5, 4), True), ((64, 5, 4), True)],
                         ids=lambda s: str(s[0]) if isinstance(s, tuple) else "crowded" if s else "alone")
@pytest.mark.parametrize("q,collision,storage,ext", list(itertools.product((19, 27), ("SRT", "TRT"), ("FP16S", "FP16C"), SETS)))
def test_les_kernels_match_oracle(oracle, crowd, q, collision, storage, ext, size, crowded):
    Nx, Ny, Nz = size
    names = SETS[ext]
    rho, u, flags = scenes.random_scene(Nx, Ny, Nz, seed=31, solid_fraction=0.05, equilibrium_faces="EQUILIBRIUM_BOUNDARIES" in names)
    x, y, z = scenes.coords(Nx, Ny, Nz)
    flags[(y == 1) & (x < 128)] = scenes.TYPE_S               # a row's first wave
    flags[(y == 2) & (z == 3) & (x >= 128)] = scenes.TYPE_S   # a row's last wave (the +x wrap's source)
    flags[(y == 3) & (x % 8 < 2)] = scenes.TYPE_S             # lanes with both cells solid
    N = Nx * Ny * Nz
    F = (1e-4 * np.random.default_rng(7).uniform(-1, 1, 3 * N)).astype(np.float32) if "FORCE_FIELD" in names else None
    lbm, ref = setup_pair(oracle, Nx, Ny, Nz, 0.01, q, collision, storage, names, rho, u, flags, F)
    try:
        lbm.initialize()
        ref.initialize()
        if "MOVING_BOUNDARIES" in names:
            assert (ref.flags & 3 == 3).any()
        for s in range(6):
            step(lbm, crowd if crowded else None)
            if crowded:  # FX_FORM_TWO_CELLS, and pair_extensions
                two_cells = q == 19 and Nx == 256 and not (collision == "TRT" and storage == "FP16C" and "SUBGRID" in names)
                assert bool(lbm.ctx.launches().step_form & 4) == two_cells
            ref.step(1)
            compare_state(lbm, ref, oracle, storage, f"after step {s + 1}")
        lbm.u.read_from_device()
        ref.update_fields()
        assert np.array_equal(lbm.u.host, ref.u)
    finally:
        lbm.close()
