"""The kernels of lattices too large for the caches, and the cached ones of mid-sized lattices,
against the oracle: the oracle steps one periodic tile, the GPU a lattice of many copies of it.
Every copy's DDFs are the same bits, and the first copy's are the oracle's.  The sizes lie on
either side of the lines of the dispatch (L2_BYTES = 32 MiB and CACHED_BYTES = 224 MiB of DDFs)."""
import itertools
import os
import shutil
import subprocess

import numpy as np
import pytest

from tests import scenes
from tests.test_gpu_parity import decoded, ext_bits

SETS = {
    "plain": (), "equilibrium": ("EQUILIBRIUM_BOUNDARIES",), "volume_force": ("VOLUME_FORCE",),
    "drag": ("EQUILIBRIUM_BOUNDARIES", "FORCE_FIELD"), "porous": ("VOLUME_FORCE", "POROSITY", "PRECISE_DENSITY"),
    "subgrid": ("EQUILIBRIUM_BOUNDARIES", "SUBGRID"), "moving": ("MOVING_BOUNDARIES",), "moving_subgrid": ("MOVING_BOUNDARIES", "SUBGRID"),
    "all": ("VOLUME_FORCE", "FORCE_FIELD", "EQUILIBRIUM_BOUNDARIES", "UPDATE_FIELDS"),
}
# rows of one block, of half a wave of two-cell lanes, off the cache lines, of several blocks
GRIDS = {"256": (256, 5, 4), "64": (64, 5, 4), "150": (150, 6, 5), "1024": (1024, 3, 2)}
MIB = 1 << 20


def run_tiled(oracle, q, collision, storage, names, tile, at_least):
    import fluidx3d_amd as fx
    Tx, Ty, Tz = tile
    n = Tx * Ty * Tz
    copies = at_least // (n * q * (4 if storage == "FP32" else 2)) + 1
    ky = int(np.sqrt(copies * Tz / Ty)) + 1
    kz = -(-copies // ky)
    rho, u, flags = scenes.random_scene(Tx, Ty, Tz, seed=41, solid_fraction=0.08, equilibrium_faces="EQUILIBRIUM_BOUNDARIES" in names)
    if "PRECISE_DENSITY" in names:
        u *= np.float32(0.02)
    rng = np.random.default_rng(9)
    F = (1e-4 * rng.uniform(-1, 1, 3 * n)).astype(np.float32) if "FORCE_FIELD" in names else None
    alpha = rng.uniform(0, 1, n).astype(np.float32) if "POROSITY" in names else None
    f = (2e-5, -1e-5, 3e-6) if "VOLUME_FORCE" in names else (0.0, 0.0, 0.0)

    def tiled(a):
        return np.tile(a.reshape(-1, Tz, Ty, Tx), (1, kz, ky, 1)).reshape(-1)

    lbm = fx.LBM(Tx, Ty * ky, Tz * kz, 0.03, *f, velocity_set=q, collision=collision, storage=storage, extensions=names)
    ref = oracle.OracleLBM(Tx, Ty, Tz, w=lbm.w, q=q, trt=(collision == "TRT"), storage=storage, ext=ext_bits(names),
                           fx=np.float32(f[0]), fy=np.float32(f[1]), fz=np.float32(f[2]))
    try:
        lbm.rho.host[:], lbm.u.host[:], lbm.flags.host[:] = tiled(rho), tiled(u), tiled(flags)
        ref.rho[:], ref.u[:], ref.flags[:] = rho, u, flags
        if F is not None:
            lbm.F.host[:], ref.F[:] = tiled(F), F
        if alpha is not None:
            lbm.porosity.host[:], ref.alpha[:] = tiled(alpha), alpha
        lbm.initialize()
        ref.initialize()
        for _ in range(3):  # single steps, both parities
            lbm.run(1)
        lbm.run(4)
        ref.step(7)
        code = np.uint32 if storage == "FP32" else np.uint16
        got = lbm.read_ddfs().view(code).reshape(q, kz, Tz, ky, Ty, Tx)
        first = np.ascontiguousarray(got[:, 0, :, 0])
        assert np.array_equal(got, np.broadcast_to(first[:, None, :, None], got.shape)), "copies of the tile differ"
        assert np.array_equal(decoded(storage, first.reshape(-1).view(np.float32 if storage == "FP32" else code), oracle), decoded(storage, ref.fi, oracle))
        if "UPDATE_FIELDS" not in names:
            ref.update_fields()
        lbm.u.read_from_device()
        assert np.array_equal(lbm.u.host.reshape(3, kz, Tz, ky, Ty, Tx)[:, -1, :, -1].reshape(-1), ref.u)
    finally:
        lbm.close()


COMBINATIONS = list(itertools.product((19, 27), ("SRT", "TRT"), ("FP32", "FP16S", "FP16C"), SETS))


@pytest.mark.gpu
@pytest.mark.parametrize("q,collision,storage,ext,grid", [c + (list(GRIDS)[(i + i // 9) % 4],) for i, c in enumerate(COMBINATIONS)])
def test_above_the_caches(oracle, q, collision, storage, ext, grid):
    run_tiled(oracle, q, collision, storage, SETS[ext], GRIDS[grid], 225 * MIB)


@pytest.mark.gpu
@pytest.mark.parametrize("q,collision,storage,ext", [c for c in COMBINATIONS if c[0] == 19 and c[2] != "FP32"])
def test_cached_two_cells_per_lane(oracle, q, collision, storage, ext):
    run_tiled(oracle, q, collision, storage, SETS[ext], GRIDS["256"], 33 * MIB)


@pytest.mark.gpu
@pytest.mark.parametrize("storage,size", itertools.product(("FP32", "FP16S"), (32 * MIB, 224 * MIB)))
def test_lines_of_the_dispatch(oracle, storage, size):
    """The last lattice on the small side of each line (exactly or just below it)."""
    tile = (128, 4, 4)
    run_tiled(oracle, 19, "SRT", storage, (), tile, size - 19 * 128 * 16 * (4 if storage == "FP32" else 2))


PROGRAM = r'''
#include "lbm_launch.hpp"
#include <cstdio>
#include <vector>
int main() {
  using namespace fx;
  unsigned bad = 0;
  for (uint32_t d = 1; d < 5000; d++) { // every multiple and its neighbours up to a few, the largest n
    const Divisor v(d);
    for (uint32_t k = 0; k < 60; k++) for (int e = -1; e <= 1; e++) { const uint32_t n = k * d + (uint32_t)e; if (n < 0x80000000u && v.quotient(n) != n / d) bad++; }
    for (uint32_t n = 0x7FFFFFFFu - 2u * d; n < 0x80000000u; n += d / 7u + 1u) if (v.quotient(n) != n / d) bad++;
  }
  for (uint32_t d : {65535u, 65536u, 65537u, 6180000u, 0x3FFFFFFFu, 0x40000000u, 0x40000001u, 0x7FFFFFFFu, 0x80000000u})
    for (uint32_t n : {0u, 1u, d - 1u, d, 0x3FFFFFFFu, 0x40000000u, 0x7FFFFFFEu, 0x7FFFFFFFu}) if (n < 0x80000000u && Divisor(d).quotient(n) != n / d) bad++;
  for (uint64_t N : {1ull, 255ull, 256ull, 4608ull, 262144ull, 1492425ull, 6181000ull}) {
    const LaunchShape s = slab_shape(N);
    std::vector<int> seen(s.grid.x, 0);
    if (s.grid.x % 8u || (uint64_t)s.grid.x * s.block.x < N || !s.cached || !s.lin) bad++;
    for (uint64_t L = 0; L < s.grid.x; L++) { const uint64_t g = slab_segment(L, s.grid.x); if (g >= s.grid.x || seen[g]++ || g / (s.grid.x / 8u) != L % 8u) bad++; }
  }
  printf("bad %u\n", bad);
  return 0;
}
'''


def test_cell_of_a_block(tmp_path):
    """Division by multiplication (Divisor) below 2^31, and the slabs of slab_segment: each
    segment once, an eighth of them per XCD."""
    src, exe = tmp_path / "p.hip", tmp_path / "p"
    src.write_text(PROGRAM)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    subprocess.run([shutil.which("hipcc") or "/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17",
                    "-I" + os.path.join(root, "fluidx3d_amd", "csrc"), "-I" + os.path.join(root, "include"), str(src), "-o", str(exe)],
                   check=True, capture_output=True, text=True)
    assert subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.strip() == "bad 0"
