"""The kernels of lattices too large for the caches, and the cached ones of mid-sized lattices,
against the oracle: the oracle steps one periodic tile, the GPU a lattice of many copies of it.
Every copy's DDFs are the same bits, and the first copy's are the oracle's.  The sizes lie on
either side of the lines of the dispatch (L2_BYTES = 32 MiB and CACHED_BYTES = 224 MiB of DDFs), and
each test asserts the form of the launches that it is about."""
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


def two_cells(q, collision, storage, ext, cached=False):
    """Kernels with two cells per lane on rows of whole waves (tune_pairs, tune_cached_pairs)."""
    if q != 19 or storage == "FP32" or ext == "all":
        return False
    if ext in ("subgrid", "moving_subgrid"):
        return collision == "SRT" or storage == "FP16S"
    if ext == "volume_force":
        return storage == "FP16S" and (cached or collision == "SRT")
    return ext != "porous" or collision == "TRT" or storage == "FP16C"


class Tiled:
    """A lattice of ky x kz copies of a tile (rows are not tiled), and the tile for the oracle."""

    def __init__(self, oracle, q, collision, storage, names, tile, at_least, copies=None, seed=41):
        import fluidx3d_amd as fx
        Tx, Ty, Tz = tile
        n = Tx * Ty * Tz
        if copies is None:  # DDFs of more than at_least bytes
            copies = at_least // (n * q * (4 if storage == "FP32" else 2)) + 1
            self.ky = int(np.sqrt(copies * Tz / Ty)) + 1
        else:
            self.ky = max(k for k in range(1, int(copies ** 0.5) + 1) if copies % k == 0)
        self.kz = -(-copies // self.ky)
        self.shape, self.q, self.storage = (Tz, Ty, Tx), q, storage
        rho, u, flags = scenes.random_scene(Tx, Ty, Tz, seed=seed, solid_fraction=0.08, equilibrium_faces="EQUILIBRIUM_BOUNDARIES" in names)
        if "PRECISE_DENSITY" in names:
            u *= np.float32(0.02)
        rng = np.random.default_rng(9)
        F = (1e-4 * rng.uniform(-1, 1, 3 * n)).astype(np.float32) if "FORCE_FIELD" in names else None
        alpha = rng.uniform(0, 1, n).astype(np.float32) if "POROSITY" in names else None
        self.f = (2e-5, -1e-5, 3e-6) if "VOLUME_FORCE" in names else (0.0, 0.0, 0.0)
        opts = dict(velocity_set=q, collision=collision, storage=storage, extensions=names)
        self.fields = {"rho": rho, "u": u, "flags": flags, "F": F, "porosity": alpha}
        self.lbm = fx.LBM(Tx, Ty * self.ky, Tz * self.kz, 0.03, *self.f, **opts)
        self.one = lambda: self.fill(fx.LBM(Tx, Ty, Tz, 0.03, *self.f, **opts), lambda a: a)
        self.fill(self.lbm, self.tiled)
        self.ref = oracle.OracleLBM(Tx, Ty, Tz, w=self.lbm.w, q=q, trt=(collision == "TRT"), storage=storage, ext=ext_bits(names),
                                    fx=np.float32(self.f[0]), fy=np.float32(self.f[1]), fz=np.float32(self.f[2]))
        self.ref.rho[:], self.ref.u[:], self.ref.flags[:] = rho, u, flags
        if F is not None:
            self.ref.F[:] = F
        if alpha is not None:
            self.ref.alpha[:] = alpha
        self.lbm.initialize()
        self.ref.initialize()

    def fill(self, lbm, tiled):
        for name, a in self.fields.items():
            if a is not None:
                getattr(lbm, name).host[:] = tiled(a)
        return lbm

    def tiled(self, a):
        return np.tile(a.reshape(-1, *self.shape), (1, self.kz, self.ky, 1)).reshape(-1)

    def first(self, a):
        """The first copy of a field, which every other copy equals."""
        Tz, Ty, Tx = self.shape
        a = a.reshape(-1, self.kz, Tz, self.ky, Ty, Tx)
        first = np.ascontiguousarray(a[:, 0, :, 0])
        assert np.array_equal(a, np.broadcast_to(first[:, None, :, None], a.shape)), "copies of the tile differ"
        return first.reshape(-1)

    def first_ddfs(self):
        code = np.uint32 if self.storage == "FP32" else np.uint16
        return self.first(self.lbm.read_ddfs().view(code)).view(np.float32 if self.storage == "FP32" else code)

    def close(self):
        self.lbm.close()


def run_tiled(oracle, q, collision, storage, names, tile, at_least, expect, copies=None):
    """Single steps, a run of four, and the fields; `expect(form)` of every single step's launch."""
    t = Tiled(oracle, q, collision, storage, names, tile, at_least, copies)
    lbm, ref = t.lbm, t.ref
    try:
        for _ in range(3):  # single steps, both parities
            lbm.run(1)
            assert expect(lbm.ctx.launches().step_form)
        lbm.run(4)
        ref.step(7)
        assert np.array_equal(decoded(storage, t.first_ddfs(), oracle), decoded(storage, ref.fi, oracle))
        if "UPDATE_FIELDS" not in names:
            ref.update_fields()
        lbm.u.read_from_device()
        lbm.rho.read_from_device()
        assert np.array_equal(t.first(lbm.u.host), ref.u) and np.array_equal(t.first(lbm.rho.host), ref.rho)
    finally:
        t.close()


COMBINATIONS = list(itertools.product((19, 27), ("SRT", "TRT"), ("FP32", "FP16S", "FP16C"), SETS))


CACHED, TWO_CELLS, LINEAR, XCD_ROWS = 2, 4, 8, 16  # FX_FORM_


@pytest.mark.gpu
@pytest.mark.parametrize("grid", GRIDS)
@pytest.mark.parametrize("q,collision,storage,ext", COMBINATIONS)
def test_above_the_caches(oracle, q, collision, storage, ext, grid):
    pairs = grid in ("256", "1024") and two_cells(q, collision, storage, ext)
    linear = grid == "150"
    run_tiled(oracle, q, collision, storage, SETS[ext], GRIDS[grid], 225 * MIB,
              lambda form: (form & (CACHED | TWO_CELLS | LINEAR)) == (TWO_CELLS if pairs else LINEAR if linear else 0))


@pytest.mark.gpu
@pytest.mark.parametrize("q,collision,storage,ext", [c for c in COMBINATIONS if c[0] == 19 and c[2] != "FP32"])
def test_cached_two_cells_per_lane(oracle, q, collision, storage, ext):
    pairs = two_cells(q, collision, storage, ext, cached=True)
    run_tiled(oracle, q, collision, storage, SETS[ext], GRIDS["256"], 33 * MIB, lambda form: (form & (CACHED | TWO_CELLS)) == CACHED | (TWO_CELLS if pairs else 0))


@pytest.mark.gpu
@pytest.mark.parametrize("beyond", [False, True])
@pytest.mark.parametrize("storage,line", itertools.product(("FP32", "FP16S"), (32 * MIB, 224 * MIB)))
def test_lines_of_the_dispatch(oracle, storage, line, beyond):
    """The last lattice on the small side of each line and the first beyond it."""
    tile = (128, 4, 4)
    per_copy = 19 * 128 * 16 * (4 if storage == "FP32" else 2)
    cached = line == 32 * MIB or not beyond
    pairs = storage != "FP32" and (line > 32 * MIB or beyond)
    run_tiled(oracle, 19, "SRT", storage, (), tile, None, lambda form: (form & (CACHED | TWO_CELLS | LINEAR)) ==
              (CACHED if cached else 0) | (TWO_CELLS if pairs else LINEAR if cached else 0), copies=line // per_copy + beyond)


ADJOINT_SETS = {"porosity": ("VOLUME_FORCE", "POROSITY"), "precise": ("VOLUME_FORCE", "POROSITY", "PRECISE_DENSITY"),
                "all": ("VOLUME_FORCE", "POROSITY", "FORCE_FIELD", "EQUILIBRIUM_BOUNDARIES", "PRECISE_DENSITY")}
# 225 MiB of FP32 DDFs: record pass and adjoint step for arrays from HBM, the moments past the caches
# (MOMENTS_STREAM); 180: the record pass cached, the moments past the caches for D3Q19; 120: the
# record pass cached, the adjoint step (two FP32 arrays) not; 60: both on slabs
ADJOINT_SIZES = {225: (0, 0), 180: (CACHED, 0), 120: (CACHED, 0), 60: (CACHED, CACHED)}


ADJOINT_CASES = [(q, c, st, e, m, g) for q, c, st, e, m in itertools.product((19, 27), ("SRT", "TRT"), ("FP32", "FP16C"), ADJOINT_SETS, ADJOINT_SIZES)
                 if st == "FP32" or m == 225 for g in (GRIDS if m == 225 and st == "FP32" else ("150", "256"))]


@pytest.mark.gpu
@pytest.mark.parametrize("q,collision,storage,ext,mib,grid", ADJOINT_CASES)
def test_record_and_adjoint_step(oracle, q, collision, storage, ext, mib, grid):
    """One record pass and one adjoint step against the oracle: the record pass's DDFs bit for
    bit, the adjoint populations and the gradient against the FP64 oracle's adjoint step of the tile, with
    the bounds of tests/test_gpu_adjoint.py (FP32 arithmetic against FP64)."""
    import ctypes
    from fluidx3d_amd import _abi
    names = ADJOINT_SETS[ext]
    t = Tiled(oracle, q, collision, storage, names, GRIDS[grid], mib * MIB)
    lbm, ref = t.lbm, t.ref
    Tx, Ty, Tz = GRIDS[grid]
    n = Tx * Ty * Tz
    try:
        lbm.run(3)
        ref.step(3)
        state = decoded(storage, t.first_ddfs(), oracle)
        assert np.array_equal(state, decoded(storage, ref.fi, oracle))
        L, rng = lbm.ctx.lib, np.random.default_rng(11)
        moments = lbm.ctx.alloc(16 * lbm.N)
        lam, grad = lbm.ctx.alloc(4 * q * lbm.N), lbm.ctx.alloc(4 * lbm.N)
        step = (lbm.rho.device, lbm.u.device, lbm.flags.device, 3, *t.f, lbm._ptr(lbm.F), lbm.porosity.device)
        _abi.check(L.fx_lbm_stream_collide_record(lbm.ctx.h, lbm.fi, *step, moments))
        ref.step(1)
        assert np.array_equal(decoded(storage, t.first_ddfs(), oracle), decoded(storage, ref.fi, oracle)), "record pass"
        lam1 = rng.standard_normal(q * n).astype(np.float32)
        lbm.ctx.write(lam, t.tiled(lam1))
        lbm.ctx.fill(grad, 4 * lbm.N, 0)
        plane_x, weight = Tx - 2, 0.25
        _abi.check(L.fx_lbm_adjoint_step(lbm.ctx.h, lam, *step, moments, plane_x, weight, grad))
        forms = lbm.ctx.launches()
        if storage == "FP32":
            assert (forms.record_form & CACHED, forms.adjoint_form & CACHED) == ADJOINT_SIZES[mib]
        else:
            assert not (forms.record_form | forms.adjoint_form) & CACHED
        g_lam, g_grad = np.empty(q * lbm.N, np.float32), np.empty(lbm.N, np.float32)
        lbm.ctx.read(lam, g_lam)
        lbm.ctx.read(grad, g_grad)
        g_lam, g_grad = t.first(g_lam), t.first(g_grad)
        o = oracle.OracleLBM(Tx, Ty, Tz, w=lbm.w, q=q, trt=collision == "TRT", storage="FP64", ext=ext_bits(names), fx=t.f[0], fy=t.f[1], fz=t.f[2])
        o.rho[:], o.u[:], o.flags[:], o.alpha[:] = t.fields["rho"], t.fields["u"], t.fields["flags"], t.fields["porosity"]
        if o.F is not None:
            o.F[:] = t.fields["F"]
        o_lam, o_grad, state = lam1.astype(np.float64), np.zeros(n), state.astype(np.float64)
        rc = oracle.lib().fxo_adjoint_step(ctypes.byref(o.cfg), oracle._ptr(state), oracle._ptr(o_lam), o.flags_ptr, 3, *t.f, oracle._ptr(o.F), oracle._ptr(o.alpha),
                                           plane_x, weight, oracle._ptr(o_grad), oracle._ptr(o.rho), oracle._ptr(o.u))
        assert rc == 0
        assert np.max(np.abs(g_lam - o_lam)) < 2e-6 * np.max(np.abs(o_lam))
        assert np.max(np.abs(g_grad - o_grad)) < 2e-5 * np.max(np.abs(o_grad))
    finally:
        t.close()


@pytest.mark.gpu
@pytest.mark.parametrize("grid", ["150", "256"])
@pytest.mark.parametrize("q,collision,storage", [(19, "SRT", "FP32"), (19, "TRT", "FP16S"), (27, "SRT", "FP16C"), (27, "TRT", "FP32")])
def test_gradient_of_a_tiled_lattice(oracle, q, collision, storage, grid):
    """The objective is a sum over the copies, so each copy's gradient is that of the tile alone
    (slabs, which tests/test_gpu_adjoint.py checks against FP64), bit for bit: checkpointed forward
    and backward with the kernels for arrays from HBM, the first record step out of place."""
    from fluidx3d_amd.adjoint import Adjoint
    names = ADJOINT_SETS["all"]
    t = Tiled(oracle, q, collision, storage, names, GRIDS[grid], 225 * MIB)
    one = t.one()
    try:
        results = []
        for lbm in (one, t.lbm):
            adj = Adjoint(lbm, steps=13, window_begin=8, plane_x=lbm.Nx - 2, checkpoint_interval=5)
            results.append((adj.forward(), adj.backward()))
            adj.close()
        forms = t.lbm.ctx.launches()
        assert not (forms.record_form | forms.adjoint_form | forms.step_form) & CACHED
        (J1, g1), (J, g) = results
        assert np.abs(g1).max() > 0 and np.array_equal(t.first(g), g1)
        assert abs(J - t.ky * t.kz * J1) <= 1e-9 * abs(J)  # FP64 sums in another order, with cancellation
    finally:
        one.close()
        t.close()


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
  for (uint64_t b = 1; b < 1000; b++) { // XCDs with blocks of the lattice, not only padding (slab_segment's comment)
    const LaunchShape s = slab_shape(b * 256);
    unsigned used = 0;
    for (uint64_t xcd = 0; xcd < 8; xcd++) used += slab_segment(xcd, s.grid.x) < b;
    if ((b == 18 && used != 3) || (b == 65 && used != 5) || (b == 392 && used == 8) || (b > 392 && used != 8)) bad++;
  }
  printf("bad %u\n", bad);
  return 0;
}
'''


def test_cell_of_a_block(tmp_path):
    """Division by multiplication (Divisor) below 2^31, and the slabs of slab_segment: each
    segment of the padded grid once, an eighth of them per XCD."""
    src, exe = tmp_path / "p.hip", tmp_path / "p"
    src.write_text(PROGRAM)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    subprocess.run([shutil.which("hipcc") or "/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17",
                    "-I" + os.path.join(root, "fluidx3d_amd", "csrc"), "-I" + os.path.join(root, "include"), str(src), "-o", str(exe)],
                   check=True, capture_output=True, text=True)
    assert subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.strip() == "bad 0"
