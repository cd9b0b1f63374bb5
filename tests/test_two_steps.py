"""fx_lbm_run takes FP32 lattices two steps per launch (k_two_steps, lbm_two_steps.hpp) where
that pays.  CPU: the launch shapes (two_step_shape) cover every cell once within the kernel's
limits, and the rule (two_steps_pay) excludes what the kernel does not do.  GPU: the DDFs
after a run equal those of single steps (fx_lbm_stream_collide) bit for bit, on lattices with
clipped tiles, idle lanes, several segments and rows off the cache lines, at both parities and
with 0 to 3 single steps left over; the oracle for one lattice; the adjoint's forward pass."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from tests import scenes

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

PROGRAM = r'''
#include "lbm_launch.hpp"
#include <cstdio>
#include <vector>
int main() {
  using namespace fx;
  unsigned bad = 0, shapes = 0;
  for (unsigned cus : {1u, 104u, 256u}) for (unsigned nx : {1u, 31u, 33u, 63u, 64u, 65u, 96u, 127u, 128u, 129u, 200u, 257u, 385u})
    for (unsigned ny : {1u, 2u, 4u, 5u, 6u, 13u, 27u, 64u}) for (unsigned nz : {1u, 2u, 5u, 16u, 37u}) {
      const TwoStepShape s = two_step_shape(nx, ny, nz, cus);
      const unsigned TX = s.wide ? 128u : 64u, TY = s.wide ? 5u : 13u;
      shapes++;
      if (s.width == 0 || s.width > TX || s.height == 0 || s.height > TY || two_step_threads(TX, s.height) > 1024u || s.grid < s.tiles || s.grid % 8u) bad++;
      std::vector<int> seen((size_t)nx * ny * nz, 0), started(s.tiles, 0);
      for (unsigned b = 0; b < s.grid; b++) { // the kernel's block -> tile map
        const unsigned per = s.grid >> 3, tile = (b & 7u) * per + (b >> 3);
        if (tile >= s.tiles) continue;
        started[tile]++;
        const unsigned tx = tile % s.tiles_x, tr = tile / s.tiles_x, ty = tr % s.tiles_y, tz = tr / s.tiles_y;
        const unsigned x0 = tx * s.width, y0 = ty * s.height, z0 = tz * s.zlen;
        if (x0 >= nx || y0 >= ny || z0 >= nz) { bad++; continue; }
        for (unsigned z = z0; z < z0 + s.zlen && z < nz; z++) for (unsigned y = y0; y < y0 + s.height && y < ny; y++)
          for (unsigned x = x0; x < x0 + s.width && x < nx; x++) seen[((size_t)z * ny + y) * nx + x]++;
      }
      for (int v : started) bad += v != 1;
      for (int v : seen) bad += v != 1;
    }
  printf("shapes %u bad %u\n", shapes, bad);
  auto pay = [](unsigned nx, unsigned ny, unsigned nz, unsigned q, bool trt, unsigned ext) {
    return (int)two_steps_pay(two_step_shape(nx, ny, nz, 256), nx, ny, nz, q, trt, ext);
  };
  printf("pay %d%d%d%d%d%d%d%d%d%d%d%d%d%d%d%d\n",
         pay(256, 256, 256, 19, false, 0), pay(64, 64, 64, 19, false, 0), pay(128, 64, 64, 19, false, 0), // L2_BYTES
         pay(80, 80, 80, 19, false, 0), pay(96, 96, 96, 19, false, 0), pay(96, 96, 96, 19, true, EXT_VOLUME_FORCE),
         pay(128, 128, 128, 19, true, EXT_VOLUME_FORCE), pay(128, 128, 128, 19, true, EXT_VOLUME_FORCE | EXT_POROSITY),
         pay(201, 75, 120, 19, false, 0), pay(201, 75, 99, 19, false, 0), // both arrays in the cache or not
         pay(130, 170, 170, 19, false, 0), pay(160, 160, 160, 19, false, 0), // above CACHED_BYTES
         pay(16, 1024, 250, 19, false, 0), pay(2000, 2000, 3, 19, false, 0), pay(2000, 1, 2000, 19, false, 0),
         pay(200, 200, 200, 27, true, EXT_VOLUME_FORCE));
  for (int q : {19, 27}) for (unsigned st : {ST_FP32, ST_FP16S, ST_FP16C}) for (unsigned ext : {0u, (unsigned)EXT_FORCE_FIELD, (unsigned)EXT_POROSITY, (unsigned)EXT_UPDATE_FIELDS, (unsigned)EXT_MOVING_BOUNDARIES, (unsigned)EXT_SUBGRID}) {
    const bool k = q == 19 ? tune_two_steps(19, st, true, ext ? EXT_ALL : 0u) : tune_two_steps(27, st, false, ext ? EXT_ALL : 0u);
    if (k != (st == ST_FP32 && ext == 0u)) printf("tune %d %u %u\n", q, st, ext);
  }
  return 0;
}
'''


@pytest.fixture(scope="module")
def lines(tmp_path_factory):
    d = tmp_path_factory.mktemp("two")
    src = d / "p.hip"
    src.write_text(PROGRAM)
    exe = d / "p"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17", "-I" + os.path.join(ROOT, "fluidx3d_amd", "csrc"),
                    "-I" + os.path.join(ROOT, "include"), str(src), "-o", str(exe)], check=True, capture_output=True, text=True)
    return subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.splitlines()


def test_shapes_cover_every_cell_once(lines):
    assert lines[0].startswith("shapes ") and lines[0].endswith(" bad 0"), lines[0]


def test_rule(lines):
    assert lines[1:] == ["pay 1010101001010000"], lines


POROUS = ("VOLUME_FORCE", "POROSITY", "PRECISE_DENSITY")
EQ_FF = ("EQUILIBRIUM_BOUNDARIES", "FORCE_FIELD")
# (size, q, collision, extensions): every kernel, on lattices that the rule takes but for one
CASES = [
    ((128, 61, 58), 19, "SRT", ()),              # one tile across, clipped in y and z
    ((64, 143, 51), 19, "SRT", ()),              # 64-wide tiles
    ((50, 143, 63), 19, "SRT", ()),              # 14 lanes idle
    ((321, 81, 34), 19, "SRT", ()),              # three tiles across, the last of 65 cells
    ((350, 81, 82), 19, "SRT", ()),              # 91 %, one array of two in the caches
    ((300, 2, 800), 19, "SRT", ()),              # rows 0 and 1 are each other's neighbours twice
    ((300, 400, 4), 19, "SRT", ()),
    ((128, 64, 61), 19, "TRT", ()),
    ((257, 151, 84), 19, "SRT", ()),             # above CACHED_BYTES, 66 %
    ((129, 64, 60), 27, "SRT", ()),              # 51 % of the lanes: single steps
    ((250, 50, 37), 27, "TRT", ()),
    ((240, 41, 53), 19, "SRT", EQ_FF),
    ((100, 73, 61), 19, "TRT", ("EQUILIBRIUM_BOUNDARIES",)),
    ((128, 64, 45), 27, "TRT", EQ_FF),
    ((251, 53, 39), 19, "SRT", ("VOLUME_FORCE",)),
    ((120, 91, 47), 19, "TRT", ("VOLUME_FORCE",)),
    ((125, 191, 97), 27, "TRT", ("VOLUME_FORCE",)),   # above CACHED_BYTES from here
    ((125, 191, 131), 19, "SRT", POROUS),
    ((123, 191, 133), 19, "TRT", POROUS),
    ((254, 71, 131), 27, "TRT", POROUS),
    ((160, 170, 133), 19, "SRT", ("SUBGRID",)),
    ((128, 70, 61), 19, "SRT", ("EQUILIBRIUM_BOUNDARIES", "SUBGRID")),
    ((128, 140, 173), 19, "TRT", ("EQUILIBRIUM_BOUNDARIES", "SUBGRID")),
    ((240, 40, 53), 19, "SRT", ("MOVING_BOUNDARIES",)),
    ((100, 63, 57), 27, "SRT", ("MOVING_BOUNDARIES", "FORCE_FIELD", "EQUILIBRIUM_BOUNDARIES")),
    ((128, 191, 97), 27, "TRT", ("MOVING_BOUNDARIES", "SUBGRID")),
]
SINGLE_STEPS = [((129, 64, 60), 27, "SRT", ())]


def test_rule_of_the_cases(tmp_path):
    """two_steps_pay takes every lattice of CASES but SINGLE_STEPS, and the kernel subsets that have
    a k_two_steps are all FP32 ones but the one with every extension."""
    bits = {"VOLUME_FORCE": 1, "FORCE_FIELD": 2, "EQUILIBRIUM_BOUNDARIES": 4, "POROSITY": 16, "PRECISE_DENSITY": 32, "MOVING_BOUNDARIES": 64, "SUBGRID": 128}
    rows = "".join("{%d,%d,%d,%d,%d,%d}," % (*size, q, collision == "TRT", sum(bits[e] for e in ext)) for size, q, collision, ext in CASES)
    program = r'''
#include "lbm_launch.hpp"
#include <cstdio>
using namespace fx;
template<int Q, bool TRT, uint32_t EXT> void tune() {
  printf("%d%d%d ", (int)tune_two_steps(Q, ST_FP32, TRT, EXT), (int)tune_two_steps(Q, ST_FP16S, TRT, EXT), (int)tune_two_steps(Q, ST_FP16C, TRT, EXT));
}
template<uint32_t EXT> void tune_all() { tune<19, false, EXT>(); tune<19, true, EXT>(); tune<27, false, EXT>(); tune<27, true, EXT>(); }
int main() {
  constexpr uint32_t E = EXT_EQUILIBRIUM_BOUNDARIES, FF = EXT_FORCE_FIELD, VF = EXT_VOLUME_FORCE, POROUS = VF | EXT_POROSITY | EXT_PRECISE_DENSITY;
  tune_all<0u>(); tune_all<E>(); tune_all<VF>(); tune_all<E | FF>(); tune_all<POROUS>(); tune_all<EXT_LES>(); tune_all<EXT_LES_MOVING>();
  printf("\n");
  tune_all<EXT_ALL>();
  printf("\n");
  const unsigned cases[][6] = {ROWS};
  for (const auto& c : cases) printf("%d", (int)two_steps_pay(two_step_shape(c[0], c[1], c[2], 256), c[0], c[1], c[2], c[3], c[4], c[5]));
  return 0;
}
'''.replace("ROWS", rows)
    src, exe = tmp_path / "p.hip", tmp_path / "p"
    src.write_text(program)
    subprocess.run([HIPCC, "--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17", "-I" + os.path.join(ROOT, "fluidx3d_amd", "csrc"),
                    "-I" + os.path.join(ROOT, "include"), str(src), "-o", str(exe)], check=True, capture_output=True, text=True)
    subsets, everything, taken = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.splitlines()
    assert set(subsets.split()) == {"100"} and set(everything.split()) == {"000"}
    assert taken == "".join("0" if c in SINGLE_STEPS else "1" for c in CASES)


def scene_lbm(fx, size, q, collision, extensions, nu=0.03):
    rho, u, flags = scenes.random_scene(*size, seed=5, equilibrium_faces="EQUILIBRIUM_BOUNDARIES" in extensions)
    force = (1e-4, -2e-4, 3e-4) if "VOLUME_FORCE" in extensions else (0.0, 0.0, 0.0)
    lbm = fx.LBM(*size, nu, *force, velocity_set=q, collision=collision, extensions=extensions)
    lbm.rho.host[:], lbm.u.host[:], lbm.flags.host[:] = rho, u, flags
    if lbm.F is not None:
        lbm.F.host[:] = np.random.default_rng(2).uniform(-1e-4, 1e-4, 3 * lbm.N)
    if lbm.porosity is not None:
        lbm.porosity.host[:] = np.random.default_rng(3).uniform(0.0, 0.5, lbm.N)
    lbm.initialize()
    return lbm


def single_steps(lbm, steps):
    from fluidx3d_amd._abi import check
    for _ in range(steps):
        check(lbm.ctx.lib.fx_lbm_stream_collide(*lbm._step_args(), lbm.t, lbm.fx, lbm.fy, lbm.fz, lbm._ptr(lbm.F), lbm._ptr(lbm.porosity)))
        lbm.t += 1
    lbm.ctx.sync()


@pytest.mark.gpu
@pytest.mark.parametrize("size,q,collision,extensions", CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) and v and isinstance(v[0], int) else str(v))
def test_run_equals_single_steps(size, q, collision, extensions):
    import fluidx3d_amd as fx
    a, b = (scene_lbm(fx, size, q, collision, extensions) for _ in range(2))
    takes = (size, q, collision, extensions) not in SINGLE_STEPS
    try:
        for steps in (4, 1, 7, 10):  # from even and odd t; 0, 1, 3 and 2 single steps after the pairs
            before = a.ctx.launches()
            a.run(steps)
            after = a.ctx.launches()
            two = steps // 4 * 2 if takes else 0
            assert (after.two_steps - before.two_steps, after.one_step - before.one_step) == (two, steps - 2 * two)
            single_steps(b, steps)
            x, y = a.read_ddfs(), b.read_ddfs()
            same = x.view(np.uint32) == y.view(np.uint32)
            assert same.all(), (a.t, int((~same).sum()))
    finally:
        a.close()
        b.close()


@pytest.mark.gpu
def test_run_equals_oracle(oracle):
    import fluidx3d_amd as fx
    size = (128, 64, 55)
    lbm = scene_lbm(fx, size, 19, "TRT", ())
    rho, u, flags = scenes.random_scene(*size, seed=5)
    ref = oracle.OracleLBM(*size, w=lbm.w, trt=True)
    try:
        ref.rho[:], ref.u[:], ref.flags[:] = rho, u, flags
        ref.initialize()
        lbm.run(9)
        ref.step(9)
        assert lbm.ctx.launches().two_steps == 4
        assert np.array_equal(lbm.read_ddfs(), ref.fi)
    finally:
        lbm.close()


@pytest.mark.gpu
@pytest.mark.parametrize("interval,window", [(9, 25), (10, 25), (10, 20), (10, 21), (10, 2), (4, 30), (31, 30), (5, 0)])
def test_adjoint_equals_single_steps(interval, window):
    """Adjoint.forward: the objective, the DDFs and the gradient with the spans between
    checkpoints taken two steps at a time, from one checkpoint to the next (an even interval),
    back into the lattice's own array (an odd one, the window), and spans of one step."""
    import fluidx3d_amd as fx
    from fluidx3d_amd.adjoint import Adjoint
    rho, u, flags, alpha = scenes.porous_channel(128, 64, 58)
    states = []
    for k in (interval, 1):  # an interval of 1 leaves single steps only
        lbm = fx.LBM(128, 64, 58, 1.0 / 6.0, 1e-5, 0.0, 0.0, extensions=POROUS)
        lbm.rho.host[:], lbm.u.host[:], lbm.flags.host[:], lbm.porosity.host[:] = rho, u, flags, alpha
        adj = Adjoint(lbm, steps=31, window_begin=window, plane_x=127, checkpoint_interval=k)
        states.append((adj.forward(), lbm.read_ddfs(), adj.backward(), adj.backward()))
        spans = [min(k - t % k, window - t) for t in range(0, window, k)]
        assert lbm.ctx.launches().two_steps == sum(n // 2 for n in spans)
        adj.close()
        lbm.close()
    (J, f, g, again), (J1, f1, g1, _) = states
    assert J == J1 and np.array_equal(f, f1) and np.array_equal(g, g1) and np.array_equal(g, again)
