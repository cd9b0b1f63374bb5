"""The second DDF array when device memory is short.  hipMalloc and hipMemGetInfo are replaced
on the host, in a process of its own: a small library, loaded before the HIP library with its
symbols global, fails a chosen number of allocations of one size and reports a chosen amount of
free memory.  Every allocation that it lets through is the runtime's.  It also counts the host
allocations (operator new) of libfx_lbm.so: a run makes none, so it cannot throw through the C
interface."""
import json
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

INTERPOSER = r'''
#include <dlfcn.h>
#include <stddef.h>
#include <stdlib.h>
#include <string.h>
#include <new>
extern "C" {
static void* hip(const char* name) {
	static void* lib = 0;
	if(!lib) lib = dlopen("libamdhip64.so", RTLD_NOW | RTLD_LOCAL);
	return dlsym(lib, name);
}
size_t fail_size = 0, fake_free = 0, fake_total = 0;
int fail_count = 0, mallocs = 0, failed = 0;
int hipMalloc(void** p, size_t n) {
	mallocs++;
	if(fail_count > 0 && n == fail_size) { fail_count--; failed++; *p = 0; return 2; } /* hipErrorOutOfMemory */
	return ((int (*)(void**, size_t))hip("hipMalloc"))(p, n);
}
int hipMemGetInfo(size_t* f, size_t* t) {
	if(fake_total) { *f = fake_free; *t = fake_total; return 0; }
	return ((int (*)(size_t*, size_t*))hip("hipMemGetInfo"))(f, t);
}
int counting = 0, news = 0;
}
void* operator new(size_t n) {
	if(counting) {
		Dl_info i;
		if(dladdr(__builtin_return_address(0), &i) && i.dli_fname && strstr(i.dli_fname, "libfx_lbm")) news++;
	}
	void* p = malloc(n ? n : 1);
	if(!p) throw std::bad_alloc();
	return p;
}
'''

PROGRAM = r'''
import ctypes, json, sys
I = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
var = lambda name, t=ctypes.c_int: t.in_dll(I, name)
size_t = ctypes.c_size_t
import numpy as np
import fluidx3d_amd as fx
from fluidx3d_amd import _abi
from tests.test_two_steps import scene_lbm, single_steps
out = {}
SIZE = (128, 96, 96)
a, b = (scene_lbm(fx, SIZE, 19, "SRT", ()) for _ in range(2))
array = 19 * a.N * 4
def run(steps):
    n = a.ctx.launches().two_steps
    var("counting").value = 1
    a.run(steps)
    var("counting").value = 0
    single_steps(b, steps)
    same = bool(np.array_equal(a.read_ddfs().view(np.uint32), b.read_ddfs().view(np.uint32)))
    return [a.ctx.launches().two_steps - n, a.ctx.second_array_bytes()[0] // array, same]
def memory(free, total):
    var("fake_free", size_t).value, var("fake_total", size_t).value = free, total
GB = 10 ** 9
memory(15 * array, 288 * GB)       # little is free
out["scarce"] = run(8)
memory(140 * GB, 288 * GB)         # less than half, and the array is small
out["small"] = run(8)
a.set_second_array(False); a.set_second_array(True)
memory(0, 0)
var("fail_size", size_t).value, var("fail_count").value = array, 1
out["malloc fails"] = run(8) + [var("failed").value]
out["next run"] = run(8)           # the failure left nothing behind
# another context's allocation fails once while a holds its array: given back, then tried again
n = var("failed").value
var("fail_size", size_t).value, var("fail_count").value = 12345 * 16, 1
p = b.ctx.alloc(12345 * 16)
out["given back"] = [a.ctx.second_array_bytes()[0], var("failed").value - n, bool(p)]
out["after"] = run(9)
# nothing to give back: the caller's allocation fails, and the next launches do not report it
a.set_second_array(False)
var("fail_count").value = 2
try:
    b.ctx.alloc(12345 * 16)
    out["refused"] = False
except _abi.FxError as e:
    out["refused"] = e.code == _abi.FX_ERR_MEMORY
var("fail_count").value = 0
out["then"] = run(5)
out["host allocations of the runs"] = var("news").value
a.set_second_array(True)
var("counting").value = 1
c = scene_lbm(fx, SIZE, 19, "SRT", ())
var("counting").value = 0
out["counted"] = var("news").value > 0  # a context is allocated
a.close(); b.close(); c.close()
print(json.dumps(out))
'''


@pytest.fixture(scope="module")
def outcome(tmp_path_factory):
    d = tmp_path_factory.mktemp("interposer")
    (d / "i.cpp").write_text(INTERPOSER)
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", str(d / "i.cpp"), "-o", str(d / "i.so"), "-ldl"], check=True)
    r = subprocess.run([sys.executable, "-c", PROGRAM, str(d / "i.so")], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-3000:]
    return json.loads(r.stdout.strip().splitlines()[-1])


# [launches of two steps, second arrays held, DDFs equal those of single steps, ...]
@pytest.mark.parametrize("what,expected", [
    ("scarce", [0, 0, True]), ("small", [4, 1, True]), ("malloc fails", [0, 0, True, 1]), ("next run", [4, 1, True]),
    ("given back", [0, 1, True]), ("after", [4, 1, True]), ("refused", True), ("then", [0, 0, True]),
    ("host allocations of the runs", 0), ("counted", True)])
def test_short_memory(outcome, what, expected):
    assert outcome[what] == expected, outcome
