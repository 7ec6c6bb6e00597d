"""What a context takes of the device's memory, on the CPU: a stand-in for the runtime's memory
calls (malloc under a byte limit), loaded ahead of the library in a process of its own, counts
what cmdg_create asks for.  The third state buffer is an optional one: it is the last thing
asked for, and only where it takes a small share of what is left."""
import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "climatemachine.jl_amd")

RUNTIME = r"""
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <map>
static std::map<void *, size_t> live;
static size_t limit_ = 0, used_ = 0;
extern "C" {
void mem_limit(size_t n) { limit_ = n; }
size_t mem_used() { return used_; }
int hipMalloc(void **p, size_t n) {
    *p = nullptr;
    if (used_ + n > limit_ || !(*p = std::malloc(n ? n : 1))) return 2;  // hipErrorOutOfMemory
    used_ += live[*p] = n;
    return 0;
}
int hipFree(void *p) {
    const auto it = live.find(p);
    if (it == live.end()) return 0;
    used_ -= it->second;
    live.erase(it);
    std::free(p);
    return 0;
}
int hipMemcpy(void *d, const void *s, size_t n, int) { return std::memcpy(d, s, n), 0; }
int hipMemset(void *d, int v, size_t n) { return std::memset(d, v, n), 0; }
int hipMemGetInfo(size_t *f, size_t *t) { return *f = limit_ - used_, *t = limit_, 0; }
int hipGetLastError() { return 0; }
int hipHostFree(void *) { return 0; }
}
"""

SCRIPT = r"""
import ctypes as C, json, sys
rt = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
rt.mem_limit.argtypes, rt.mem_used.restype = [C.c_size_t], C.c_size_t
from cmdg import abi, atmos
from cmdg.grid import uniform_brick
kind, limit = sys.argv[2], int(sys.argv[3])
prm = atmos.ideal_gas_parameters()
grid = uniform_brick((4, 3, 5), (0, 0, 0), (400.0, 300.0, 500.0), N=4, periodicity=(True, True, False),
                     boundary=((0, 0), (0, 0), (1, 2)), lean=kind.endswith("lean"))
cfg = atmos.AtmosConfig(prm) if kind.startswith("euler") else atmos.AtmosConfig(
    prm, orientation=abi.FLAT_ORIENTATION, ref_profile=atmos.DryAdiabaticProfile(300.0, 0.0), gravity_source=True,
    turbulence=abi.SMAGORINSKY_LILLY, C_smag=0.23)
full = uniform_brick((4, 3, 5), (0, 0, 0), (400.0, 300.0, 500.0), N=4, periodicity=(True, True, False),
                     boundary=((0, 0), (0, 0), (1, 2)))
aux = atmos.init_aux(cfg, full)
d, keep = cfg.descriptor(grid, aux, abi.MIXED if "mixed" in kind else abi.FP64)
lib = abi.load_library()
rt.mem_limit(limit)
ctx = C.c_void_p()
if grid.lean:
    b, bk = abi.brick_descriptor(grid)
    rc = lib.cmdg_create_brick(C.byref(d), C.byref(b), None, C.byref(ctx))
else:
    rc = lib.cmdg_create(C.byref(d), None, C.byref(ctx))
used = rt.mem_used()
lib.cmdg_destroy(ctx)
print(json.dumps(dict(rc=rc, used=used, left=rt.mem_used(), state=grid.nelem * 125 * 5 * 8)))
"""


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    d = tmp_path_factory.mktemp("runtime")
    src, lib = d / "runtime.cpp", d / "libruntime.so"
    src.write_text(RUNTIME)
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-o", str(lib), str(src)], check=True)
    return str(lib)


def _create(runtime, kind, limit, **env):
    e = dict(os.environ, PYTHONPATH=PKG, **env)
    r = subprocess.run([sys.executable, "-c", SCRIPT, runtime, kind, str(int(limit))], env=e, capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stderr
    return json.loads(r.stdout.splitlines()[-1])


KINDS = ["euler", "les", "les lean", "les mixed", "les mixed lean", "les general"]


@pytest.mark.parametrize("kind", KINDS)
def test_the_optional_buffer_takes_no_room_that_is_needed(runtime, kind):
    env = {"CMDG_GENERAL_GEOMETRY": "1"} if "general" in kind else {}
    without = _create(runtime, kind, 1 << 30, CMDG_THIRD_STATE_BUFFER="0", **env)
    assert without["rc"] == 0 and without["left"] == 0
    need, state = without["used"], without["state"]
    # exactly what a context needs, and what it needs with one state, or several, beside it
    for spare in (0, state, 10 * state):
        got = _create(runtime, kind, need + spare, **env)
        assert got["rc"] == 0 and got["used"] == need and got["left"] == 0, (spare, got)
    # on an empty card it is taken, and given back
    got = _create(runtime, kind, need + 100 * state, **env)
    assert got["rc"] == 0 and got["used"] == need + state and got["left"] == 0, got


@pytest.mark.parametrize("kind", ["les", "les mixed"])
def test_creation_fails_where_the_needed_memory_is_missing(runtime, kind):
    need = _create(runtime, kind, 1 << 30, CMDG_THIRD_STATE_BUFFER="0")["used"]
    got = _create(runtime, kind, need - 1)
    assert got["rc"] != 0 and got["left"] == 0
