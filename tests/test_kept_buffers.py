"""Buffers that a context keeps from finished calls for the next ones (csrc/gpi_util.hip: dev_alloc,
free_allocs): in the CPU build, whose device memory can be counted."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EMU = os.path.join(ROOT, "tests", "cpu_emu")

# One model and the calls of its shots, straight through the C interface.
PRELUDE = r"""
import ctypes as C, sys
import numpy as np
sys.path[:0] = [{pkg!r}, {tests!r}]
from geophyinv import _lib
lib = _lib.load({lib!r})
import geophyinv as G
from helpers import experiment, layered_acoustic

def free_bytes():
    fr, tot = C.c_size_t(), C.c_size_t()
    getattr(lib, "_Z13hipMemGetInfoPmS_")(C.byref(fr), C.byref(tot))
    return fr.value

def shot(ctx, nt, n=60, nr=9):
    return experiment(layered_acoustic(nz=n, nx=n), nt=nt, npml=6, nr=nr, rfields=("p",), ctx=ctx)
"""


def run(script, marker, args=(), env=()):
    jobs = str(min(8, os.cpu_count() or 1))
    subprocess.run(["make", "-s", "-j", jobs, "-C", EMU, "all"], check=True)
    code = PRELUDE.format(pkg=os.path.join(ROOT, "geophyinv.jl_amd"), tests=os.path.join(ROOT, "tests"),
                          lib=os.path.join(EMU, "_build", "libgpi_emu.so")) + script
    env = dict(os.environ, GLIBC_TUNABLES="glibc.rtld.optional_static_tls=8000000", **dict(env))
    r = subprocess.run([sys.executable, "-W", "ignore", "-c", code, *args], capture_output=True, text=True, timeout=600,
                       cwd=ROOT, env=env)
    assert r.returncode == 0 and marker in r.stdout, (r.returncode, r.stdout[-500:], r.stderr[-3000:])
    return r.stdout


BUDGET = r"""
before = free_bytes()
budget = int(sys.argv[1])
ctx = _lib.Context(0, budget)
pa, pb = shot(ctx, 200), shot(ctx, 185)
def save(p):
    p.run_shot(0, save=True)
    return p._stores.pop(0)
def saves(p):
    n = 0
    try:
        while True:
            save(p)
            n += 1
            held = before - free_bytes()
            assert held <= budget + 256 * 100, (n, held, budget)   # the CPU build rounds to 256 bytes
    except _lib.GpiError as e:
        assert e.code == -2, e
    return n
pa._ensure_model()
stores = [save(pa) for _ in range(8)] if sys.argv[2] == "kept" else []
for s in stores:
    ctx.check(lib.gpi_store_free(ctx.h, s))
# stores of a little less than the kept buffers, until the budget is spent
print("stores", saves(pb))
"""


def test_a_budget_holds_whatever_was_kept():
    """Never more device memory than the budget, and never fewer stores than on a fresh context."""
    for budget in ("12000000", "11800000"):
        fresh, kept = (run(BUDGET, "stores", [budget, k]).split()[-1] for k in ("fresh", "kept"))
        assert int(fresh) >= 12 and kept == fresh, (budget, fresh, kept)
