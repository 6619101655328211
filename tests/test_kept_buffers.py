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


OTHERS = r"""
from geophyinv.serve import JobServer
def stores(ctx, p):
    n = 0
    try:
        while True:
            p.run_shot(0, save=True)
            p._stores.pop(0)
            n += 1
    except _lib.GpiError as e:
        assert e.code == -2, e
    return n
a = _lib.Context(0)
pa = shot(a, 90)
if sys.argv[1] == "kept":
    want = pa.run_shot(0)[0]["p"].copy()
else:
    pa._ensure_model()
js = JobServer(workers=1)
queue = js.stats()["hbm_budget"]
js.close()
b = _lib.Context(0)
n = stores(b, shot(b, 40))
b.close()
if sys.argv[1] == "kept":   # its buffers are gone, its results are not
    assert np.array_equal(pa.run_shot(0)[0]["p"], want)
print("stores", n, queue)
"""


def test_other_contexts_get_kept_buffers_back():
    """What one idle context keeps is memory that another context and a job queue can have: as much
    fits as if nothing were kept."""
    env = dict(EMU_HBM_GB="0.02")
    (n0, q0), (n1, q1) = (map(int, run(OTHERS, "stores", [k], env).split()[-2:]) for k in ("fresh", "kept"))
    assert n0 >= 20 and n1 == n0, (n0, n1)
    assert abs(q1 - q0) <= 256 * 50, (q0, q1)   # of some 30 buffers, which the CPU build rounds to 256 bytes


THREADS = r"""
import threading
want, errors = {}, []
def work(k, first):
    ctx = _lib.Context(0)
    try:
        for nt in (60, 75, 60, 90, 75):
            pa = shot(ctx, nt + k)
            for _ in range(3):
                got = pa.run_shot(0, save=True)[0]["p"].copy()
                if first:
                    want[nt + k] = got
                elif not np.array_equal(got, want[nt + k]):
                    errors.append((k, nt))
            pa.free()
    except Exception as e:
        errors.append(e)
    finally:
        ctx.close()
for k in range(3):
    work(k, True)
ts = [threading.Thread(target=work, args=(k, False)) for k in range(3)]
[t.start() for t in ts]
ctx, refused = _lib.Context(0, 1 << 40), 0
big = shot(ctx, 20000)   # more than the device has: every attempt takes what the others keep
while any(t.is_alive() for t in ts):
    try:
        big.run_shot(0, save=True)
    except _lib.GpiError as e:
        assert e.code == -2, e
        refused += 1
[t.join() for t in ts]
assert not errors and refused, (errors, refused)
print("threads agree")
"""


def test_contexts_on_threads_share_what_memory_there_is():
    run(THREADS, "threads agree", env=dict(EMU_HBM_GB="0.02", EMU_THREADS="2"))


REVERSED = r"""
import test_time_reversal_steps as T
held = []
for sampling in (2, 0):   # sampled: one pass per step, no rings
    ctx = _lib.Context(0)
    ctx.set_pass_sampling(sampling)
    keep, G.SeisForwExpt.free = G.SeisForwExpt.free, lambda self: None   # the model's end would free them
    before = free_bytes()
    T.gradient(dict(T.CASES[sys.argv[1]], nt=10), ctx)
    held.append(before - free_bytes())
    G.SeisForwExpt.free = keep
print("held", *held)
"""


def test_time_reversal_takes_rings_only_for_several_steps():
    """Order 8 runs pass by pass: its gradient takes (and keeps) the same buffers with and without
    pass sampling.  Order 2 takes rings."""
    for case, same in (("order8", True), ("odd", False)):
        a, b = map(int, run(REVERSED, "held", [case]).split()[-2:])
        assert (a == b) if same else (b > a), (case, a, b)
