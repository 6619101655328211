"""Grids whose inner rectangle (csrc/fdtd2d_steps.hip) is narrow and close to the grid's edge: thin
or no absorbing strips, a few tiles across.  Cores are dealt evenly, so the last tile's core can be
much smaller than a full one, and its tile must still end inside the arrays.

Heights keep the grid out of one launch; widths and strips are those where a tile that starts at
core - halo would end outside.  Against the oracle bit for bit; with rings (boundary saving,
checkpointed gradients) against one pass per step.  The CPU build checks every access; its run comes
before any on the GPU."""
import os
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EMU = os.path.join(ROOT, "tests", "cpu_emu")

# physics, order, nz, nx, npml, nt
FORWARD = [
    (0, 2, 2000, 54, 0, 9), (0, 2, 2492, 85, 4, 9), (0, 2, 4000, 85, 10, 9), (1, 2, 4000, 86, 4, 9),
    (1, 2, 2100, 67, 0, 9), (0, 4, 2000, 122, 2, 4), (1, 4, 2000, 118, 0, 4),
    # the same across z, and a width where the tile ends with the grid
    (0, 2, 54, 2000, 0, 9), (0, 4, 122, 2000, 2, 4), (0, 2, 2000, 101, 0, 9), (0, 2, 4000, 58, 40, 9),
]
REVERSED = [dict(n=(2492, 85), npml=4, nt=13, order=2), dict(n=(85, 2492), npml=4, nt=13, order=2),
            dict(n=(2000, 122), npml=2, nt=7, order=4)]
CHECKPOINT = [dict(physics=0, n=(2492, 85), npml=4, nt=11, order=2, rho=True),
              dict(physics=1, n=(2100, 71), npml=2, nt=11, order=2, rho=True),
              dict(physics=1, n=(2000, 122), npml=2, nt=7, order=4, rho=True)]


def forward(case, ctx):
    import oracle as O
    from helpers import experiment, layered_acoustic, layered_elastic

    physics, order, nz, nx, npml, nt = case
    med = (layered_acoustic if physics == 0 else layered_elastic)(nz=nz, nx=nx)
    kw = dict(pml_faces=[]) if npml == 0 else {}
    pa = experiment(med, nt=nt, order=order, npml=npml, ctx=ctx, ns=2, nr=11, rec_depth=2.5 * nz,
                    sfields=("p",) if physics == 0 else ("tauxx",),
                    rfields=("p", "vx", "vz") if physics == 0 else ("vx", "vz"), **kw)
    fields = ["p", "vx", "vz"] if physics == 0 else ["tauxx", "tauzz", "tauxz", "vx", "vz"]
    recs, fin = pa.run_shot(0, final_fields=fields)
    launches = pa.timing["launches"]
    orc = O.from_experiment(pa)
    orc.run()
    for q, f in enumerate(pa.rfields):
        assert np.array_equal(recs[f], orc.records(q)), (case, f)
    for f in fields:
        assert np.abs(orc.field(f)).max() > 0, f
        assert np.array_equal(fin[f], orc.field(f)), (case, f)
    assert launches < 2 * nt, (case, launches)
    pa.free()


def reversed_gradient(case, ctx):
    import test_time_reversal_steps as T

    got = T.gradient(case, ctx)
    ctx.set_pass_sampling(2)   # one pass per step
    try:
        want = T.gradient(case, ctx)
    finally:
        ctx.set_pass_sampling(0)
    for a, b in zip(got, want):
        assert np.abs(b).max() > 0
        assert np.array_equal(a, b), case


def checkpointed_gradient(case, ctx):
    import test_gradient_rings as T

    J, got = T.gradients(case, ctx, 5)
    ctx.set_pass_sampling(2)
    try:
        J0, want = T.gradients(case, ctx, 5)
    finally:
        ctx.set_pass_sampling(0)
    assert J == J0
    for k in want:
        assert np.abs(want[k]).max() > 0
        assert np.array_equal(got[k], want[k]), (case, k)


def check(k, ctx):
    for fn, cases in ((forward, FORWARD), (reversed_gradient, REVERSED), (checkpointed_gradient, CHECKPOINT)):
        for case in cases[k::2]:
            print(fn.__name__, case, flush=True)
            fn(case, ctx)


SCRIPT = r"""
import sys
sys.path[:0] = [{pkg!r}, {orc!r}, {tests!r}]
from geophyinv import _lib
_lib.load({lib!r})
import test_inner_tiles_2d as T
T.check({k}, _lib.Context(0))
print("all equal")
"""


@pytest.mark.parametrize("k", [0, 1])
def test_narrow_inner_rectangles_in_the_cpu_build(k):
    jobs = str(min(8, os.cpu_count() or 1))
    subprocess.run(["make", "-s", "-j", jobs, "-C", EMU, "all"], check=True)
    code = SCRIPT.format(pkg=os.path.join(ROOT, "geophyinv.jl_amd"), orc=os.path.join(ROOT, "oracle"),
                         tests=os.path.join(ROOT, "tests"), lib=os.path.join(EMU, "_build", "libgpi_emu.so"), k=k)
    env = dict(os.environ, GLIBC_TUNABLES="glibc.rtld.optional_static_tls=8000000")
    r = subprocess.run([sys.executable, "-W", "ignore", "-c", code], capture_output=True, text=True, timeout=900,
                       cwd=ROOT, env=env)
    assert r.returncode == 0 and "all equal" in r.stdout, (r.returncode, r.stdout[-500:], r.stderr[-3000:])


@pytest.mark.gpu
@pytest.mark.parametrize("k", [0, 1])
def test_narrow_inner_rectangles(gpu_ctx, k):
    check(k, gpu_ctx)
