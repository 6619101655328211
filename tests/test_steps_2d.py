"""Several time steps per launch of a 2-D shot (csrc/fdtd2d_steps.hip) against the oracle, which
steps pass by pass: records and final wavefields equal bit for bit.

The sizes sit where the tiling can go wrong: a grid inside one tile, tile remainders of one
cell, the largest grid of one launch per group of steps and the smallest of two (the frame of
strips and faces around an inner rectangle), grids too narrow for that, step counts that leave
a remainder, sources and receivers on tile borders and in the inner rectangle, no absorbing
strips, a free surface, velocity and stress sources on shared cells.  The same cases run on the
GPU and through the CPU build (tests/cpu_emu), where every access is checked."""
import os
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EMU = os.path.join(ROOT, "tests", "cpu_emu")

FS = dict(pml_faces=["zmax", "xmin", "xmax"], stressfree_faces=["zmin"])
CASES = {
    # physics, order, nz, nx, npml, nt, options
    "one-tile": (0, 2, 9, 8, 3, 21, {}),
    "one-tile-elastic": (1, 2, 9, 8, 3, 21, {}),
    "remainder": (0, 2, 37, 42, 6, 33, dict(sfields=("p", "vx", "vz"), ns=3)),
    "remainder-elastic": (1, 2, 38, 41, 6, 33, dict(sfields=("tauxx", "tauzz", "vx", "vz"), ns=3)),
    "free-surface": (1, 2, 60, 47, 7, 30, dict(sfields=("vz", "tauxx"), **FS)),
    "no-strips": (0, 2, 50, 61, 0, 29, dict(pml_faces=[])),
    "no-strips-elastic": (1, 2, 50, 61, 0, 29, dict(pml_faces=[])),
    "one-face": (1, 2, 45, 66, 9, 25, dict(pml_faces=["xmax"])),
    "order4": (0, 4, 52, 57, 9, 22, dict(sfields=("p", "vz"))),
    "order4-elastic": (1, 4, 45, 63, 9, 23, dict(sfields=("tauxx", "vx"))),
    "order6": (0, 6, 52, 57, 9, 21, {}),
    "order6-elastic": (1, 6, 40, 63, 9, 21, {}),
    "order8": (0, 8, 40, 44, 9, 11, {}),
    # 22-cell cores: 16 x 16 tiles are one launch, one more column of tiles makes two launches
    "largest-single": (0, 2, 331, 331, 10, 12, {}),
    "smallest-split": (0, 2, 353, 332, 10, 12, dict(rec_depth=800.0)),
    "smallest-split-elastic": (1, 2, 353, 332, 10, 12, dict(rec_depth=800.0, sfields=("tauxx", "vz"))),
    "split-wide": (0, 2, 610, 555, 20, 17, dict(src_depth=1500.0, rec_depth=1490.0)),
    "split-wide-elastic": (1, 2, 610, 555, 20, 17, dict(src_depth=1500.0, rec_depth=1490.0)),
    "narrow": (0, 2, 40, 1900, 30, 14, dict(nr=700)),
    "split-order4": (0, 4, 355, 380, 9, 11, dict(rec_depth=900.0)),
    "split-order4-elastic": (1, 4, 355, 380, 9, 11, dict(rec_depth=900.0)),
    "wide-strips-order4": (0, 4, 440, 800, 43, 7, dict(nr=200)),
    "narrow-order4": (1, 4, 60, 1500, 20, 9, dict(nr=400)),
}


def check(name, ctx):
    import oracle as O
    from helpers import experiment, layered_acoustic, layered_elastic

    physics, order, nz, nx, npml, nt, opt = CASES[name]
    kw = dict(ns=2, nr=11, sfields=("p",) if physics == 0 else ("tauxx",),
              rfields=("p", "vx", "vz") if physics == 0 else ("vx", "vz"))
    kw.update(opt)
    med = (layered_acoustic if physics == 0 else layered_elastic)(nz=nz, nx=nx)
    pa = experiment(med, nt=nt, order=order, npml=npml, ctx=ctx, **kw)
    fields = ["p", "vx", "vz"] if physics == 0 else ["tauxx", "tauzz", "tauxz", "vx", "vz"]
    recs, fin = pa.run_shot(0, final_fields=fields)
    recs = {f: r.copy() for f, r in recs.items()}
    again, _ = pa.run_shot(0)
    launches = pa.timing["launches"]
    orc = O.from_experiment(pa)
    orc.run()
    for q, f in enumerate(pa.rfields):
        assert np.array_equal(recs[f], orc.records(q)), f
        assert np.array_equal(again[f], recs[f]), f
    for f in fields:
        assert np.abs(orc.field(f)).max() > 0, f
        assert np.array_equal(fin[f], orc.field(f)), f
    # two launches a step and the trailing half step where the passes ran
    assert (launches < 2 * nt) == (order < 8), launches
    pa.free()


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(CASES))
def test_steps_equal_the_oracle(gpu_ctx, name):
    print(f"several steps per launch: {name}", flush=True)
    check(name, gpu_ctx)


SCRIPT = r"""
import sys
sys.path[:0] = [{pkg!r}, {orc!r}, {tests!r}]
from geophyinv import _lib
_lib.load({lib!r})
import test_steps_2d as T
ctx = _lib.Context(0)
for name in T.CASES:
    T.check(name, ctx)
print("all equal")
"""


def test_steps_equal_the_oracle_in_the_cpu_build():
    jobs = str(min(8, os.cpu_count() or 1))
    subprocess.run(["make", "-s", "-j", jobs, "-C", EMU, "all"], check=True)
    code = SCRIPT.format(pkg=os.path.join(ROOT, "geophyinv.jl_amd"), orc=os.path.join(ROOT, "oracle"),
                         tests=os.path.join(ROOT, "tests"), lib=os.path.join(EMU, "_build", "libgpi_emu.so"))
    env = dict(os.environ, GLIBC_TUNABLES="glibc.rtld.optional_static_tls=8000000")
    r = subprocess.run([sys.executable, "-W", "ignore", "-c", code], capture_output=True, text=True, timeout=900,
                       cwd=ROOT, env=env)
    assert r.returncode == 0 and "all equal" in r.stdout, (r.returncode, r.stdout[-500:], r.stderr[-3000:])
