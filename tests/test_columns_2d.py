"""The acoustic passes that give a thread two columns (csrc/fdtd2d.hip: vel_ac_columns,
str_ac_columns) against the oracle: records and final wavefields equal bit for bit.

Odd widths leave a thread with one column at the right edge, rigid faces mirror their first and
last velocities, sources sit on both columns of a pair.  On the GPU the grids are just above
the size from which the passes take this shape; the CPU build runs small ones with the shape
asked for (GPI_TILE2D), where every access is checked."""
import os
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EMU = os.path.join(ROOT, "tests", "cpu_emu")

SMALL = [  # order, nz, nx, npml, nt, options
    (8, 40, 45, 9, 12, {}),
    (8, 67, 44, 9, 12, dict(pml_faces=["xmax", "zmin"])),
    (6, 51, 38, 7, 12, dict(sfields=("p", "vx", "vz"), ns=3)),
    (4, 33, 70, 0, 12, dict(pml_faces=[])),
]
LARGE = [(8, 1220, 1209, 10, 9, {}), (6, 1230, 1200, 7, 9, dict(sfields=("p", "vx", "vz"), ns=3))]


def check(case, ctx):
    import oracle as O
    from helpers import experiment, layered_acoustic

    order, nz, nx, npml, nt, opt = case
    kw = dict(ns=2, nr=11, sfields=("p",), rfields=("p", "vx", "vz"))
    kw.update(opt)
    pa = experiment(layered_acoustic(nz=nz, nx=nx), nt=nt, order=order, npml=npml, ctx=ctx, **kw)
    pa.run_shot(0)
    pa._ctx.set_pass_sampling(1)   # order 4 too: the passes, not several steps per launch
    try:
        recs, fin = pa.run_shot(0, final_fields=["p", "vx", "vz"])
    finally:
        pa._ctx.set_pass_sampling(0)
    orc = O.from_experiment(pa)
    orc.run()
    for q, f in enumerate(pa.rfields):
        assert np.array_equal(recs[f], orc.records(q)), f
    for f in ("p", "vx", "vz"):
        assert np.abs(orc.field(f)).max() > 0, f
        assert np.array_equal(fin[f], orc.field(f)), f
    pa.free()


@pytest.mark.gpu
@pytest.mark.parametrize("case", LARGE, ids=str)
def test_two_columns_equal_the_oracle(gpu_ctx, case):
    print(f"two columns per thread: {case}", flush=True)
    check(case, gpu_ctx)


SCRIPT = r"""
import sys
sys.path[:0] = [{pkg!r}, {orc!r}, {tests!r}]
from geophyinv import _lib
_lib.load({lib!r})
import test_columns_2d as T
ctx = _lib.Context(0)
for case in T.SMALL:
    T.check(case, ctx)
print("all equal")
"""


@pytest.mark.parametrize("shape", ["2", "3"])
def test_two_columns_equal_the_oracle_in_the_cpu_build(shape):
    jobs = str(min(8, os.cpu_count() or 1))
    subprocess.run(["make", "-s", "-j", jobs, "-C", EMU, "all"], check=True)
    code = SCRIPT.format(pkg=os.path.join(ROOT, "geophyinv.jl_amd"), orc=os.path.join(ROOT, "oracle"),
                         tests=os.path.join(ROOT, "tests"), lib=os.path.join(EMU, "_build", "libgpi_emu.so"))
    env = dict(os.environ, GLIBC_TUNABLES="glibc.rtld.optional_static_tls=8000000", GPI_TILE2D=shape)
    r = subprocess.run([sys.executable, "-W", "ignore", "-c", code], capture_output=True, text=True, timeout=900,
                       cwd=ROOT, env=env)
    assert r.returncode == 0 and "all equal" in r.stdout, (r.returncode, r.stdout[-500:], r.stderr[-3000:])
