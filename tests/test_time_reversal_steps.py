"""The time-reversed 2-D acoustic gradient with several steps per launch: boundary saving out of a
ring, the stored planes forced inside a launch, both wavefields imaged over up to eight steps at
once (csrc/gpi_shot.hip: gpi_adjoint; csrc/fdtd2d_steps.hip: FORCE; csrc/strips.hip).

No operation and no order changes against one pass per step, which the oracle's tests pin, so
records, misfit and gradients have to be the same bits: sizes that are no multiple of a tile,
step counts that end in a part of a launch and of a batch, planes in corner tiles, in one tile
with both ends and next to the split of the grid in a frame and an inner rectangle, rigid and
absorbing faces, and the orders that never take several steps."""
import os
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EMU = os.path.join(ROOT, "tests", "cpu_emu")

CASES = {
    "small": dict(n=(23, 18), npml=5, nt=21, order=2),
    "odd": dict(n=(45, 61), npml=6, nt=35, order=2),
    "two-steps": dict(n=(45, 38), npml=6, nt=2, order=2),
    "rigid": dict(n=(40, 33), npml=6, nt=19, order=2, pml=["zmax", "xmin"], rigid=["zmin", "xmax"]),
    "order4": dict(n=(39, 52), npml=7, nt=20, order=4),
    "order6": dict(n=(42, 40), npml=9, nt=13, order=6),
    "order8": dict(n=(38, 45), npml=9, nt=10, order=8),
    "frame": dict(n=(352, 331), npml=9, nt=18, order=2),
    "frame-narrow-strips": dict(n=(512, 391), npml=4, nt=17, order=2),
    "frame-order4": dict(n=(611, 497), npml=20, nt=14, order=4),
}


def gradient(case, ctx):
    import geophyinv as G

    n, nt, ds = case["n"], case["nt"], 10.0
    rng = np.random.Generator(np.random.PCG64(3))
    grid = [G.Grid.range(0.0, ds * (m - 1), length=m) for m in n]
    vp = np.asfortranarray(rng.uniform(1800.0, 2600.0, n), dtype=np.float32)
    rho = np.asfortranarray(rng.uniform(1900.0, 2300.0, n), dtype=np.float32)
    tgrid = G.Grid(0.0, 0.25 * ds / 3000.0, nt)
    mid = [0.5 * ds * (m - 1) for m in n]
    x = np.linspace(mid[1] - 5.2 * ds, mid[1] + 5.2 * ds, 5)
    ag = [G.AGeomss({"z": [mid[0]], "x": [mid[1]]}, {"z": np.full(5, mid[0] - 2.3 * ds), "x": x})]
    src = G.Srcs(1, tgrid, ["vz"])
    src.update(["vz"], 1e6 * rng.normal(size=nt))
    kw = {k + "_faces": case[k] for k in ("pml", "rigid") if k in case}
    pa = G.SeisForwExpt(G.FdtdAcoustic("forward_save", 2), medium=G.AcousticMedium(grid, vp, rho), tgrid=tgrid,
                        ageom=ag, srcwav=[src], rfields=["vz"], order=case["order"], npml=case["npml"], compat=0,
                        context=ctx, **kw)
    dobs = [G.Recs(5, tgrid, ["vz"])]
    dobs[0].d["vz"][:, :] = rng.normal(size=(nt, 5)).astype(np.float32)
    m = pa.model_vector()
    g = np.zeros(m.size)
    try:
        J = G.gradient(g, m, G.L2DistLoss(), dobs, pa)
        return [np.array(J), g.copy(), *[v.copy() for v in pa.gradients.values()]]
    finally:
        pa.free()


def check(name, ctx):
    got = gradient(CASES[name], ctx)
    ctx.set_pass_sampling(2)   # one pass per step
    try:
        want = gradient(CASES[name], ctx)
    finally:
        ctx.set_pass_sampling(0)
    for a, b in zip(got, want):
        assert np.abs(b).max() > 0
        assert np.array_equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(CASES))
def test_steps_give_the_gradient_of_the_passes(gpu_ctx, name):
    print(f"time reversal: {name}", flush=True)
    check(name, gpu_ctx)


SCRIPT = r"""
import sys
sys.path[:0] = [{pkg!r}, {tests!r}]
from geophyinv import _lib
_lib.load({lib!r})
import test_time_reversal_steps as T
T.check({name!r}, _lib.Context(0))
print("all equal")
"""


@pytest.mark.parametrize("name", list(CASES))
def test_steps_give_the_gradient_of_the_passes_in_the_cpu_build(name):
    jobs = str(min(8, os.cpu_count() or 1))
    subprocess.run(["make", "-s", "-j", jobs, "-C", EMU, "all"], check=True)
    code = SCRIPT.format(pkg=os.path.join(ROOT, "geophyinv.jl_amd"), tests=os.path.join(ROOT, "tests"),
                         lib=os.path.join(EMU, "_build", "libgpi_emu.so"), name=name)
    env = dict(os.environ, GLIBC_TUNABLES="glibc.rtld.optional_static_tls=8000000")
    r = subprocess.run([sys.executable, "-W", "ignore", "-c", code], capture_output=True, text=True, timeout=900,
                       cwd=ROOT, env=env)
    assert r.returncode == 0 and "all equal" in r.stdout, (r.returncode, r.stdout[-500:], r.stderr[-3000:])
