"""Checkpointed gradients whose wavefields move through rings of slabs, several adjoint steps
imaged per launch (csrc/gpi_shot.hip: Mover, AdjointRing; csrc/strips.hip).

Neither the checkpoint interval, nor the steps imaged together, nor the several-step launches
change a single operation or its order, so every way of running one gradient gives the same
bits: intervals around the eight steps imaged together (a step, one batch and one more, a
remainder, a single segment), the passes instead of the several-step launches (pass sampling
is on), and every memory budget down to the smallest that the run accepts, which takes away
the ring slot by slot until each step is imaged between its two passes.  The passes with one
slot restate the flow that the finite-difference and oracle tests pin."""
import os
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EMU = os.path.join(ROOT, "tests", "cpu_emu")

CASES = {
    "acoustic-2d": dict(physics=0, n=(34, 41), npml=6, nt=37, order=2, rho=True),
    "acoustic-2d-invK": dict(physics=0, n=(34, 41), npml=6, nt=37, order=2, rho=False),
    "acoustic-2d-order8": dict(physics=0, n=(38, 45), npml=9, nt=19, order=8, rho=True),
    "acoustic-2d-frame": dict(physics=0, n=(352, 331), npml=9, nt=18, order=2, rho=True),
    "elastic-2d": dict(physics=1, n=(34, 41), npml=6, nt=37, order=2, rho=True),
    "elastic-2d-frame": dict(physics=1, n=(352, 331), npml=9, nt=18, order=2, rho=True),
    "elastic-2d-order4": dict(physics=1, n=(35, 42), npml=7, nt=21, order=4, rho=True),
    "acoustic-3d": dict(physics=0, n=(14, 12, 16), npml=4, nt=21, order=2, rho=True),
    "elastic-3d": dict(physics=1, n=(14, 12, 16), npml=4, nt=21, order=2, rho=True),
    "elastic-3d-order4": dict(physics=1, n=(16, 14, 18), npml=5, nt=19, order=4, rho=True),
}


def gradients(case, ctx, every):
    import geophyinv as G

    n, nt = case["n"], case["nt"]
    rng = np.random.Generator(np.random.PCG64(7))
    ds = 10.0
    grid = [G.Grid.range(0.0, ds * (m - 1), length=m) for m in n]
    vp = np.asfortranarray(rng.uniform(1800.0, 2600.0, n), dtype=np.float32)
    rho = np.asfortranarray(rng.uniform(1900.0, 2300.0, n), dtype=np.float32)
    med = (G.AcousticMedium(grid, vp, rho) if case["physics"] == 0
           else G.ElasticMedium(grid, vp, vp / np.float32(1.8), rho))
    dt = 0.25 * ds / 3000.0
    tgrid = G.Grid(0.0, dt, nt)
    mid = [0.5 * ds * (m - 1) for m in n]
    names = ["z", "x"] if len(n) == 2 else ["z", "y", "x"]
    rec = {k: np.full(5, v - 2.3 * ds) for k, v in zip(names, mid)}
    rec["x"] = np.linspace(mid[-1] - 5.2 * ds, mid[-1] + 5.2 * ds, 5)
    ag = [G.AGeomss({k: [v] for k, v in zip(names, mid)}, rec)]
    sf = "p" if case["physics"] == 0 else "tauxx"
    src = G.Srcs(1, tgrid, [sf])
    t = tgrid.values()
    src.update([sf], np.exp(-((t - 5.0 * dt) / (2.0 * dt)) ** 2))
    rf = ["vz"] if case["physics"] == 0 else ["v" + k for k in names]
    att = (G.FdtdAcoustic if case["physics"] == 0 else G.FdtdElastic)("forward_save", 2)
    pa = G.SeisForwExpt(att, medium=med, tgrid=tgrid, ageom=ag, srcwav=[src], rfields=rf, order=case["order"],
                        npml=case["npml"], compat=0, context=ctx, checkpoint=every, grad_rho=case["rho"])
    dobs = [G.Recs(5, tgrid, rf)]
    for f in rf:
        dobs[0].d[f][:, :] = rng.normal(size=(nt, 5)).astype(np.float32)
    m = pa.model_vector()
    g = np.zeros(m.size)
    try:
        J = G.gradient(g, m, G.L2DistLoss(), dobs, pa)
        return J, {k: v.copy() for k, v in pa.gradients.items()}
    finally:
        pa.free()


def check(name, ctx, everys=(1, 8, 16, 0, 5), shrink=0.87):
    from geophyinv import _lib

    case = CASES[name]
    nt = case["nt"]
    J, ref = gradients(case, ctx, 9)
    for k, v in ref.items():
        if case["rho"] or k != "rho":
            assert np.abs(v).max() > 0, k

    def same(got, what):
        assert got[0] == J, what
        for k in ref:
            assert np.array_equal(got[1][k], ref[k]), (k, what)

    for every in everys:
        every = every if every and every != 5 else nt + every
        same(gradients(case, ctx, every), f"every {every}")
    ctx.set_pass_sampling(3)
    try:
        same(gradients(case, ctx, 9), "passes")
    finally:
        ctx.set_pass_sampling(0)
    # budgets: large ones first; the first refusal ends it
    cells = int(np.prod([k + 2 * case["npml"] + 2 * case["order"] + 32 for k in case["n"]]))
    budget, runs = 8 * cells * 140, 0
    while True:
        small = _lib.Context(0, budget)
        try:
            same(gradients(case, small, 9), f"budget {budget}")
            runs += 1
        except _lib.GpiError as e:
            assert e.code == -2, e
            break
        finally:
            small.close()
        budget = int(budget * shrink)
    assert runs > 2, runs


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(CASES))
def test_every_way_gives_the_same_gradient(gpu_ctx, name):
    print(f"gradient rings: {name}", flush=True)
    check(name, gpu_ctx)


SCRIPT = r"""
import sys
sys.path[:0] = [{pkg!r}, {tests!r}]
from geophyinv import _lib
_lib.load({lib!r})
import test_gradient_rings as T
ctx = _lib.Context(0)
T.check({name!r}, ctx, (8, 0), 0.8)
print("all equal")
"""


@pytest.mark.parametrize("name", [k for k in CASES if "frame" not in k])
def test_every_way_gives_the_same_gradient_in_the_cpu_build(name):
    jobs = str(min(8, os.cpu_count() or 1))
    subprocess.run(["make", "-s", "-j", jobs, "-C", EMU, "all"], check=True)
    code = SCRIPT.format(pkg=os.path.join(ROOT, "geophyinv.jl_amd"), tests=os.path.join(ROOT, "tests"),
                         lib=os.path.join(EMU, "_build", "libgpi_emu.so"), name=name)
    env = dict(os.environ, GLIBC_TUNABLES="glibc.rtld.optional_static_tls=8000000")
    r = subprocess.run([sys.executable, "-W", "ignore", "-c", code], capture_output=True, text=True, timeout=900,
                       cwd=ROOT, env=env)
    assert r.returncode == 0 and "all equal" in r.stdout, (r.returncode, r.stdout[-500:], r.stderr[-3000:])
