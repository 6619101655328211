"""Gradients in little memory: what a gradient takes on top (rings of adjoint arrays, the second
states of several-step launches) comes after everything it cannot run without, so a larger budget
never turns a gradient that ran into one that is refused, and every budget gives the same bits.

LEAST is what a gradient needs that advances and images one step at a time with copies of the
arrays it compares (10 steps, a checkpoint every 4): the context's memory for the model, the store
and the adjoint run, to 512 bytes."""
import os
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EMU = os.path.join(ROOT, "tests", "cpu_emu")

LEAST = {
    "acoustic-2d": 707955, "acoustic-2d-invK": 459223, "acoustic-2d-order8": 913367, "elastic-2d": 1160639,
    "elastic-2d-order4": 1264318, "acoustic-3d": 4794754, "elastic-3d": 10329650, "elastic-3d-order4": 15732147,
    "reversed-odd": 630075, "reversed-order4": 586267, "reversed-order8": 594055,
}


def run(name, ctx):
    import test_gradient_rings as R
    import test_time_reversal_steps as T

    if name.startswith("reversed-"):
        out = T.gradient(dict(T.CASES[name[len("reversed-"):]], nt=10), ctx)
    else:
        J, g = R.gradients(dict(R.CASES[name], nt=10), ctx, 4)
        out = [np.array(J), *g.values()]
    return out, ctx.timing()["launches"]


def check(name):
    from geophyinv import _lib

    ctx = _lib.Context(0)
    want, most = run(name, ctx)
    ctx.close()
    launches = []
    for k in range(22):
        budget = int(LEAST[name] * 1.1 ** k)
        print(name, budget, flush=True)
        ctx = _lib.Context(0, budget)
        try:
            got, n = run(name, ctx)   # GpiError: refused
        finally:
            ctx.close()
        launches.append(n)
        for a, b in zip(got, want):
            assert np.array_equal(a, b), (name, budget)
    # the smallest budget images every step by itself, the largest several together
    assert launches[-1] == most, (name, launches, most)
    assert launches[0] > most or name == "reversed-order8", (name, launches, most)


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(LEAST))
def test_more_memory_never_refuses_a_gradient(gpu_ctx, name):
    check(name)


SCRIPT = r"""
import sys
sys.path[:0] = [{pkg!r}, {tests!r}]
from geophyinv import _lib
_lib.load({lib!r})
import test_gradient_budgets as T
T.check({name!r})
print("all accepted")
"""


@pytest.mark.parametrize("name", list(LEAST))
def test_more_memory_never_refuses_a_gradient_in_the_cpu_build(name):
    jobs = str(min(8, os.cpu_count() or 1))
    subprocess.run(["make", "-s", "-j", jobs, "-C", EMU, "all"], check=True)
    code = SCRIPT.format(pkg=os.path.join(ROOT, "geophyinv.jl_amd"), tests=os.path.join(ROOT, "tests"),
                         lib=os.path.join(EMU, "_build", "libgpi_emu.so"), name=name)
    # one thread: every context's stream keeps its fibers' stacks
    env = dict(os.environ, GLIBC_TUNABLES="glibc.rtld.optional_static_tls=8000000", EMU_THREADS="0")
    r = subprocess.run([sys.executable, "-W", "ignore", "-c", code], capture_output=True, text=True, timeout=900,
                       cwd=ROOT, env=env)
    assert r.returncode == 0 and "all accepted" in r.stdout, (r.returncode, r.stdout[-500:], r.stderr[-3000:])
