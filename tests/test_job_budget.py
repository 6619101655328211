"""Job queue: the memory that jobs use only where there is some (several steps per launch, rings of
adjoint arrays; csrc/gpi_jobs.hip: spare) keeps no two jobs from running together that fit the
budget without it, and is never taken beyond the budget.  In the CPU build, whose device memory
can be counted."""
import pytest

from test_kept_buffers import run

SCRIPT = r"""
import time
from geophyinv.serve import JobServer
from helpers import fwi_experiment
ctx = _lib.Context(0)
if sys.argv[1] == "forward":
    pa, dobs = shot(ctx, 500, n=40, nr=5), None
    want = {"records": pa.run_shot(0)[0]}
else:
    pa = fwi_experiment(layered_acoustic(nz=30, nx=34), nss=1, nt=130, ctx=ctx, checkpoint=20, grad_rho=True)
    recs = pa.run_shot(0)[0]
    dobs = G.Recs(next(iter(recs.values())).shape[1], pa.tgrid, list(recs))
    for f in recs:
        dobs.d[f][:, :] = 0.5 * recs[f]
pa._free_store(0)

def serve(budget, workers, jobs):
    before, most, together = free_bytes(), 0, 0
    with JobServer(workers=workers, hbm_budget_bytes=budget) as js:
        ts = [js.submit(pa, 0, **({"dobs": dobs} if dobs else {})) for _ in range(jobs)]
        while js.stats()["completed"] + js.stats()["failed"] < jobs:
            together = max(together, js.stats()["running"])
            most = max(most, before - free_bytes())
            time.sleep(0.002)
        out = [js.wait(t) for t in ts]
    return out, together, most

def fits(budget):
    with JobServer(workers=1, hbm_budget_bytes=budget) as js:
        try:
            js.wait(js.submit(pa, 0, **({"dobs": dobs} if dobs else {})))
        except _lib.GpiError as e:
            assert e.code == -2, e
            return False
    return True

lo, hi = 10_000, 16_000_000   # what the queue takes a job to need
while hi - lo > hi // 20:
    mid = (lo + hi) // 2
    if fits(mid): hi = mid
    else: lo = mid
need = hi

def flat(o):
    return [a for k in sorted(o) for a in ([o[k][f] for f in sorted(o[k])] if isinstance(o[k], dict) else [o[k]])]

one, _, _ = serve(0, 1, 1)
for factor, workers in ((1.0, 2), (1.0, 3), (1.6, 2), (8.0, 2)):
    budget = int(2 * need * factor)
    out, together, most = serve(budget, workers, 3)
    print(sys.argv[1], need, factor, together, most, flush=True)
    assert together == 2, (factor, together)
    assert most <= budget + 256 * 400, (factor, most, budget)   # the CPU build rounds to 256 bytes
    for o in out:
        for a, b in zip(flat(o), flat(one[0])):
            assert np.array_equal(a, b), factor
print("two at a time")
"""


@pytest.mark.parametrize("kind", ["forward", "gradient"])
def test_jobs_that_fit_run_together(kind):
    run(SCRIPT, "two at a time", [kind], env=dict(EMU_THREADS="1"))
