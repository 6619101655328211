"""Served batches above and below the size of the workgroup map (csrc/fdtd2d.h: BATCH_MAP): 64
shots of 330 x 330 cells in workgroups of 2 x 64 threads with two columns each need more
workgroups than the map holds while all are resident, and fewer before and after.  Records equal
the plain path's bit for bit; the chunks are long enough in number that some are replayed."""
import numpy as np
import pytest

import geophyinv as G
from geophyinv.serve import Server
from helpers import layered_acoustic, wavelet

pytestmark = pytest.mark.gpu
SHOTS, SIDE, NT, CHUNK = 64, 330, 240, 8


def test_batches_on_both_sides_of_the_map(gpu_ctx):
    med = layered_acoustic(nz=SIDE, nx=SIDE, seed=4)
    gz, gx = med.grid
    tg = G.Grid(0.0, 0.4 * gz.step / (1.6 * float(med.vp.m.max())), NT)
    shots = []
    for k in range(SHOTS):
        z = 0.3 * gz.last + 0.37 * k * gz.step
        ag = G.AGeomss({"z": [z], "x": [0.5 * gx.last]}, {"z": [z + 5.3 * gz.step], "x": [0.5 * gx.last]})
        s = G.Srcs(1, tg, ["p"])
        s.update(["p"], wavelet(NT, tg.step, 25.0, 0.02) * 1e3)
        shots.append(G.SeisForwExpt(G.FdtdAcoustic(), medium=med, tgrid=tg, ageom=[ag], srcwav=[s], rfields=["p", "vz"],
                                    order=2, npml=20, context=gpu_ctx))
    need = ((SIDE + 40) // 64 + 1) * ((SIDE + 40) // 4) * SHOTS
    assert need > 1 << 15
    print(f"batch map: {need} workgroups", flush=True)
    with Server(0, 2, max_shots=SHOTS, chunk_steps=CHUNK, autotune=False, tile=2) as srv:
        tickets = [srv.submit(pa, 0) for pa in shots]
        served = [srv.wait(t, timeout=60.0) for t in tickets]
    for pa, got in list(zip(shots, served))[::9]:
        want, _ = pa.run_shot(0)
        for f in want:
            assert np.abs(want[f]).max() > 0, f
            assert np.array_equal(got[f], want[f]), f
        pa.free()
