"""The one-launch time loop with several rows of cells per thread: which runs
take it."""
import time

import numpy as np
import pytest

import ifos_amd
from ifos_amd import workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("NX,NY,L,order,DTINV,taken", [
    (1024, 1472, 0, 8, 1, False), (1024, 1472, 0, 8, 6, True), (1024, 800, 2, 8, 1, False), (1024, 800, 2, 4, 4, True),
    (1024, 640, 3, 6, 1, False), (1024, 640, 3, 4, 1, True), (1024, 768, 2, 8, 1, True), (1024, 300, 2, 8, 1, True)])
def test_16bit_snapshots_on_large_tiles(gpu_lib, NX, NY, L, order, DTINV, taken):
    """Forward runs that store 16-bit snapshots take it where it is the faster
    one; runs that store none do not depend on the snapshots' precision."""
    print(f"[resident] {NX}x{NY} L={L} FDORDER {order} DTINV {DTINV}, 16-bit", flush=True)
    w = workloads.small_case(seed=13, NX=NX, NY=NY, L=L, NT=12, FW=10, DTINV=DTINV, VELOCITY=1, FDORDER=order)
    eng = ifos_amd.Engine(w.cfg)
    eng.set_model(**w.start)
    eng.set_shot(w.shots[0].srcpos, w.shots[0].recpos)
    plain = eng.get_resident()[0]
    eng.set_snapshot_precision("bf16")
    assert eng.get_resident()[0] == taken
    eng.forward(snapshots=True)
    assert eng.get_resident()[1] == taken
    obs = np.zeros((2, len(w.shots[0].recpos), 12), np.float32)
    eng.residual(obs[0], obs[1])
    eng.adjoint()
    assert eng.get_resident()[1] == plain
    eng.forward(snapshots=False)
    assert eng.get_resident()[1] == plain


def test_autotuner_reports_the_run_that_follows(gpu_lib):
    """The time per step is that of the one launch where runs take it: the
    per-step kernels take more than twice as long on this grid."""
    print("[resident] autotuner's time", flush=True)
    w = workloads.small_case(seed=14, NX=400, NY=200, L=0, NT=1000, FW=10, DTINV=4, VELOCITY=1, FDORDER=4)
    eng = ifos_amd.Engine(w.cfg)
    eng.set_model(**w.start)
    eng.set_shot(w.shots[0].srcpos, w.shots[0].recpos)
    eng.forward(snapshots=False)
    want = [np.array(x) for x in eng.seismograms()]
    ms = eng.autotune(reps=3)[2]
    took = []
    for _ in range(5):
        t0 = time.perf_counter()
        eng.forward(snapshots=False)
        took.append((time.perf_counter() - t0) * 1e3 / w.cfg.NT)
    assert eng.get_resident()[1]
    print(f"autotuner {ms * 1e3:.2f} us a step, run {min(took) * 1e3:.2f}", flush=True)
    assert ms < 1.5 * min(took)
    for x, y in zip(want, eng.seismograms()):
        assert np.array_equal(x, y)
