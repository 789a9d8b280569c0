"""The one-launch time loop with several rows of cells per thread: against the
per-step kernels, bit for bit, with every option of a run on and the fields
alive everywhere; which runs take it; the autotuner's report of it."""
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


# rows of cells per thread that the plan gives on 256 compute units, NX, NY, shots, L,
# FDORDER and the options: stretched CPML unless k=1, bottom and top strips, integrated
# adjoint velocity, 16-bit scales over several rows of a thread, energies, several shots
ROWS = [
    dict(R=2, NX=1024, NY=509, L=2, FDORDER=8, snap="bf16", FREE_SURF=0),
    dict(R=2, NX=500, NY=480, shots=2, L=0, FDORDER=4, VELOCITY=0, ep=1),
    dict(R=2, NX=1000, NY=300, L=3, FDORDER=12, snap="fp16", ep=3, DTINV=1),
    dict(R=3, NX=1024, NY=760, L=2, FDORDER=8, VELOCITY=0, ep=1, ep64=1, FREE_SURF=0),
    dict(R=3, NX=510, NY=700, shots=2, L=1, FDORDER=6, snap="bf16", ep=1),
    dict(R=3, NX=1024, NY=767, L=3, FDORDER=8, snap="fp16", DTINV=2, FREE_SURF=0),
    dict(R=3, NX=960, NY=768, L=0, FDORDER=2, VELOCITY=0, k=1.0),
    dict(R=4, NX=1024, NY=1010, L=2, FDORDER=8, snap="bf16", ep=1, FREE_SURF=0),
    dict(R=4, NX=500, NY=1000, shots=2, L=1, FDORDER=12, VELOCITY=0, ep=3, ep64=1),
    dict(R=4, NX=1024, NY=900, L=0, FDORDER=10, snap="fp16", DTINV=1, FREE_SURF=0),
    dict(R=5, NX=1024, NY=1270, L=0, FDORDER=12, ep=1, ep64=1, FREE_SURF=0),
    dict(R=5, NX=1024, NY=1034, L=0, FDORDER=8, FREE_SURF=0),
    dict(R=5, NX=500, NY=1250, shots=2, L=0, FDORDER=8, VELOCITY=0, snap="bf16", ep=1),
    dict(R=6, NX=1024, NY=1530, L=0, FDORDER=8, snap="fp16", ep=1, FREE_SURF=0),
    dict(R=6, NX=500, NY=1500, shots=2, L=0, FDORDER=4, VELOCITY=0, ep=3, DTINV=1),
]


def plan(c):
    """Rows of cells per thread and of a tile (resident_plan, 256 compute units)."""
    nbx, N = -(-c["NX"] // 64), c["FDORDER"] // 2
    across = 256 // (nbx * c.get("shots", 1))
    th = max(-(-c["NY"] // across), N + c.get("FREE_SURF", 1))
    rows = next(r for r in range(1, 7) if th <= 16 * r)
    ty = -(-th // rows)
    while c.get("snap") and ty * rows % 8:
        ty += 1
    return rows, ty * rows


def full_run(c, mode):
    """Gradient and forward run with sources and receivers all over the grid: in several
    rows of one thread, on both sides of every tile edge, in the strips and corners."""
    NX, NY, shots, NT = c["NX"], c["NY"], c.get("shots", 1), 24
    w = workloads.small_case(seed=15, NX=NX, NY=NY, L=c["L"], NT=NT, FW=12, DTINV=c.get("DTINV", 3),
                             VELOCITY=c.get("VELOCITY", 1), FDORDER=c["FDORDER"], FREE_SURF=c.get("FREE_SURF", 1))
    w.cfg.k_max_PML, w.cfg.npower = c.get("k", 8.0), 4.0
    edge = plan(c)[1]
    ys = sorted({y for e in range(0, NY + edge, edge) for y in (e - 1, e, e + 1, e + 2) if 1 <= y <= NY} | {NY})
    ys += [y for y in range(5, NY, 29)]
    rng = np.random.default_rng(16)
    eng = ifos_amd.Engine(w.cfg, slots=shots)
    eng.set_resident(mode)
    if c.get("snap"):
        eng.set_snapshot_precision(c["snap"])
    if c.get("ep"):
        eng.set_eprecond(c["ep"], per_shot=True)
        eng.set_eprecond_fp64(c.get("ep64", 0))
    eng.set_model(**w.start)
    run = []
    for k in range(shots):
        xy = [(x, y) for y in ys for x in range(1 + (7 * y + 3 * k) % 23, NX + 1, 23)]
        src = np.stack([workloads.source_row(x, y, 25.0, amp=10.0 ** rng.uniform(9, 10), stype=1 + (x + y) % 4,
                                             azimuth=30.0) for x, y in xy])
        src[-1, 7] = 1 + k  # the last one's type says whether explosive ones act
        rec = [(x, y) for x in (5, 64, 65, NX) for y in range(1, NY + 1)] + [(x, NY) for x in range(1, NX + 1, 3)]
        rec += [(x + 1 if x < NX else x, y) for x, y in xy[::5]]
        run.append((src, np.array(rec, np.int32)))
    eng.set_shots(run)
    obs = rng.standard_normal((2, sum(len(r) for _, r in run), NT)).astype(np.float32)
    out = [np.array(eng.shot_gradient(obs[0], obs[1]))]
    last = eng.get_resident()[1]
    out += [np.array(g) for g in eng.gradient()] + [np.array(s) for s in eng.seismograms()]
    out += [np.array(g) for k in range(shots) for g in eng.slot_gradient(k)]
    if c.get("ep"):
        out.append(np.array(eng.energy_weight(0)))
    adjoint_fields = np.array(eng.fields())
    eng.forward(snapshots=False)
    return out, adjoint_fields, np.array(eng.fields()), last and eng.get_resident()[1]


@pytest.mark.parametrize("c", ROWS, ids=lambda c: "-".join(f"{k}{v}" for k, v in c.items()))
def test_rows_of_a_thread_equal_per_step_kernels(gpu_lib, c):
    print(f"[resident] {c}", flush=True)
    rows, edge = plan(c)
    assert rows == c["R"]
    want, want_adj, want_fwd, used = full_run(c, 0)
    assert not used
    have, have_adj, have_fwd, used = full_run(c, 1)
    assert used
    for fields in (want_adj, want_fwd):  # what crosses the tile edges is not zero
        for e in range(edge, c["NY"], edge):
            assert np.mean(fields[:, e - 1:e + 1] != 0) > 0.9
        assert np.mean(fields[:, :, 63:65] != 0) > 0.9 and np.isfinite(fields).all()
    for k, (a, b) in enumerate(zip(want + [want_adj, want_fwd], have + [have_adj, have_fwd])):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), f"output {k}"
