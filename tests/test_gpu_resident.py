"""The time loop as one launch (k_resident) against the per-step kernels, bit
for bit, at the sizes where its tiles can go wrong: one cell past a tile edge,
tiles lower than the stencil's reach allows to go, a last tile row with a
single live row, the largest tiles of each row count, every stencil order and
mechanism count, 16-bit snapshots whose scales span workgroup rows; and a run
that is given up and repeated."""
import numpy as np
import pytest

import ifos_amd
from ifos_amd import workloads

pytestmark = pytest.mark.gpu


def outputs(w, mode, shots=1, snap="fp32", eprecond=0, wait=None):
    NX, NY = w.cfg.NX, w.cfg.NY
    eng = ifos_amd.Engine(w.cfg, slots=shots)
    eng.set_snapshot_precision(snap)
    if eprecond:
        eng.set_eprecond(eprecond, per_shot=True)
    eng.set_model(**w.start)
    rec = np.array([(x, 3) for x in range(1, NX + 1, 2)] + [(NX, NY), (1, NY), (min(64, NX), 3)], np.int32)
    src = [np.stack([workloads.source_row(NX // 2 + k, min(8, NY), 25.0, amp=1e10, stype=1 + k % 3),
                     workloads.source_row(NX // 2 + k, min(8, NY), 25.0, amp=3e9, stype=2)]) for k in range(shots)]
    eng.set_shots([(s, rec) for s in src])
    eng.set_resident(mode)
    if wait is not None:
        eng.set_resident_wait(wait)
    obs = np.random.default_rng(3).standard_normal((2, len(rec) * shots, w.cfg.NT)).astype(np.float32)
    misfit = eng.shot_gradient(obs[0], obs[1])
    last = eng.get_resident()[1]
    out = [np.array(misfit)] + [np.array(g) for g in eng.gradient()] + list(eng.seismograms()) + [eng.fields()]
    return out, last


def same_bits(a, b):
    return all(np.array_equal(x.view(np.uint8), y.view(np.uint8)) for x, y in zip(a, b))


CASES = [dict(NX=65, NY=43, FDORDER=2, L=1), dict(NX=64, NY=40, FDORDER=4, L=0, VELOCITY=0),
         dict(NX=129, NY=33, FDORDER=6, L=2, VELOCITY=0), dict(NX=70, NY=41, FDORDER=8, L=3),
         dict(NX=127, NY=49, FDORDER=10, L=0), dict(NX=130, NY=57, FDORDER=12, L=2, FREE_SURF=0)]


@pytest.mark.parametrize("c", CASES, ids=lambda c: "-".join(f"{k}{v}" for k, v in c.items()))
@pytest.mark.parametrize("kw", [{}, dict(shots=3, eprecond=1), dict(snap="bf16")], ids=["plain", "shots3", "bf16"])
def test_resident_equals_per_step_kernels(gpu_lib, c, kw):
    w = workloads.small_case(seed=7, NT=36, FW=8, DTINV=3, **dict(dict(VELOCITY=1), **c))
    print(f"[resident] {c} {kw}", flush=True)
    want, used = outputs(w, 0, **kw)
    assert not used
    have, used = outputs(w, 1, **kw)
    assert used and same_bits(want, have)


# NX, NY, L: the lowest and highest tiles of the row counts on 256 compute units,
# and the highest order for which the run takes them
LARGE = [(64, 4096, 0, 12), (64, 4097, 2, 12), (1024, 512, 1, 12), (1024, 640, 3, 12), (960, 816, 2, 12),
         (1024, 768, 3, 12), (1024, 896, 2, 8), (1024, 1024, 1, 12), (900, 1224, 0, 12), (1024, 1408, 0, 8),
         (1024, 1536, 0, 8), (1024, 513, 3, 2)]


@pytest.mark.parametrize("NX,NY,L,highest", LARGE)
@pytest.mark.parametrize("order", [2, 8, 12])
def test_resident_large_tiles(gpu_lib, NX, NY, L, highest, order):
    """Every row count, from one row per thread of a full chip to the largest tile."""
    w = workloads.small_case(seed=8, NX=NX, NY=NY, L=L, NT=12, FW=10, DTINV=2, VELOCITY=1, FDORDER=order)
    print(f"[resident] {NX}x{NY} L={L} FDORDER {order}", flush=True)
    want, _ = outputs(w, 0)
    have, used = outputs(w, 1)
    assert same_bits(want, have) and used == (order <= highest)


def test_run_given_up_is_repeated(gpu_lib):
    """With no patience at all a workgroup gives up at its first unanswered
    look; the per-step kernels then deliver the run."""
    w = workloads.small_case(seed=9, NX=200, NY=90, NT=36, FW=8, DTINV=3, FDORDER=4, L=2, VELOCITY=1)
    want, _ = outputs(w, 0, eprecond=1)
    have, used = outputs(w, 1, eprecond=1, wait=0.0)
    assert not used and same_bits(want, have)
    # by rule: given up, one run without it, tried again (given up, two without)
    eng = ifos_amd.Engine(w.cfg)
    eng.set_model(**w.start)
    eng.set_shot(w.shots[0].srcpos, w.shots[0].recpos)
    eng.set_resident_wait(0.0)
    seen = []
    for _ in range(6):
        seen.append(eng.get_resident()[0])
        eng.forward(snapshots=False)
        assert not eng.get_resident()[1]
    assert seen == [True, False, True, False, False, True]
    eng.set_resident_wait(-1.0)
    eng.set_resident(-1)
    eng.forward(snapshots=False)
    assert eng.get_resident() == (True, True)


def test_which_runs_take_it(gpu_lib):
    w = workloads.small_case(seed=9, NX=200, NY=90, NT=12, FW=8, FDORDER=4)
    eng = ifos_amd.Engine(w.cfg)
    eng.set_model(**w.start)
    eng.set_shot(w.shots[0].srcpos, w.shots[0].recpos)
    assert eng.get_resident() == (True, False)
    eng.forward(snapshots=False)
    assert eng.get_resident() == (True, True)
    eng.set_graphs(1)  # a loop of the caller's choice
    eng.forward(snapshots=False)
    assert eng.get_resident() == (False, False)
    big = workloads.small_case(seed=9, NX=64, NY=40, NT=12, FW=8, FDORDER=4)
    big.cfg.BOUNDARY = 1  # periodic sides: per-step kernels
    eng = ifos_amd.Engine(big.cfg)
    eng.set_model(**big.start)
    eng.set_shot(big.shots[0].srcpos, big.shots[0].recpos)
    eng.set_resident(1)
    assert not eng.get_resident()[0]
