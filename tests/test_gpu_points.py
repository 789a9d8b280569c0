"""Sources and receivers looked up by cell: several points at one cell act in
the caller's order, dense receiver lines cross tile edges, and points sit in
the last, partly filled tile -- bit for bit against the oracle, with every
velocity-step shape and the one-kernel step."""
import numpy as np
import pytest

import ifos_amd
from ifos_amd import workloads
import oracle_lib as O
from test_precision import params_of

pytestmark = pytest.mark.gpu


def points(NX, NY):
    """A receiver in every cell of row 3, doubled at tile edges (in an order
    that is not the cells'), and in the corners."""
    rec = [(x, 3) for x in range(1, NX + 1)]
    rec += [(x, 3) for x in (64, 65, 1, NX, 64)] + [(NX, NY), (1, NY), (NX, 1), (NX, NY)]
    src = [workloads.source_row(x, y, 25.0, amp=a, stype=t, azimuth=30.0)
           for x, y, a, t in ((30, 8, 1e10, 4), (30, 8, 3e9, 2), (64, 9, 2e9, 3), (30, 8, 5e9, 1), (65, 9, 1e9, 1))]
    return np.stack(src), np.array(rec, np.int32)


@pytest.mark.parametrize("shape", [1, 2, 4, "fused"])
@pytest.mark.parametrize("case", [dict(FDORDER=4, L=0, VELOCITY=0, DTINV=2), dict(FDORDER=8, L=2, VELOCITY=1, DTINV=3)],
                         ids=["el4_v0", "visc8_v1"])
def test_points_by_cell_match_oracle(gpu_lib, case, shape):
    w = workloads.small_case(seed=81, NX=70, NY=43, NT=120, FW=8, **case)
    print(f"[points] {case} shape {shape}", flush=True)
    p = params_of(w)
    src, rec = points(70, 43)
    ovx, ovy, _ = O.forward(p, w.true, src, rec)
    ovx[:, 0] = 0
    ovy[:, 0] = 0
    ref = O.gradient(p, w.start, src, rec, ovx, ovy)
    eng = ifos_amd.Engine(w.cfg)
    eng.set_model(**w.start)
    eng.set_shot(src[:1], rec[:4])  # points of an earlier shot leave no trace
    eng.set_shot(src, rec)
    if shape == "fused":
        eng.set_fused(True)
    else:
        eng.set_velocity_rows(shape)
    eng.shot_gradient(ovx, ovy)
    vx, vy = eng.seismograms()
    g = eng.gradient()
    eng.close()
    np.testing.assert_array_equal(vx, ref["seis_vx"])
    np.testing.assert_array_equal(vy, ref["seis_vy"])
    for k, n in enumerate(("vp", "vs", "rho")):
        np.testing.assert_array_equal(g[k], ref["grad_" + n], err_msg=n)
