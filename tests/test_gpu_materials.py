"""Materials formed on the device (k_materials): averages across the last row
and column (which wrap), cells without shear stiffness, sizes around its 64x4
blocks -- forward traces bit for bit against the oracle, whose materials the
host code forms."""
import numpy as np
import pytest

import ifos_amd
from ifos_amd import workloads
import oracle_lib as O
from test_precision import params_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [0, 2])
@pytest.mark.parametrize("NX,NY", [(63, 41), (64, 44), (65, 45)])
def test_materials_match_oracle(gpu_lib, NX, NY, L):
    w = workloads.small_case(seed=91, NX=NX, NY=NY, NT=90, FW=8, FDORDER=4, L=L, FREE_SURF=0)
    print(f"[materials] {NX}x{NY} L={L}", flush=True)
    model = {k: v.copy() for k, v in w.true.items()}
    model["vs"][18:22, 5:NX - 4] = 0.0  # a fluid layer
    src = workloads.source_row(NX // 2, 12, 25.0, amp=1e10)[None, :]
    # receivers beside the last row and column, where the averages wrap
    rec = np.array([(x, 25) for x in range(2, NX + 1, 3)] + [(NX, y) for y in range(3, NY, 5)] +
                   [(x, NY) for x in range(1, NX, 7)], np.int32)
    ovx, ovy, _ = O.forward(params_of(w), model, src, rec)
    eng = ifos_amd.Engine(w.cfg)
    eng.set_model(**w.start)  # another model first: nothing of it stays
    eng.set_model(**model)
    eng.set_shot(src, rec)
    eng.forward(snapshots=False)
    vx, vy = eng.seismograms()
    assert np.array_equal(vx, ovx) and np.array_equal(vy, ovy)
