"""The bitwise comparisons with the reference's golden vectors and with the
oracle, over both time loops: the one launch (k_resident), which these small
grids take by default, and the per-step kernels, which the large ones keep."""
import pytest

import ifos_amd
import test_gpu_eprecond as eprecond
import test_gpu_materials as materials
import test_gpu_parity as parity
import test_gpu_precision as precision

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[0, 1], ids=["per_step", "one_launch"], autouse=True)
def loop(request, monkeypatch):
    """Engines of the test take one loop, and every run is seen to have taken it."""
    runs = []

    class Engine(ifos_amd.Engine):
        def __init__(self, *args, **kw):
            super().__init__(*args, **kw)
            self.set_resident(request.param)

        def _ran(self):
            runs.append(self.get_resident()[1])

        def forward(self, *args, **kw):
            super().forward(*args, **kw)
            self._ran()

        def shot_gradient(self, *args, **kw):
            out = super().shot_gradient(*args, **kw)
            self._ran()
            return out

    monkeypatch.setattr(ifos_amd, "Engine", Engine)
    print(f"[both loops] {request.node.name}", flush=True)
    yield
    assert runs and set(runs) == {bool(request.param)}


@pytest.mark.parametrize("name", parity.CASES)
def test_golden_forward(gpu_lib, name):
    parity.test_forward_matches_reference(gpu_lib, name)


@pytest.mark.parametrize("name", parity.CASES)
def test_golden_gradient(gpu_lib, name):
    parity.test_gradient_matches_reference(gpu_lib, name)


@pytest.mark.parametrize("case", [(10, 0, 0, 1, 1), (12, 2, 1, 1, 1), (8, 3, 1, 0, 3), (4, 2, 0, 1, 2), (2, 1, 1, 0, 4)],
                         ids=str)
def test_oracle_forward(gpu_lib, case):
    parity.test_forward_matches_oracle(gpu_lib, *case)


@pytest.mark.parametrize("kmax,npower", [(4.0, 2.0), (2.5, 3.0), (8.0, 4.0)])
def test_stretched_pml(gpu_lib, kmax, npower):
    parity.test_stretched_pml_matches_oracle(gpu_lib, kmax, npower)


@pytest.mark.parametrize("adj", [2, 3])
def test_adjoint_type(gpu_lib, adj):
    parity.test_adjoint_type_matches_oracle(gpu_lib, adj)


def test_kill_mask(gpu_lib):
    parity.test_gradient_matches_oracle_with_kill(gpu_lib)


def test_two_shots_sum(gpu_lib):
    parity.test_two_shots_sum(gpu_lib)


@pytest.mark.parametrize("mode,per_shot,L,fp64", [(1, 1, 0, 0), (1, 0, 2, 1), (3, 1, 2, 0), (3, 0, 0, 1)])
def test_energy_preconditioner(gpu_lib, mode, per_shot, L, fp64):
    eprecond.test_eprecond_matches_oracle(gpu_lib, mode, per_shot, L, fp64)


@pytest.mark.parametrize("case", precision.PREC_CASES, ids=["visc8_v1", "el4_v0"])
def test_16bit_snapshots(gpu_lib, case):
    precision.test_snapshot16_gradient_matches_oracle(gpu_lib, case)


@pytest.mark.parametrize("L", [0, 2])
def test_materials(gpu_lib, L):
    materials.test_materials_match_oracle(gpu_lib, 65, 45, L)
