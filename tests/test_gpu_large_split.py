"""V = phi0 Y^T of a large Fock build: FP32 accumulation in ranges of about 2048
grid points, FP64 accumulation in any."""
import pytest
import torch

from pyscf_ipu_amd import _lib, device
from pyscf_ipu_amd.gto import build_mol
from pyscf_ipu_amd.precision import LargeRKS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gemm,points", [("f32/f32", 2048), ("f64/f32", 2048), ("f32/f64", 4096), ("f64/f64", 4096)])
def test_fock_potential_ranges(hip, gemm, points):
    """Equal to a product in ranges of `points` up to FP64 rounding, 4096 x 2^-53 =
    5e-13 of a sum's size at worst: 1e-12 of the largest element (another length
    of FP32 range moves it by 1e-8)."""
    r = LargeRKS(build_mol("C 0 0 0; O 1.2 0 0; N -1.1 0.6 0; H -1.9 0.1 0.2; H -1.2 1.5 0", "6-31g"), 1, gemm, "fp64")
    r.setup()
    r.fock_parts()
    N, G, P = r.N, r.g, device.ptr
    assert G > 4 * 2048
    V = torch.zeros((N, N), device="cuda", dtype=torch.float64)
    _lib.call("pscf_gemm", r.gemm_type, r.acc64, 0, 1, 1, N, N, G, P(r.phi), G, P(r.Y), G, P(V), N, G // points,
              device.stream())
    assert float((r.Vh - V).abs().max()) < 1e-12 * float(V.abs().max())
