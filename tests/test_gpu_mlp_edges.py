"""The network's GEMM entry at the ends of its argument ranges, for aligned rows
(tiled kernel) and others (general one)."""
import pytest
import torch

from pyscf_ipu_amd import _lib, device

pytestmark = pytest.mark.gpu
P = device.ptr


@pytest.mark.parametrize("ld", [72, 71])
@pytest.mark.parametrize("op", [0, 1, 2, 3, 4])
def test_no_inner_dimension(hip, op, ld):
    """K = 0: an empty sum is zero, and the epilogue still runs.  Exact."""
    if op == 4 and ld % 8:
        pytest.skip("column sums need aligned rows")
    M, N = 70, 40
    A = torch.full((M, ld), float("nan"), device="cuda", dtype=torch.bfloat16)
    bias = torch.randn(N, device="cuda")
    aux = torch.randn(M, N, device="cuda")
    out = torch.full((M, N), 7.0, device="cuda")
    out2 = torch.full((M, N), 7.0, device="cuda", dtype=torch.bfloat16)
    _lib.call("pscf_mlp_gemm", op, M, N, 0, P(A), ld, P(A), ld, P(bias), P(aux), P(out), P(out2), N, 1,
              device.stream())
    torch.cuda.synchronize()
    z = bias.expand(M, N)
    if op in (0, 1):
        assert torch.equal(out, z)
    else:  # op 2 stores zeros; 3 and 4 add nothing to what is there
        assert torch.equal(out, torch.full_like(out, 0.0 if op == 2 else 7.0))
    if op == 0:
        assert float((out2.float() - torch.nn.functional.silu(z)).abs().max()) < 2 ** -8 * float(z.abs().max())
    if op in (2, 4):
        assert torch.equal(out2, torch.zeros_like(out2))
