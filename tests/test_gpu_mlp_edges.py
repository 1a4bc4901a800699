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


@pytest.mark.parametrize("M,K,N", [(70, 43, 45), (1, 1, 1), (129, 130, 33)])
def test_operands_end_with_their_last_row(hip, M, K, N):
    """Buffers of (rows - 1) ld + columns elements: nothing is read behind them
    (the elements that follow here are NaN).  Sums of up to 130 products of
    magnitude |a||b|, FP32 accumulation: 1e-5 of the largest row sum."""
    ld = 136
    gen = torch.Generator(device="cuda").manual_seed(7)

    def operand(rows, cols):
        n = (rows - 1) * ld + cols
        buf = torch.full((rows * ld + 64,), float("nan"), device="cuda", dtype=torch.bfloat16)
        buf[:n] = torch.randn(n, device="cuda", generator=gen).to(torch.bfloat16)
        return buf, torch.as_strided(buf, (rows, cols), (ld, 1)).float()

    def check(op, m, n, k, A, B, ref, scale, ks=1):
        out = torch.zeros(m, n, device="cuda")
        out2 = torch.empty(m, n, device="cuda", dtype=torch.bfloat16)
        zero, one = torch.zeros(n, device="cuda"), torch.full((m, n), 1e4, device="cuda")  # silu'(1e4) = 1
        _lib.call("pscf_mlp_gemm", op, m, n, k, P(A), ld, P(B), ld, P(zero), P(one), P(out), P(out2), n, ks,
                  device.stream())
        torch.cuda.synchronize()
        assert float((out - ref).abs().max()) < 1e-5 * float(scale.max())

    (A, a), (B, b), (W, w), (Y, y) = operand(M, K), operand(K, N), operand(N, K), operand(M, N)
    check(1, M, N, K, A, B, a @ b, a.abs() @ b.abs())
    check(2, M, N, K, A, W, a @ w.T, a.abs() @ w.abs().T)
    check(3, K, N, M, A, Y, a.T @ y, a.abs().T @ y.abs(), 2)
