"""The network's tiled GEMM (csrc/mlp.hip) at the edges of its tiles, against
FP32 products of the same BF16 operands.

Tolerance: FP32 accumulation of K products of size about |a||b|: 2^-24 sqrt(K)
of the row sums of |a||b| is below 1e-5 of their largest for K <= 4096; BF16
results add their rounding, 2^-8 of the value."""
import numpy as np
import pytest
import torch

from pyscf_ipu_amd import _lib, device

pytestmark = pytest.mark.gpu
P = device.ptr


def _rand(rows, cols, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(rows, cols, device="cuda", generator=g).to(torch.bfloat16)


def _gemm(op, M, N, K, A, lda, B, ldb, bias, aux, out, out2, ldc, ks=1):
    _lib.call("pscf_mlp_gemm", op, M, N, K, P(A), lda, P(B), ldb, P(bias), P(aux), P(out), P(out2), ldc, ks,
              device.stream())
    torch.cuda.synchronize()


def _close(got, ref, scale, tol=1e-5):
    assert float(((got - ref).abs() / scale).max()) < tol


# 16-byte aligned rows (tiled kernel) and odd leading dimensions (general one);
# one row, tile edges, and enough rows for the 128 x 128 tiles
@pytest.mark.parametrize("M", [1, 63, 65, 129, 16400])
@pytest.mark.parametrize("K,lda,N,ldb", [(43, 64, 256, 256), (256, 256, 256, 256), (256, 256, 32, 32),
                                         (33, 40, 72, 72), (45, 47, 30, 31)])
def test_forward_layers(hip, M, K, lda, N, ldb):
    A, B = _rand(M, lda, 1), _rand(K, ldb, 2)
    bias = torch.randn(N, device="cuda")
    z, h = torch.empty(M, N, device="cuda"), torch.empty(M, N, device="cuda", dtype=torch.bfloat16)
    a, b = A[:, :K].float(), B[:, :N].float()
    ref = a @ b + bias
    scale = (a.abs() @ b.abs()).max()
    _gemm(0, M, N, K, A, lda, B, ldb, bias, None, z, h, N)
    _close(z, ref, scale)
    _close(h.float(), torch.nn.functional.silu(ref), scale, 5e-3)
    _gemm(1, M, N, K, A, lda, B, ldb, bias, None, z, None, N)
    _close(z, ref, scale)


@pytest.mark.parametrize("M", [1, 63, 129, 16400])
@pytest.mark.parametrize("K,ld,N", [(32, 32, 256), (256, 256, 256), (40, 48, 24)])
def test_backward_data(hip, M, K, ld, N):
    A, W = _rand(M, ld, 3), _rand(N, ld, 4)
    aux = torch.randn(M, N, device="cuda")
    s = torch.sigmoid(aux)
    a, w = A[:, :K].float(), W[:, :K].float()
    ref = (a @ w.T) * (s * (1 + aux * (1 - s)))
    scale = (a.abs() @ w.abs().T).max()
    out, o2 = torch.empty(M, N, device="cuda"), torch.empty(M, N, device="cuda", dtype=torch.bfloat16)
    _gemm(2, M, N, K, A, ld, W, ld, None, aux, out, o2, N)
    _close(out, ref, scale)
    # the form with column sums: the same BF16 values, sums added to what is there
    db, o3 = torch.full((N,), 2.0, device="cuda"), torch.empty_like(o2)
    _gemm(4, M, N, K, A, ld, W, ld, None, aux, db, o3, N)
    assert torch.equal(o2, o3)
    _close(db, 2.0 + out.sum(0), scale * M ** 0.5)


@pytest.mark.parametrize("rows,ksplit", [(1, 1), (31, 1), (1000, 1), (1000, 7), (4097, 64)])
@pytest.mark.parametrize("M,lda,N,ldb", [(43, 64, 256, 256), (256, 256, 256, 256), (256, 256, 32, 32), (30, 33, 29, 29)])
def test_weight_gradient(hip, rows, ksplit, M, lda, N, ldb):
    X, dY = _rand(rows, lda, 5), _rand(rows, ldb, 6)
    out = torch.ones(M, N, device="cuda")
    _gemm(3, M, N, rows, X, lda, dY, ldb, None, None, out, None, N, ksplit)
    x, y = X[:, :M].float(), dY[:, :N].float()
    _close(out, 1.0 + x.T @ y, (x.abs().T @ y.abs()).max())


@pytest.mark.parametrize("M,N,ld", [(1, 32, 32), (33, 256, 256), (5000, 45, 50)])
def test_colsum(hip, M, N, ld):
    dz = torch.randn(M, ld, device="cuda")
    db = torch.empty(N, device="cuda")
    _lib.call("pscf_mlp_colsum", M, N, P(dz), ld, P(db), device.stream())
    torch.cuda.synchronize()
    _close(db, dz[:, :N].double().sum(0).float(), dz.abs().sum(0).max())
