"""pscf_jk_sparse on lists that do and do not let a wave sum its lanes first:
packed order, shuffled, single lines, elements out of range anywhere, few and
many elements, nao up to where the copies leave the LDS; symmetric dm and any
other (one element off symmetry included).  Against the
16 patterns in FP64 on the host: 1e-13 (FP64) and 1e-6 (FP32: a few dozen
additions of values near the largest result's size) of the largest sum of
magnitudes."""
import numpy as np
import pytest
import torch

from pyscf_ipu_amd.nanoDFT import sparse_symmetric_ERI as sse

pytestmark = pytest.mark.gpu
TOL = {"float64": 1e-13, "float32": 1e-6}


def _reference(v, idx, dm, N, absolute=False):
    d = np.abs(dm) if absolute else dm
    v = np.abs(v) if absolute else v
    i, j, k, l = idx.astype(np.int64).T
    ok = (idx >= 0).all(1) & (idx < N).all(1)
    v, i, j, k, l = v[ok], i[ok], j[ok], k[ok], l[ok]
    out = np.zeros((N, N))
    h = 0.1 if absolute else -0.1
    for a, b, val in ((k, l, v * (d[i, j] + d[j, i])), (l, k, v * (d[i, j] + d[j, i])),
                      (i, j, v * (d[k, l] + d[l, k])), (j, i, v * (d[k, l] + d[l, k])),
                      (i, l, h * v * d[k, j]), (j, l, h * v * d[k, i]), (i, k, h * v * d[l, j]), (j, k, h * v * d[l, i]),
                      (k, j, h * v * d[i, l]), (l, j, h * v * d[i, k]), (k, i, h * v * d[j, l]), (l, i, h * v * d[j, k])):
        np.add.at(out, (a, b), val)
    return out


def _packed(N, rng, keep):
    P = N * (N + 1) // 2
    nz = np.sort(rng.choice(P * (P + 1) // 2, size=min(keep, P * (P + 1) // 2), replace=False)).astype(np.uint64)
    ij, kl = sse.get_i_j(nz)
    return np.stack(sse.get_i_j(ij) + sse.get_i_j(kl), axis=1).astype(np.int16)


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("order", ["packed", "shuffled", "dropped", "line"])
@pytest.mark.parametrize("sym", ["symmetric", "any", "nearly"])
@pytest.mark.parametrize("N,nnz", [(1, 1), (7, 63), (7, 406), (24, 64), (24, 30000), (59, 65), (60, 50000), (101, 9000),
                                   (144, 5000), (160, 3000)])
def test_jk_sparse_lists(hip, dtype, order, sym, N, nnz):
    rng = np.random.default_rng(N + nnz)
    idx = _packed(N, rng, nnz)
    if order == "shuffled":
        idx = idx[rng.permutation(len(idx))]
    elif order == "dropped":  # out of range here and there, and a block at the end
        idx[rng.random(len(idx)) < 0.01, rng.integers(4)] = N
        idx[len(idx) - len(idx) // 10:, 0] = -1
    elif order == "line":  # one i, j for all
        idx[:, 0], idx[:, 1] = N - 1, N // 2
    v = rng.standard_normal(len(idx)).astype(dtype)
    dm = rng.standard_normal((N, N)).astype(dtype)
    if sym != "any":
        dm = np.tril(dm) + np.tril(dm, -1).T
        if sym == "nearly":
            dm[0, N - 1] += 0.5
    got = sse.sparse_symmetric_einsum(torch.from_numpy(v).cuda(), torch.from_numpy(idx).cuda(),
                                      torch.from_numpy(dm).cuda()).cpu().numpy().reshape(N, N)
    v64, d64 = v.astype(np.float64), dm.astype(np.float64)
    scale = _reference(v64, idx, d64, N, absolute=True).max()
    assert np.abs(got - _reference(v64, idx, d64, N)).max() <= TOL[dtype] * max(scale, 1e-30)
