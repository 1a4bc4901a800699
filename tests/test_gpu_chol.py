"""pscf_batch_chol's one-pass elimination at small, block-edge and the largest
nao its LDS holds (143), against NumPy's Cholesky and triangular inverse in FP64.
The substitution's error is below N eps times the condition number of S (at most
50 here): 1e-11 of the largest element of L^-1."""
import numpy as np
import pytest
import torch

from pyscf_ipu_amd import _lib, device

pytestmark = pytest.mark.gpu


def _run(mats, sizes):
    desc = np.zeros((len(sizes), 16), np.int64)
    off = np.concatenate([[0], np.cumsum([n * n for n in sizes])])
    for m, n in enumerate(sizes):
        desc[m, 2], desc[m, 12] = n, off[m]  # nao, mat0
    d_desc, S = device.to_dev(desc), device.to_dev(np.concatenate([a.reshape(-1) for a in mats]))
    out, ctl = torch.full_like(S, float("nan")), device.zeros((len(sizes), 8), torch.float64)
    ctl[:, 1] = 1.0
    _lib.call("pscf_batch_chol", device.ptr(d_desc), len(sizes), max(sizes), device.ptr(S), device.ptr(out),
              device.ptr(ctl), device.stream())
    o = out.cpu().numpy()
    return [o[off[m]:off[m + 1]].reshape(n, n) for m, n in enumerate(sizes)], ctl.cpu().numpy()


def test_chol_sizes(hip):
    sizes = [1, 2, 16, 63, 64, 65, 143]
    rng = np.random.default_rng(2)
    mats = []
    for n in sizes:
        q = np.linalg.qr(rng.standard_normal((n, n)))[0]
        mats.append((q * np.linspace(0.1, 5.0, n)) @ q.T)
    got, ctl = _run([0.5 * (a + a.T) for a in mats], sizes)
    assert (ctl[:, 1] == 1.0).all() and (ctl[:, 2] == 0.0).all()
    for a, g in zip(mats, got):
        ref = np.linalg.inv(np.linalg.cholesky(0.5 * (a + a.T)))
        assert np.array_equal(np.triu(g, 1), np.zeros_like(g))
        assert np.abs(g - np.tril(ref)).max() < 1e-11 * np.abs(ref).max()


def test_chol_not_positive_definite(hip):
    a = np.diag([1.0, 2.0, -1.0, 3.0])
    _, ctl = _run([np.eye(3), a], [3, 4])
    assert list(ctl[:, 1]) == [1.0, 0.0] and list(ctl[:, 2]) == [0.0, -1.0]
