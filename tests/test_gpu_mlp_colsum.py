"""Bias gradients: a fixed order of summation, bit for bit."""
import pytest
import torch

from pyscf_ipu_amd import _lib, device

pytestmark = pytest.mark.gpu


def _ordered(dz):
    """256 sums over every 256th row, a tree over each 64 of them, the four in order."""
    s = torch.zeros(256, dz.shape[1], device=dz.device)
    for m in range(0, len(dz), 256):
        s[:len(dz[m:m + 256])] += dz[m:m + 256]
    s = s.reshape(4, 64, -1)
    for off in (32, 16, 8, 4, 2, 1):
        s = s[:, :off] + s[:, off:2 * off]
    return s[0, 0] + s[1, 0] + s[2, 0] + s[3, 0]


@pytest.mark.parametrize("M,N,ld", [(0, 5, 5), (1, 1, 1), (255, 31, 33), (257, 32, 32), (5000, 256, 256),
                                    (2049, 70, 71)])
def test_colsum_order(hip, M, N, ld):
    dz = torch.randn(max(M, 1), ld, device="cuda", generator=torch.Generator(device="cuda").manual_seed(M))
    db = torch.full((N,), float("nan"), device="cuda")
    _lib.call("pscf_mlp_colsum", M, N, device.ptr(dz), ld, device.ptr(db), device.stream())
    ref = _ordered(dz[:M, :N])
    assert torch.equal(db, ref)
    db.fill_(float("nan"))
    ws = torch.empty(256, N, device="cuda")
    _lib.call("pscf_mlp_colsum_ws", M, N, device.ptr(dz), ld, device.ptr(db), device.ptr(ws), device.stream())
    assert torch.equal(db, ref)


def test_colsum_many_rows(hip):
    """More rows than 65535 blocks of 256 hold: ones in the last 300, exact."""
    M = 65535 * 256 + 300
    dz = torch.zeros(M, 1, device="cuda")
    dz[-300:] = 1
    db = torch.empty(1, device="cuda")
    _lib.call("pscf_mlp_colsum", M, 1, device.ptr(dz), 1, device.ptr(db), device.stream())
    assert db.item() == 300


def test_bias_gradients_repeat(hip):
    from pyscf_ipu_amd import learned_guess as lg
    B = 5000
    gen = torch.Generator(device="cuda").manual_seed(3)
    X = torch.randn(B, lg.NIN_PAD, device="cuda", generator=gen).to(torch.bfloat16)
    X[:, lg.NIN:] = 0
    Y = torch.randn(B, lg.NOUT_PAD, device="cuda", generator=gen)
    mask = torch.ones_like(Y)
    model = lg.PairMLP.load()
    got = []
    for _ in range(4):
        model.loss_and_grads(X, Y, mask, B, nvalid=float(mask.sum()))
        g, at, one = model.g.clone(), 0, {}
        for name, r, c in lg.LAYOUT:
            one[name] = g[at:at + r * c]
            at += r * c
        got.append(one)
    for other in got[1:]:
        assert all(torch.equal(got[0][b], other[b]) for b in ("b0", "b1", "b2", "b3"))
