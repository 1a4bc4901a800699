"""The fused pointwise stage of the large-molecule XC (stage 2 of
pscf_xc_large_stage) against stages 0 and 1, at the edges of its 16-point tiles
and of its variants' nao (128, 176, 256) and past the largest.  Both form the same FP64
sums in another order: 1e-12 of the largest value; Y rounded to a narrower type
may then fall to the neighbouring value, one unit of its last place."""
import numpy as np
import pytest
import torch

from pyscf_ipu_amd import _lib, device

pytestmark = pytest.mark.gpu
TYPES = {0: (torch.bfloat16, 2.0 ** -7), 1: (torch.float16, 2.0 ** -10), 2: (torch.float32, 2.0 ** -23),
         3: (torch.float64, 1e-12)}


@pytest.mark.parametrize("ty", list(TYPES))
@pytest.mark.parametrize("N,g", [(1, 1), (15, 16), (17, 17), (128, 257), (129, 15), (176, 1000), (177, 33),
                                 (256, 40), (257, 40)])
def test_fused_stage_equals_two(hip, ty, N, g):
    tdt, unit = TYPES[ty]
    gen = torch.Generator().manual_seed(N + g)
    phi = (torch.rand((4, N, g), generator=gen, dtype=torch.float64) * 0.2).to(tdt).cuda()
    X = (torch.rand((N, g), generator=gen, dtype=torch.float64) + 0.05).cuda()
    w = torch.rand(g, generator=gen, dtype=torch.float64).cuda()
    P, st = device.ptr, device.stream()
    n = _lib.lib().pscf_xc_large_parts(g)
    out = []
    for fused in (False, True):
        coef = torch.full((4, g), float("nan"), dtype=torch.float64, device="cuda")
        e = torch.full((n,), float("nan"), dtype=torch.float64, device="cuda")
        Y = torch.zeros((N, g), dtype=tdt, device="cuda")
        if fused:
            _lib.call("pscf_xc_large_stage", 2, ty, N, g, P(X), P(phi), P(w), 1e-20, P(coef), P(e), P(Y), st)
        else:
            _lib.call("pscf_xc_large_stage", 0, ty, N, g, P(X), P(phi), P(w), 1e-20, P(coef), P(e), None, st)
            _lib.call("pscf_xc_large_stage", 1, ty, N, g, None, P(phi), None, 1e-20, P(coef), None, P(Y), st)
        Vh = torch.zeros((N, N), dtype=torch.float64, device="cuda")
        V, exc = torch.empty_like(Vh), torch.empty(1, dtype=torch.float64, device="cuda")
        _lib.call("pscf_xc_large_finish", N, P(Vh), P(e), n, P(V), P(exc), st)
        out.append([x.double().cpu().numpy() for x in (coef, exc, Y)])
    for a, b, tol in zip(out[0], out[1], (1e-12, 1e-12, max(unit, 1e-12))):
        assert np.all(np.isfinite(a)) and np.all(np.isfinite(b))
        assert np.abs(a - b).max() <= tol * np.abs(a).max()
