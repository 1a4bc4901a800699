"""pscf_xc's wave-private tiles against the NumPy oracle at their edges: nao at
both sides of a padded block (16 columns), grids at both sides of a wave's
share (16 points), a tile (64) and the 256 workgroups of a launch, both AO
layouts.  Synthetic AO values: the kernel takes any."""
import numpy as np
import pytest

from oracle import xc as oracle_xc

pytestmark = pytest.mark.gpu

# FP32: the longest chain is a density of N^2 <= 6400 products summed in blocks
# (about 80 + 5 + 4 additions deep) and its functional, a handful of powers and
# logarithms with amplification below ten: 100 * 10 * 2^-24 = 6e-5 at worst,
# rounding errors of random sign giving about its square root's share.
TOL = {"fp64": 1e-10, "fp32": 2e-5}


def _inputs(N, g, seed):
    rng = np.random.default_rng(seed)
    ao = np.empty((4, g, N))
    ao[0] = rng.uniform(0.1, 1.0, (g, N))
    ao[1:] = 0.5 * rng.standard_normal((3, g, N))
    C = rng.standard_normal((N, max(1, N // 2))) / np.sqrt(N)
    return ao, 2.0 * C @ C.T, rng.uniform(0.0, 2.0 / g, g)


@pytest.mark.parametrize("dtype", ["fp64", "fp32"])
@pytest.mark.parametrize("layout", ["g_N", "N_g"])
@pytest.mark.parametrize("N,g", [(1, 1), (1, 130), (15, 16), (16, 17), (17, 63), (33, 64), (48, 65), (49, 700),
                                 (64, 16400), (65, 129), (80, 3), (80, 16500)])
def test_xc_wave_tiles(hip, dtype, layout, N, g):
    import torch
    from pyscf_ipu_amd import _lib, device
    npdt, code = (np.float64, _lib.F64) if dtype == "fp64" else (np.float32, _lib.F32)
    ao, dm, w = (x.astype(npdt) for x in _inputs(N, g, 100 * N + g))
    E_ref, V_ref, _ = oracle_xc.exchange_correlation(*(x.astype(np.float64) for x in (dm, ao, w)))
    a = ao if layout == "g_N" else np.ascontiguousarray(ao.transpose(0, 2, 1))
    smu, sp = (1, N) if layout == "g_N" else (g, 1)
    d_ao, d_dm, d_w = (device.to_dev(torch.from_numpy(x)) for x in (a, dm, w))
    exc = device.empty(1, torch.float64)
    vxc = device.empty((N, N), torch.from_numpy(dm).dtype)
    n = _lib.lib().pscf_xc_workspace_bytes(code, N, g)
    ws = device.workspace(n)
    out = []
    for _ in range(2):
        _lib.call("pscf_xc", code, device.ptr(d_ao), g * N, smu, sp, g, N, device.ptr(d_dm), device.ptr(d_w), 1e-20,
                  device.ptr(exc), device.ptr(vxc), device.ptr(ws), n, device.stream())
        out.append((float(exc.item()), vxc.cpu().numpy().copy()))
    (E, V), (E2, V2) = out
    assert E == E2 and np.array_equal(V, V2)  # repeats bit for bit
    assert np.array_equal(V, V.T)
    tol = TOL[dtype]
    assert abs(E - E_ref) < tol * max(1.0 if dtype == "fp64" else 0.0, abs(E_ref))
    assert np.abs(V - V_ref).max() < tol * max(1.0 if dtype == "fp64" else 0.0, np.abs(V_ref).max())
