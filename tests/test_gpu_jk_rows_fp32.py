"""pscf_jk_s8_large with FP32 ERIs at the nao where its rows pass no longer keeps
a packed D in LDS (187), takes four columns a lane (193) and leaves the register
form (257).  The reference adds the same FP32 ERIs in FP64 (pscf_jk_s1): an
element collects at most about 4 nao terms rounded to 2^-40, so 1e-9."""
import pytest
import torch

from pyscf_ipu_amd import _lib, device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [192, 193, 256, 257])
def test_rows_forms_fp32(hip, N):
    pairs = N * (N + 1) // 2
    gen = torch.Generator(device="cuda").manual_seed(N)
    s8 = torch.rand(pairs * (pairs + 1) // 2, generator=gen, device="cuda", dtype=torch.float32) / N
    D = torch.randn((N, N), generator=gen, device="cuda", dtype=torch.float64)
    D = (0.5 * (D + D.T)).contiguous()
    P, st = device.ptr, device.stream()
    s1 = torch.empty(N ** 4, device="cuda", dtype=torch.float32)
    _lib.call("pscf_eri_s8_to_s1", _lib.F32, P(s8), _lib.F32, P(s1), N, st)
    ref = torch.empty((N, N), device="cuda", dtype=torch.float64)
    _lib.call("pscf_jk_s1", _lib.F32, P(s1), N, P(D), 0.2, P(ref), st)
    del s1
    n = _lib.lib().pscf_jk_s8_large_workspace_bytes(N)
    ws, out = device.workspace(n), torch.full((N, N), float("nan"), device="cuda", dtype=torch.float64)
    _lib.call("pscf_jk_s8_large", _lib.F32, P(s8), N, P(D), 0.2, P(out), P(ws), n, st)
    assert float((out - ref).abs().max()) < 1e-9 * max(1.0, float(ref.abs().max()))
    torch.cuda.empty_cache()
