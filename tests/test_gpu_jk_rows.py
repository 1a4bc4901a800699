"""pscf_jk_s8_large at the nao where its rows pass changes form (64-column
registers, packed D in LDS or not, the general kernel), against the streaming
pass over the expanded tensor (pscf_jk_s1, another kernel, FP64 sums).  An
element collects at most about 4 nao terms rounded to 2^-40: 5e-10 at nao 257,
so 1e-9."""
import pytest
import torch

from pyscf_ipu_amd import _lib, device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["fp64", "fp32"])
@pytest.mark.parametrize("N", [2, 9, 63, 64, 65, 128, 129, 161, 186, 187, 192, 193, 257])
def test_rows_forms(hip, dtype, N):
    if N > 190 and dtype == "fp32":
        pytest.skip("the forms above nao 190 once, in FP64")
    tdt, code = (torch.float64, _lib.F64) if dtype == "fp64" else (torch.float32, _lib.F32)
    pairs = N * (N + 1) // 2
    gen = torch.Generator(device="cuda").manual_seed(N)
    s8 = torch.rand(pairs * (pairs + 1) // 2, generator=gen, device="cuda", dtype=tdt) / N
    D = torch.randn((N, N), generator=gen, device="cuda", dtype=torch.float64)
    D = (0.5 * (D + D.T)).contiguous()
    P, st = device.ptr, device.stream()
    s1 = torch.empty(N ** 4, device="cuda", dtype=tdt)
    _lib.call("pscf_eri_s8_to_s1", code, P(s8), code, P(s1), N, st)
    ref = torch.empty((N, N), device="cuda", dtype=torch.float64)
    _lib.call("pscf_jk_s1", code, P(s1), N, P(D), 0.2, P(ref), st)
    del s1
    n = _lib.lib().pscf_jk_s8_large_workspace_bytes(N)
    ws, out = device.workspace(n), [torch.full((N, N), float("nan"), device="cuda", dtype=torch.float64) for _ in "ab"]
    for o in out:
        _lib.call("pscf_jk_s8_large", code, P(s8), N, P(D), 0.2, P(o), P(ws), n, st)
    assert torch.equal(out[0], out[1])  # repeats bit for bit
    assert float((out[0] - ref).abs().max()) < 1e-9 * max(1.0, float(ref.abs().max()))
    torch.cuda.empty_cache()
