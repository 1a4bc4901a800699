"""The shell-pair ERI engine (csrc/eri_pairs.h) at the sizes where its tiles,
chunks and stages break: against the FP64 CPU oracle.

Tolerances as for the other ERI tests: FP64 1e-12, FP32 2e-6 of the largest
integral (at least 1)."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import cint
from pyscf_ipu_amd import batch, device, gto, molgen
from pyscf_ipu_amd.gto import build_mol

pytestmark = pytest.mark.gpu
TOL = {"fp64": 1e-12, "fp32": 2e-6}


def _check(got, ref, dtype):
    assert got.shape == ref.shape
    assert np.abs(got.astype(np.float64) - ref).max() < TOL[dtype] * max(1.0, np.abs(ref).max())


def _contract(mol, nprims, seed=0):
    """mol with its shells' contractions replaced by nprims[i] primitives each,
    exponents spread over 0.2 .. 30."""
    rng = np.random.default_rng(seed)
    env, bas = list(mol._env), mol._bas.copy()
    for ib, n in enumerate(nprims):
        e = np.exp(rng.uniform(np.log(0.2), np.log(30.0), n))
        c = gto.normalized_coefficients(int(bas[ib, 1]), e, rng.uniform(0.1, 1.0, n))
        bas[ib, 2], bas[ib, 5] = n, len(env)
        env.extend(e.tolist())
        bas[ib, 6] = len(env)
        env.extend(c.tolist())
    mol._bas, mol._env = bas, np.array(env)
    return mol


@pytest.mark.parametrize("dtype", ["fp64", "fp32"])
@pytest.mark.parametrize("heavy,basis", [(1, "6-31g"), (4, "6-31g"), (6, "sto-3g")])
def test_eri_s8_tiles(hip, heavy, basis, dtype):
    """Several bra and ket tiles per class, uneven contractions (1 to 36
    primitives per pair)."""
    from pyscf_ipu_amd.electron_repulsion import direct
    mol = build_mol(molgen.plain_set(1, heavy, seed=11)[0], basis)
    print(f"eri tiles nao={mol.nao_nr()} {dtype}", flush=True)
    _check(direct.eri_s8(mol, dtype).cpu().numpy(), cint.eri_s8(mol), dtype)


@pytest.mark.parametrize("dtype", ["fp64", "fp32"])
@pytest.mark.parametrize("nprims", [(9, 1, 3, 8), (9, 9, 2, 1), (16, 14, 1, 15), (1, 1, 1, 1)])
def test_eri_s8_long_contractions(hip, nprims, dtype):
    """Pairs with more primitives than the 64 lanes of a chunk (81) and than an
    FP64 ket stage holds (256): their pieces add up.  One p shell."""
    from pyscf_ipu_amd.electron_repulsion import direct
    mol = build_mol("O 0 0 0; H 0.9 0.2 0; H -0.3 0.8 0.1")  # shells s, s, p, s, s
    assert mol.nbas == 5
    mol = _contract(mol, nprims[:2] + (nprims[3],) + nprims[2:])
    print(f"eri contractions {nprims} {dtype}", flush=True)
    _check(direct.eri_s8(mol, dtype).cpu().numpy(), cint.eri_s8(mol), dtype)


@pytest.mark.parametrize("dtype", ["fp64", "fp32"])
def test_eri_s8_contractions_beyond_a_stage(hip, dtype):
    """Pairs of 23 x 23 primitives, more than any stage holds on either side
    (and than the oracle takes): against the quartet kernel."""
    from pyscf_ipu_amd.electron_repulsion import direct
    mol = _contract(build_mol("O 0 0 0; H 0.9 0.2 0"), (23, 2, 22, 1))  # s, s, p, s
    assert mol.nbas == 4
    N, loc = mol.nao_nr(), mol.ao_loc_nr()
    q = np.array([(i, j, k, l) for i in range(4) for j in range(4) for k in range(4) for l in range(4)], np.int32)
    flat = direct.eri_quartets(mol, q, "fp64").cpu().numpy()
    s1, at = np.zeros((N, N, N, N)), 0
    for sh in q:
        d = [loc[x + 1] - loc[x] for x in sh]
        n = int(np.prod(d))
        s1[tuple(slice(loc[x], loc[x + 1]) for x in sh)] = flat[at:at + n].reshape(d[::-1]).transpose(3, 2, 1, 0)
        at += n
    i, j = np.tril_indices(N)
    r, c = np.tril_indices(len(i))
    _check(direct.eri_s8(mol, dtype).cpu().numpy(), s1[i, j][:, i, j][r, c], dtype)


@pytest.mark.parametrize("dtype", ["fp64", "fp32"])
def test_eri_s8_far_atoms(hip, dtype):
    """Shell pairs without a kept primitive pair still write their (zero)
    ERIs, and Boys arguments beyond the tables take the asymptote."""
    from pyscf_ipu_amd.electron_repulsion import direct
    mol = build_mol("C 0 0 0; H 0 0 1.1; O 30 0 0; H 0 25 3; H 1 25 3; C 31.2 0 0.1")
    _check(direct.eri_s8(mol, dtype).cpu().numpy(), cint.eri_s8(mol), dtype)


@pytest.mark.parametrize("dtype", ["fp64", "fp32"])
@pytest.mark.parametrize("count", [1, 5, 40])
def test_batch_all_equals_lists_and_oracle(hip, count, dtype):
    """Both tile shapes of the batched form, molecules without p shells among
    them, and the work-list entry on whole and on partial lists, bit for bit."""
    from pyscf_ipu_amd import _lib
    strs = (["H 0 0 0; H 0 0 0.74"] + molgen.batched_set(count, (1, 6), seed=5))[:count]
    b = batch.BatchRKS(batch.parse(strs), dtype=dtype)
    b.setup()
    print(f"batch eri {count} {dtype}", flush=True)
    eri = b.eri.cpu().numpy()
    for m in sorted({0, count // 2, count - 1}):
        mol = build_mol(strs[m])
        N = mol.nao_nr()
        i, j = np.tril_indices(N)
        pm = 1 + (i == j)
        r, c = np.tril_indices(len(i))
        ref = cint.eri_s8(mol) / (pm[r] * pm[c] * (1 + (r == c)))
        o = int(b.desc[m, 11])
        _check(eri[o:o + len(ref)], ref, dtype)
    P, st = device.ptr, device.stream()
    works = [b._work_list(c) for c in b.eri_counts]

    def lists(ws, out):
        arr = (ctypes.c_void_p * 6)(*[w.data_ptr() for w in ws])
        cnt = (ctypes.c_int * 6)(*[w.shape[0] for w in ws])
        _lib.call("pscf_batch_eri_s8_div", b.code, P(b.d_desc), b.M, arr, cnt, P(b.d_atm), P(b.d_bas), P(b.d_env),
                  P(b.d_shell_ao), P(b.d_shl), P(out), st)

    whole, halves = torch.empty_like(b.eri), torch.empty_like(b.eri)
    lists(works, whole)
    # the entries of even position, then the others: single entries, no neighbours to merge
    for k in (0, 1):
        part = [w[k::2].contiguous() for w in works]
        lists(part, halves)
        torch.cuda.synchronize()
    assert torch.equal(whole, b.eri) and torch.equal(halves, b.eri)
