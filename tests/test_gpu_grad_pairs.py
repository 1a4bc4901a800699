"""The gradient's two-electron and one-electron kernels alone (csrc/eri_grad.h,
int1e_grad_kernel) for a random symmetric density, at the sizes where their
tiles, chunks and stages break, against the derivative integrals of the FP64
CPU oracle: 1e-8 of the largest component (at least 1), the bound of the whole
gradient's test (every contribution is rounded to 2^-40)."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import cint
from oracle import grad as oracle_grad
from pyscf_ipu_amd import _lib, device, molgen
from pyscf_ipu_amd.electron_repulsion import direct
from pyscf_ipu_amd.gto import build_mol
from tests.test_gpu_eri_pairs import _contract

pytestmark = pytest.mark.gpu
HYB = 0.2


def _density(mol):
    rng = np.random.default_rng(mol.nao_nr())
    d = rng.standard_normal((mol.nao_nr(),) * 2)
    return 0.5 * (d + d.T) / np.sqrt(mol.nao_nr())


def _gpu_eri(mol, dm, natm=None):
    atm, bas, env = direct._mol_device(mol)
    natm = natm or mol.natm
    if natm > mol.natm:  # atoms without shells
        atm = torch.cat([atm.reshape(mol.natm, -1), atm.reshape(mol.natm, -1)[:1].repeat(natm - mol.natm, 1)]).contiguous()
    pairs, counts = direct.shell_pairs_by_class(mol)
    g = device.zeros((natm, 3), torch.float64)
    dp, dd = device.to_dev(pairs), device.to_dev(dm)
    _lib.call("pscf_grad_eri", device.ptr(atm), natm, device.ptr(bas), mol.nbas, device.ptr(env), device.ptr(dp),
              (ctypes.c_int * 3)(*counts), mol.nao_nr(), device.ptr(dd), HYB, device.ptr(g), device.stream())
    return g.cpu().numpy()


def _oracle_eri(mol, dm):
    ip1 = cint.eri_ip1(mol)
    vj = -np.einsum("sijkl,lk->sij", ip1, dm, optimize=True)
    vk = -np.einsum("sijkl,jk->sil", ip1, dm, optimize=True)
    v = vj - 0.5 * HYB * vk
    return np.array([2.0 * np.einsum("sij,ij->s", v[:, p0:p1], dm[p0:p1]) for p0, p1 in oracle_grad.aoslices(mol)[:, 2:]])


def _check(got, ref):
    assert got.shape == ref.shape
    assert np.abs(got - ref).max() < 1e-8 * max(1.0, np.abs(ref).max()), np.abs(got - ref).max()


@pytest.mark.parametrize("heavy,basis", [(1, "sto-3g"), (2, "6-31g"), (4, "6-31g"), (5, "sto-3g")])
def test_grad_eri_tiles(hip, heavy, basis):
    mol = build_mol(molgen.plain_set(1, heavy, seed=5)[0], basis)
    print(f"grad_eri nao={mol.nao_nr()}", flush=True)
    dm = _density(mol)
    _check(_gpu_eri(mol, dm), _oracle_eri(mol, dm))


@pytest.mark.parametrize("nprims", [(9, 1, 8, 3, 2), (16, 14, 15, 1, 1), (1, 1, 1, 1, 1)])
def test_grad_eri_long_contractions(hip, nprims):
    """Pairs with more primitives than a chunk (64) or an FP64 ket stage (192)."""
    mol = _contract(build_mol("O 0 0 0; H 0.9 0.2 0; H -0.3 0.8 0.1"), nprims)
    print(f"grad_eri contractions {nprims}", flush=True)
    dm = _density(mol)
    _check(_gpu_eri(mol, dm), _oracle_eri(mol, dm))


def test_grad_eri_many_atoms(hip):
    """More atoms than the LDS holds sums for: the same bits."""
    mol = build_mol("O 0 0 0.1; H 0 0.7 -0.4; H 0 -0.7 -0.4")
    dm = _density(mol)
    a, b = _gpu_eri(mol, dm), _gpu_eri(mol, dm, 4096)
    assert np.array_equal(a, b[:mol.natm]) and not b[mol.natm:].any()
