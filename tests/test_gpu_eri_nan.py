"""An atom whose position is not a number: every ERI of its AOs is not a number,
every other keeps its bits."""
import numpy as np
import pytest

from pyscf_ipu_amd import batch
from pyscf_ipu_amd.gto import build_mol

pytestmark = pytest.mark.gpu
GEOM = "C 0 0 0; H 0 0 1.1; O 1.2 0.3 0; H 1.5 1.1 0.2"


def _touches(mol, atom):
    """Per packed s8 element: whether an AO of `atom` is among its four."""
    on = np.repeat(mol._bas[:, 0], np.diff(mol.ao_loc_nr())) == atom
    i, j = np.tril_indices(mol.nao_nr())
    p = on[i] | on[j]
    r, c = np.tril_indices(len(i))
    return p[r] | p[c]


@pytest.mark.parametrize("dtype", ["fp64", "fp32"])
@pytest.mark.parametrize("atom", [1, 2])
def test_nan_position(hip, atom, dtype):
    from pyscf_ipu_amd.electron_repulsion import direct
    mol = build_mol(GEOM)
    ref = direct.eri_s8(mol, dtype).cpu().numpy()
    mol._env[mol._atm[atom, 1]] = np.nan
    got = direct.eri_s8(mol, dtype).cpu().numpy()
    hit = _touches(mol, atom)
    assert np.isnan(got[hit]).all() and np.array_equal(got[~hit], ref[~hit])


@pytest.mark.parametrize("dtype", ["fp64", "fp32"])
def test_nan_position_in_a_batch(hip, dtype):
    mols = batch.parse([GEOM, GEOM])
    mols[1][1][2, 0] = np.nan
    b = batch.BatchRKS(mols, dtype=dtype)
    b.setup()
    n = int(b.desc[1, 11])
    eri = b.eri.cpu().numpy()
    hit = _touches(build_mol(GEOM), 2)
    assert np.isnan(eri[n:][hit]).all() and np.array_equal(eri[n:][~hit], eri[:n][~hit])
