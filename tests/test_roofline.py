"""The ERI operation counts that rooflines are priced with (CPU)."""
import itertools

import numpy as np
import pytest

from pyscf_ipu_amd import batch, gto, molgen, roofline


@pytest.mark.parametrize("basis", ["sto-3g", "6-31g"])
@pytest.mark.parametrize("dtype", ["fp64", "fp32"])
def test_hermite_count_is_the_sum_over_shell_quartets(basis, dtype):
    """Against a plain loop over unique quartets of shell pairs, the pair of the
    higher class (or the earlier of two in one class) holding the lanes."""
    mol = gto.build_mol("O 0 0 0; H 0.9 0.2 0; C 9 0 0.5", basis)
    cut = 1e-20 if dtype == "fp64" else 1e-15
    bas, xyz, pairs = mol._bas, np.asarray(mol.atom_coords()), []
    prims = [list(zip(mol._env[b[5]:b[5] + b[2]], mol._env[b[6]:b[6] + b[2]])) for b in bas]  # as the kernels read them
    for i in range(mol.nbas):
        for j in range(i + 1):
            r2 = ((xyz[bas[i, 0]] - xyz[bas[j, 0]]) ** 2).sum()
            n = sum(abs(ca * cb) * np.exp(-a * b / (a + b) * r2) / (a + b) >= cut
                    for (a, ca), (b, cb) in itertools.product(prims[i], prims[j]))
            pairs.append((int(bas[i, 1] + bas[j, 1]), n))
    ref = 0.0
    for a in range(len(pairs)):
        for b in range(a + 1):
            (X, m), (Y, k) = sorted((pairs[a], pairs[b]), key=lambda t: t[0])
            one, once = roofline.eri_hermite_flops_per_primitive(X, Y, dtype)
            # within one class either pair may hold the lanes: the mean
            ref += one * m * k + once * (k if X != Y else (m + k) / 2)
    assert abs(roofline.eri_hermite_flops(mol, dtype) - ref) < 1e-9 * ref


def test_batch_count_adds_up():
    strs = molgen.batched_set(12, (1, 6), seed=5)
    b = batch.BatchRKS(batch.parse(strs), dtype="fp32")
    ref = sum(roofline.eri_hermite_flops(gto.build_mol(s), "fp32") for s in strs)
    assert abs(roofline.batch_eri_flops(b) - ref) < 1e-9 * ref


def test_counts_per_primitive_quartet():
    """Between the instruction counts of the compiled kernels (33 for (ss|ss) to
    520 for (pp|pp), an FMA being one) and twice them."""
    for X, Y, n in ((0, 0, 33), (2, 2, 520)):
        one, _ = roofline.eri_hermite_flops_per_primitive(X, Y, "fp32")
        assert 0.75 * n < one < 2 * n
