"""FP64 batches reproduce their results to the last bits of the integrals: a
molecule that has not converged within its iterations amplifies a change of one
unit in the last place of an ERI or of V_xc to 1e-9 .. 1e-6 Ha of its gap.

tests/golden/batch_fp64_slow.json holds recorded energies, gaps and iteration
counts of four molecules that do not converge in 20 iterations, two that do so
late and one ordinary one.  Every sum of the path has a fixed order or is exact,
so the results repeat; the tolerance, 1e-10 relative, is a tenth of what FP64
results of this size are compared with."""
import json
import os

import numpy as np
import pytest

from pyscf_ipu_amd import batch

pytestmark = pytest.mark.gpu
GOLDEN = os.path.join(os.path.dirname(__file__), "golden", "batch_fp64_slow.json")


@pytest.mark.parametrize("graph", [True, False])
def test_slow_molecules_reproduce(hip, graph):
    with open(GOLDEN) as f:
        ref = json.load(f)["molecules"]
    mols = [(np.array(m["Z"], np.int32), np.array([[float.fromhex(x) for x in p] for p in m["R"]])) for m in ref]
    r = batch.BatchRKS(mols, dtype="fp64").run(max_its=20, conv_tol=1e-8, graph=graph)
    for k, m in enumerate(ref):
        energy, gap = float.fromhex(m["energy"]), float.fromhex(m["gap"])
        assert r.iterations[k] == m["iterations"], k
        assert abs(r.energy[k] - energy) <= 1e-10 * abs(energy), k
        assert abs(r.hlgap[k] - gap) <= 1e-10 * abs(gap), k
