"""The batch autotuner compares launches that differ (CPU: shapes only)."""
import pytest

from pyscf_ipu_amd import _lib, batch, molgen


@pytest.mark.parametrize("count", [3, 40, 700])
@pytest.mark.parametrize("dtype", ["fp64", "fp32"])
def test_candidates_are_distinct_launches(dtype, count):
    base = batch.parse(molgen.batched_set(20, (1, 9), seed=3))
    b = batch.BatchRKS([base[k % 20] for k in range(count)], dtype=dtype)
    L = _lib.lib()
    shapes = {"xc": [], "jk": []}
    cands = b.tune_candidates()
    for tile, split in cands["xc"]:
        shapes["xc"].append((tile, *(L.pscf_batch_xc_split(b.code, batch.class_split(split, n))
                                     for _, n, _ in b.nao_classes)))
    for threads, split in cands["jk"]:
        shapes["jk"].append((threads, *(L.pscf_batch_jk_split(b.code, n, cmax, int(dtype == "fp32"),
                                                              batch.class_split(split, n), threads)
                                        for _, n, cmax in b.nao_classes)))
    for name in ("xc", "jk"):
        assert cands[name] and len(set(shapes[name])) == len(shapes[name])
        assert all(c[1] in batch.SPLITS for c in cands[name])
    assert {t for t, _ in cands["jk"]} == set(batch.JK_THREADS)


def test_launch_splits():
    """At least four workgroups per molecule where the sums are exact, and no
    more than the column form's 128 row lists have waves for."""
    L = _lib.lib()
    assert [L.pscf_batch_xc_split(_lib.F32, k) for k in (1, 2, 4, 8)] == [4, 4, 4, 8]
    assert [L.pscf_batch_xc_split(_lib.F64, k) for k in (1, 2, 4, 8)] == [1, 2, 4, 8]
    jk = L.pscf_batch_jk_split
    assert [jk(_lib.F32, 1024, 60, 0, k, 256) for k in (1, 8, 64)] == [1, 8, 32]  # atomics that are not exact
    assert [jk(_lib.F32, 1024, 60, 1, k, 256) for k in (1, 8, 64)] == [4, 8, 32]
    assert [jk(_lib.F64, 24, 60, 0, k, 512) for k in (1, 24)] == [16, 16]
    assert [jk(_lib.F64, 24, 80, 0, k, 512) for k in (1, 64)] == [64, 64]
