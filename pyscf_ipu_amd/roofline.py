"""Algorithmic work per launch of each kernel group (frozen models for rooflines).

eri_s8   FP VALU-bound.  FLOPs of the Hermite (McMurchie-Davidson) form that the
         shell-pair engine runs (csrc/eri_pairs.h), on the primitive pairs it
         keeps: per primitive quartet the Boys values, the Hermite Coulomb
         integrals and the bra expansion, per bra pair and ket primitive the
         horizontal step, the ket expansion and the sum over primitives.
         eri_s8_flops counts the Rys form's operations instead (libcint's
         quadrature, all primitives), the size of the problem whatever the
         method: F = 40 (ket pair + prefactor) + 2*(TAYLOR+1) + 4*(2R-1) + 1 (Boys)
           + ROOTS[R] (Rys roots from moments)
           + R * (10 + 3*(8 + 5*(n+1)(m+1) + 3*prod(l+1)) + 4*nc)
         per primitive quartet (per root: B coefficients, per axis C coefficients +
         2D recurrence over (n, m) = (li+lj, lk+ll) + horizontal transfer, then 4
         flops per output component for w*Ix*Iy*Iz), R = (li+lj+lk+ll)/2 + 1.
jk_s8    HBM-bound.  Bytes = (#unique s8 ERIs) * sizeof(dtype): each ERI is read
         once; dm and the J/K accumulator live in LDS, indices are regenerated.
xc       HBM-bound.  Bytes = 4 g N sizeof(dtype) (AO values + gradients) +
         g sizeof(dtype) (weights).
scf_step FP64, latency-bound.  FLOPs = 38 N^3 (DIIS products 6N^3, L H L^T 4N^3,
         warm-start transform 4N^3, three Jacobi sweeps 18N^3, C and D 4N^3,
         extrapolation and errors 2N^3).
"""
from __future__ import annotations

import numpy as np

TAYLOR = 8
ROOTS = {1: 1, 2: 25, 3: 120}


def eri_flops_per_primitive(li, lj, lk, ll) -> int:
    R = (li + lj + lk + ll) // 2 + 1
    n, m = li + lj, lk + ll
    nc = (2 * li + 1) * (2 * lj + 1) * (2 * lk + 1) * (2 * ll + 1)
    per_root = 10 + 3 * (8 + 5 * (n + 1) * (m + 1) + 3 * (li + 1) * (lj + 1) * (lk + 1) * (ll + 1)) + 4 * nc
    return 40 + 2 * (TAYLOR + 1) + 4 * (2 * R - 1) + 1 + ROOTS[R] + R * per_root


def eri_s8_flops(mol) -> float:
    """FLOPs of all unique shell quartets of a molecule in the Rys form."""
    return _eri_flops_shells(mol._bas[:, 1].astype(int), mol._bas[:, 2].astype(int))


def _eri_flops_shells(l, npr) -> float:
    pairs = [(i, j) for i in range(len(l)) for j in range(i + 1)]
    # aggregate pairs by (l_a, l_b sorted, nprim product)
    from collections import Counter
    pc = Counter()
    for i, j in pairs:
        la, lb = max(l[i], l[j]), min(l[i], l[j])
        pc[(la, lb, npr[i] * npr[j])] += 1
    keys = list(pc)
    tot = 0.0
    for a in range(len(keys)):
        for b in range(a + 1):
            ka, kb = keys[a], keys[b]
            cnt = pc[ka] * pc[kb] if a != b else pc[ka] * (pc[ka] + 1) // 2
            bra, ket = (ka, kb) if ka[0] + ka[1] >= kb[0] + kb[1] else (kb, ka)
            f = eri_flops_per_primitive(bra[0], bra[1], ket[0], ket[1])
            tot += cnt * ka[2] * kb[2] * f
    return tot


def _hermite_orders(L):
    return [(t, u, s - t - u) for s in range(L + 1) for t in range(s, -1, -1) for u in range(s - t, -1, -1)]


def eri_hermite_flops_per_primitive(X: int, Y: int, dtype: str) -> tuple:
    """(FLOPs per primitive quartet, FLOPs per bra pair and ket primitive) of the
    class (X|Y), X <= Y the numbers of p shells in a pair (an FMA is two)."""
    L, H = X + Y, (Y + 1) * (Y + 2) * (Y + 3) // 6
    n = 3 + 1 + 1 + 3 + 1 + 6                                        # centres, p + q, 1 / sqrt, alpha, prefactor, t
    n += 10 if dtype == "fp32" else 24                               # F_L from the table
    n += (3 if dtype == "fp32" else 20) + 3 * L if L else 0          # exp(-t), downward recursion
    n += (L + 1) + 2 * L                                             # (-2 alpha)^n F_n
    for t in _hermite_orders(L):                                     # R_tuv
        if sum(t):
            n += (3 if max(t) >= 2 else 1) * (L - sum(t) + 1)
    n += {0: H, 1: 3 + 12 * H, 2: 15 + 54 * H}[X]                    # bra expansion into the accumulators
    nb, nk = (1, 3, 9)[X], (1, 3, 9)[Y]
    once = (18 * H if X == 2 else 0) + nb * {0: 1, 1: 12, 2: 99}[Y]  # horizontal step, ket expansion
    return n, once + nb * nk                                         # and the sum over the ket's primitives


def _hermite_shells(bas, atm, env, dtype: str) -> float:
    """FLOPs of one molecule's packed ERIs in the Hermite form."""
    bas = bas.astype(int)
    l, centres = bas[:, 1], env[atm[bas[:, 0], 1].astype(int)[:, None] + np.arange(3)]
    exps, coefs = ([env[b[q]:b[q] + b[2]] for b in bas] for q in (5, 6))
    cut = 1e-20 if dtype == "fp64" else 1e-15                        # EpCut of csrc/eri_pairs.h
    i, j = np.tril_indices(len(l))
    k = max(len(e) for e in exps)
    a = np.ones((len(l), k))
    c = np.zeros((len(l), k))
    for s, (e, f) in enumerate(zip(exps, coefs)):
        a[s, :len(e)], c[s, :len(f)] = e, f
    r2 = ((centres[i] - centres[j]) ** 2).sum(1)[:, None, None]
    p = a[i][:, :, None] + a[j][:, None, :]
    pre = np.abs(c[i][:, :, None] * c[j][:, None, :]) * np.exp(-a[i][:, :, None] * a[j][:, None, :] / p * r2) / p
    kept = ((pre >= cut) & (c[i][:, :, None] * c[j][:, None, :] != 0)).sum((1, 2))
    cls = l[i] + l[j]
    tot = 0.0
    for Y in range(3):
        for X in range(Y + 1):
            one, once = eri_hermite_flops_per_primitive(X, Y, dtype)
            b, m = kept[cls == X].astype(float), kept[cls == Y].astype(float)
            if X == Y:
                tot += one * (b.sum() ** 2 + (b * b).sum()) / 2 + once * (len(b) + 1) * b.sum() / 2
            else:
                tot += one * b.sum() * m.sum() + once * len(b) * m.sum()
    return tot


def eri_hermite_flops(mol, dtype: str) -> float:
    """FLOPs of one pscf_eri_s8 call."""
    return _hermite_shells(mol._bas, mol._atm, np.asarray(mol._env), dtype)


def batch_eri_flops(b) -> float:
    """FLOPs of pscf_batch_eri_s8_all in FP32 over every molecule of a BatchRKS."""
    return float(sum(_hermite_shells(b.bas[d[5]:d[5] + d[1]], b.atm, b.env, "fp32") for d in b.desc))


def per_launch_work(kernel: str, mols, dtype: str) -> dict:
    es = 8 if dtype == "fp64" else 4
    if kernel == "eri_s8":
        f = float(np.mean([eri_hermite_flops(m, dtype) for m in mols]))
        return {"bound": "valu", "flops": f, "model": "Hermite ERI op-count model (pyscf_ipu_amd/roofline.py), "
                                                     "FP VALU; peak = MI355X FP64/FP32 vector rate"}
    if kernel == "jk_s8":
        b = float(np.mean([(m.nao_nr() * (m.nao_nr() + 1) // 2) * (m.nao_nr() * (m.nao_nr() + 1) // 2 + 1) // 2
                           for m in mols])) * es
        return {"bound": "hbm", "bytes": b, "model": "sizeof(dtype) per unique s8 ERI"}
    if kernel == "xc":
        from pyscf_ipu_amd import grids
        b = float(np.mean([(4 * m.nao_nr() + 1) * grids.atomic_grids(m, 0).size for m in mols])) * es
        return {"bound": "hbm", "bytes": b, "model": "4 g N + g elements (AO values/gradients, weights)"}
    if kernel == "scf_step":
        f = float(np.mean([38.0 * m.nao_nr() ** 3 for m in mols]))
        # FP64 arithmetic (MFMA products plus VALU rotations) whose peak is the
        # MI355X FP64 rate; what limits it is latency: one workgroup per molecule
        return {"bound": "mfma", "flops": f, "model": "38 N^3 FP64",
                "limiter": "latency: one workgroup (one CU) per molecule; its eigen-decomposition is a chain of "
                            "dependent reflector, bisection or refinement steps"}
    raise KeyError(kernel)
