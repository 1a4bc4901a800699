"""What the framework is timed on: the calls its users make, over the sizes its
own configurations, tests and benchmark use.

Kinds of case (`kind`):

  scf      RKS.run: one molecule, set-up and SCF to |dE| < 1e-8 Ha, at most 20 iterations
  eri      direct.eri_s8: the packed ERIs of one molecule
  jk       sparse_symmetric_einsum: J and K from nonzero ERIs and their indices
  xc       exchange_correlation: E_xc and V_xc from stored AO values
  grad     grad: the nuclear gradient of one molecule
  large    LargeRKS.fock_parts: one Fock build of a 6-31G molecule
  setup    BatchRKS set-up: grid, weights, one-electron integrals and ERIs of many molecules
  batch    BatchRKS: set-up and SCF of many molecules
  train    PairMLP.loss_and_grads + adam: one training step of the learned guess
  predict  PairMLP.forward: the learned guess's network on a batch of atom pairs

`exact` evaluates the same quantities in 64 bits with plain torch: ERIs by the
McMurchie-Davidson scheme, J/K as dense sums, B3LYP by automatic
differentiation, the gradient by differentiating the energy expression.  A
whole SCF has no exact value here: at its energy-change stop it is a point on
the iteration's own path.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from pyscf_ipu_amd import batch, grids, gto, learned_guess, molgen, roofline
from pyscf_ipu_amd.electron_repulsion import direct
from pyscf_ipu_amd.nanoDFT import nanoDFT as nano
from pyscf_ipu_amd.nanoDFT import sparse_symmetric_ERI as sse
from pyscf_ipu_amd.precision import LargeRKS

F64 = torch.float64
HYB = 0.2


def listed():
    return [
        # the smallest call a user makes: the README's methane, where launches and host steps are everything
        {"name": "scf_methane_fp64", "kind": "scf", "heavy": 0, "basis": "sto-3g", "level": 0},
        # the headline workload of the benchmark: one 9-heavy-atom molecule, FP64
        {"name": "scf_9heavy_fp64", "kind": "scf", "heavy": 9, "molecule": 4, "basis": "sto-3g", "level": 0},
        # integrals of one such molecule, as a program that keeps its own SCF loop asks for them
        {"name": "eri_9heavy_fp64",
         "kind": "eri", "heavy": 9, "molecule": 1, "basis": "sto-3g", "dtype": "fp64"},
        # integrals of a molecule of the precision study (6-31G, 12-16 heavy atoms), FP32
        {"name": "eri_12heavy_631g_fp32",
         "kind": "eri", "heavy": 12, "molecule": 1, "basis": "6-31g", "dtype": "fp32"},
        # the reference's own J/K call on one 9-heavy-atom molecule, in its default type
        {"name": "jk_9heavy_fp32",
         "kind": "jk", "heavy": 9, "molecule": 1, "basis": "sto-3g", "dtype": "fp32"},
        # the reference's own XC call, its (4, g, N) AO layout, the finer of the two grids in use
        {"name": "xc_9heavy_level1_fp32",
         "kind": "xc", "heavy": 9, "molecule": 1, "basis": "sto-3g", "level": 1, "dtype": "fp32"},
        # one force evaluation of a structure optimisation (always 6-31G)
        {"name": "grad_4heavy_631g", "kind": "grad", "heavy": 4, "molecule": 1, "basis": "6-31g", "level": 0},
        # one Fock build of the precision study, its FP64 reference variant
        {"name": "large_13heavy_f64",
         "kind": "large", "heavy": 13, "molecule": 1, "level": 1, "gemm": "f64/f64", "eri": "fp64"},
        # set-up of a batch of molecules of uneven size (1-9 heavy atoms), FP32
        {"name": "setup_1to9_fp32_256",
         "kind": "setup", "lo": 1, "hi": 9, "molecule": 1, "count": 256, "dtype": "fp32"},
        # a dataset-generation batch of equal sizes, FP32, set-up to converged energies
        {"name": "batch_9heavy_fp32_1024",
         "kind": "batch", "lo": 9, "hi": 9, "molecule": 1, "count": 1024, "dtype": "fp32"},
        # a small batch in FP64, the form that checks the FP32 one
        {"name": "batch_1to9_fp64_96",
         "kind": "batch", "lo": 1, "hi": 9, "molecule": 1, "count": 96, "dtype": "fp64"},
        # a training step of the learned guess at its training script's usual minibatch
        {"name": "train_16384", "kind": "train", "rows": 16384},
    ]


def draw(rng: random.Random):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["scf", "scf", "eri", "eri", "jk", "xc", "grad", "large", "setup", "setup", "batch", "batch",
                       "train", "predict"])
    dtype = rng.choice(["fp32", "fp64"])
    if kind in ("train", "predict"):
        return {"kind": kind, "rows": log_int(1000, 60000)}
    case = {"kind": kind, "molecule": rng.randint(2, 1000)}  # which generated molecule, or first of several
    if kind in ("setup", "batch"):
        case["lo"], case["hi"] = rng.choice([(1, 9), (9, 9), (3, 7), (5, 9)])
        most = 512 if kind == "setup" else (900 if dtype == "fp32" else 128)
        return {**case, "count": log_int(8, most), "dtype": dtype}
    if kind == "large":
        return {**case, "heavy": rng.randint(10, 14), "level": 1,
                "gemm": rng.choice(["f64/f64", "f32/f32", "f32/f64", "f64/f32"]), "eri": dtype}
    if kind == "jk":
        return {**case, "heavy": rng.randint(1, 10), "basis": "sto-3g", "dtype": dtype}
    if kind == "xc":
        return {**case, "heavy": rng.randint(1, 10), "basis": "sto-3g", "level": rng.choice([0, 1]), "dtype": dtype}
    small = rng.choice([True, False])  # a minimal basis, or 6-31G on fewer atoms
    case["basis"] = "sto-3g" if small else "6-31g"
    if kind == "eri":
        return {**case, "heavy": rng.randint(1, 16 if small else 12), "dtype": dtype}
    most = {"scf": (9, 4), "grad": (7, 4)}[kind][0 if small else 1]
    return {**case, "heavy": rng.randint(1, most), "level": rng.choice([0, 1])}


# ------------------------------------------------------------------ inputs ----
def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _conformer(z, r, rng):
    """Another conformer: turned at random and slightly distorted (Bohr)."""
    q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
    return z, r @ q + rng.normal(0, 0.02, r.shape)


def _mol(case, seed):
    """A conformer of the README's methane (heavy 0) or of a generated molecule."""
    name = gto.METHANE if case["heavy"] == 0 else molgen.plain_set(1, case["heavy"], case["molecule"])[0]
    z, r = _conformer(*batch.parse([name])[0], np.random.default_rng(seed))
    return gto.Mole(list(zip(z.tolist(), r)), case.get("basis", "6-31g"), unit="Bohr")


def _molecules(case, seed):
    """`count` molecules: conformers of up to 48 generated ones (a dataset
    holds several conformers of a molecule)."""
    rng = np.random.default_rng(seed)
    base = batch.parse(molgen.batched_set(min(case["count"], 48), (case["lo"], case["hi"]), case["molecule"]))
    return [_conformer(*base[m % len(base)], rng) for m in range(case["count"])]


def _shells(mol):
    """Shells grouped by (l, number of primitives): centre atom, exponents,
    coefficients and first AO of each."""
    loc, out = mol.ao_loc_nr(), {}
    for ib, (_, l, exps, coefs) in enumerate(mol.shell_arrays()):
        out.setdefault((l, len(exps)), []).append((int(mol._bas[ib, 0]), exps, coefs, int(loc[ib])))
    dev = _device()
    return [(l, torch.tensor([s[0] for s in v], device=dev), torch.tensor(np.array([s[1] for s in v]), device=dev),
             torch.tensor(np.array([s[2] for s in v]), device=dev), torch.tensor([s[3] for s in v], device=dev))
            for (l, _), v in sorted(out.items(), reverse=True)]


def _coords(mol):
    return torch.tensor(mol.atom_coords(), device=_device())


def _aos(mol, xyz, pts):
    """AO values and gradients (4, g, N) at pts; differentiable in xyz."""
    out = [None] * mol.nao_nr()
    for l, atom, ex, co, ao in _shells(mol):
        for s in range(len(atom)):
            d = pts - xyz[atom[s]]
            e = torch.exp(-(d * d).sum(1, keepdim=True) * ex[s]) * co[s]
            f, f1 = e.sum(1), (-2 * e * ex[s]).sum(1)
            if l == 0:
                out[int(ao[s])] = torch.stack([f] + [f1 * d[:, x] for x in range(3)])
            else:
                for a in range(3):
                    out[int(ao[s]) + a] = torch.stack(
                        [f * d[:, a]] + [f1 * d[:, a] * d[:, x] + (f if x == a else 0) for x in range(3)])
    return torch.stack(out, 2)


def _becke(mol, g):
    """Becke's weights of the points of atomic grids, 64 bits."""
    dev = _device()
    pts, owner = torch.tensor(g.coords, device=dev), torch.tensor(g.owner.astype(np.int64), device=dev)
    xyz, adj = _coords(mol), torch.tensor(grids.becke_adjust_table(mol.atom_charges()), device=dev)
    d = torch.stack([(pts - c).norm(dim=1) for c in xyz])
    cell = []
    for i in range(mol.natm):
        p = torch.ones_like(d[0])
        for j in range(mol.natm):
            if i != j:
                m = (d[i] - d[j]) / (xyz[i] - xyz[j]).norm()
                m = m + adj[i, j] * (1 - m * m)
                for _ in range(3):
                    m = 0.5 * m * (3 - m * m)
                p = p * 0.5 * (1 - m)
        cell.append(p)
    cell = torch.stack(cell)
    return pts, torch.tensor(g.vol, device=dev) * cell.gather(0, owner[None])[0] / cell.sum(0)


def _orbitals(mol):
    """(mo_coeff, mo_energy) of an extended Hueckel Hamiltonian: orthonormal
    orbitals of the right shape and energies of the right size."""
    S = _one_electron(mol, _coords(mol))[0].cpu().numpy()
    level = {1: (-0.5, -0.2), 6: (-0.7, -0.4), 7: (-0.9, -0.5), 8: (-1.2, -0.6)}
    h = np.zeros(len(S))
    loc, z, seen = mol.ao_loc_nr(), mol.atom_charges(), set()
    for ib in range(mol.nbas):
        ia, l = int(mol._bas[ib, 0]), int(mol._bas[ib, 1])
        core = l == 0 and z[ia] > 2 and ia not in seen  # the first s shell of a heavy atom is its core
        if l == 0:
            seen.add(ia)
        h[loc[ib]:loc[ib + 1]] = -0.3 * z[ia] ** 2 if core else level[int(z[ia])][l]
    H = 0.875 * S * (h[:, None] + h[None, :])
    H[np.diag_indices(len(h))] = h
    X = np.linalg.inv(np.linalg.cholesky(S))
    e, U = np.linalg.eigh(X @ H @ X.T)
    return X.T @ U, e


def _density(mol):
    C, _ = _orbitals(mol)
    n = mol.nelectron // 2
    return 2 * C[:, :n] @ C[:, :n].T


def _sparse_eri(case, seed):
    """Nonzero unique ERIs over their multiplicity, their AO indices and a
    density.  Values: charges of the AO pairs' overlaps at their midpoints,
    which have the range and the decay of the integrals."""
    mol, dev = _mol(case, seed), _device()
    N = mol.nao_nr()
    xyz = _coords(mol)
    S = _one_electron(mol, xyz)[0]
    atom = torch.tensor(np.repeat(mol._bas[:, 0], np.diff(mol.ao_loc_nr())), device=dev).long()
    i, j = torch.tril_indices(N, N, device=dev)
    gen = torch.Generator(device=dev).manual_seed(seed)
    q = S[i, j] + 0.05 * torch.randn(len(i), generator=gen, dtype=F64, device=dev) * torch.exp(
        -0.3 * (xyz[atom[i]] - xyz[atom[j]]).norm(dim=1) ** 2)
    mid = 0.5 * (xyz[atom[i]] + xyz[atom[j]])
    V = q[:, None] * q[None, :] / torch.sqrt(torch.cdist(mid, mid) ** 2 + 1.2)
    r, c = torch.tril_indices(len(i), len(i), device=dev)
    v = V[r, c]
    keep = v.abs() > 1e-9
    r, c, v = r[keep], c[keep], v[keep]
    rep = (1 + (i[r] == j[r]).long()) * (1 + (i[c] == j[c]).long()) * (1 + (r == c).long())
    idx = torch.stack([i[r], j[r], i[c], j[c]], 1).to(torch.int16)
    dt = torch.float64 if case["dtype"] == "fp64" else torch.float32
    return (v / rep).to(dt), idx, torch.tensor(_density(mol), device=dev).to(dt)


def _xc_inputs(case, seed):
    mol = _mol(case, seed)
    pts, w = _becke(mol, grids.atomic_grids(mol, case["level"]))
    dt = torch.float64 if case["dtype"] == "fp64" else torch.float32
    return (torch.tensor(_density(mol), device=_device()).to(dt), _aos(mol, _coords(mol), pts).to(dt).contiguous(),
            w.to(dt))


def _pair_rows(case, seed):
    """Network inputs of random atom pairs (one-hot elements, radial functions
    of the distance, direction), target blocks and masks."""
    dev, B = _device(), case["rows"]
    gen = torch.Generator(device=dev).manual_seed(seed)
    z = torch.multinomial(torch.tensor([0.6, 0.28, 0.06, 0.06], device=dev), 2 * B, True, generator=gen).reshape(B, 2)
    onsite = torch.rand(B, generator=gen, device=dev) < 0.06
    d = torch.where(onsite, torch.zeros(B, device=dev), 1 + 4 * torch.rand(B, generator=gen, device=dev) ** 0.7)
    z[:, 1] = torch.where(onsite, z[:, 0], z[:, 1])
    u = torch.nn.functional.normalize(torch.randn(B, 3, generator=gen, device=dev), dim=1) * (~onsite)[:, None]
    rbf = torch.exp(-0.5 * ((d[:, None] - torch.linspace(0, 5, 32, device=dev)) / 0.15) ** 2)
    X = torch.zeros(B, learned_guess.NIN_PAD, device=dev)
    X[:, :43] = torch.cat([torch.nn.functional.one_hot(z[:, 0], 4), torch.nn.functional.one_hot(z[:, 1], 4), rbf, u], 1)
    n = torch.tensor([1, 5, 5, 5], device=dev)[z]
    row, col = torch.arange(25, device=dev) // 5, torch.arange(25, device=dev) % 5
    mask = torch.zeros(B, learned_guess.NOUT_PAD, device=dev)
    mask[:, :25] = ((row < n[:, :1]) & (col < n[:, 1:])).float()
    Y = torch.randn(B, learned_guess.NOUT_PAD, generator=gen, device=dev) * torch.exp(-0.6 * d)[:, None] * mask
    return X.to(torch.bfloat16), Y, mask


def _weights(seed):
    """The shipped network, its weights moved a little by the seed."""
    with np.load(learned_guess.DEFAULT_WEIGHTS, allow_pickle=False) as f:
        w = f["params"].astype(np.float32)
    return (w * (1 + 0.01 * np.random.default_rng(seed).normal(size=w.shape))).astype(np.float32)


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind in ("scf", "eri"):
        s["mol"] = _mol(case, seed)
    elif kind == "jk":
        s["eri"], s["idx"], s["dm"] = _sparse_eri(case, seed)
    elif kind == "xc":
        s["dm"], s["ao"], s["w"] = _xc_inputs(case, seed)
    elif kind == "grad":
        mol = s["mol"] = _mol(case, seed)
        pts, w = _becke(mol, grids.atomic_grids(mol, case["level"]))
        s["args"] = (pts.cpu().numpy(), w.cpu().numpy(), *_orbitals(mol))
    elif kind == "large":
        mol = _mol(case, seed)
        s["rks"] = LargeRKS(mol, case["level"], case["gemm"], case["eri"])
        s["rks"].setup(dm0=_density(mol))
    elif kind in ("setup", "batch"):
        s["mols"] = _molecules(case, seed)
    else:
        s["X"], s["Y"], s["mask"] = _pair_rows(case, seed)
        s["model"] = learned_guess.PairMLP(_weights(seed))
        s["nvalid"] = float(s["mask"].sum().item())
    return s


# --------------------------------------------------------------------- run ----
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "scf":
        r = nano.RKS(s["mol"], level=case["level"]).run(its=20, conv_tol=1e-8)
        # orbitals are defined up to sign and rotation: the density they span
        return {"energy": r.energy, "mo_energy": r.mo_energy, "dm": r.dm}
    if kind == "eri":
        return direct.eri_s8(s["mol"], case["dtype"])
    if kind == "jk":
        return sse.sparse_symmetric_einsum(s["eri"], s["idx"], s["dm"])
    if kind == "xc":
        return nano.exchange_correlation(s["dm"], s["ao"], s["w"])
    if kind == "grad":
        return nano.grad(s["mol"], *s["args"])
    if kind == "large":
        r = s["rks"]
        r.fock_parts()
        # FP64 buffers of a build in lower precision carry that precision
        dt = F64 if case["gemm"] == "f64/f64" and case["eri"] == "fp64" else torch.float32
        return {"Vxc": r.Vxc.to(dt), "dJK": r.dJK.to(dt), "exc": r.exc.to(dt)}
    if kind == "setup":
        b = batch.BatchRKS(s["mols"], dtype=case["dtype"])
        b.setup()
        return {"eri": b.eri, "weights": b.w, "S": b.S, "Hcore": b.Hc, "Linv": b.Linv, "dm": b.D}
    if kind == "batch":
        b = batch.BatchRKS(s["mols"], dtype=case["dtype"])
        if case["dtype"] == "fp64":
            r = b.run(max_its=20, conv_tol=1e-8)
            return {"terms": r.terms, "gap": r.hlgap}
        # energies of an FP32 SCF, in the precision they have; the gap is left
        # out: a molecule with two close SCF solutions reaches either one
        r = b.run(max_its=20, conv_tol=1e-6)
        return r.terms.astype(np.float32)
    m = s["model"]
    if kind == "predict":
        return m.forward(s["X"], case["rows"])
    loss = m.loss_and_grads(s["X"], s["Y"], s["mask"], case["rows"], nvalid=s["nvalid"])
    m.adam(1e-3)
    return {"loss": loss, "grads": m.g}


# -------------------------------------------------------------------- work ----
def _xc_work(N, g, es):
    return (4 * N + 1) * g * es + 2 * N * N * es, g * (4 * N * N + 16 * N + 150)


def work(case):
    """Inputs read and outputs written once; operations of the method's dense
    form (Rys quadrature for ERIs, 38 N^3 for an SCF step)."""
    kind = case["kind"]
    es = 8 if case.get("dtype", "fp64") == "fp64" else 4
    if kind in ("train", "predict"):
        B, per = case["rows"], 2 * (43 * 256 + 2 * 256 * 256 + 256 * 25)
        if kind == "predict":
            return {"bytes": B * (64 * 2 + 32 * 4) + 4 * learned_guess.NPARAM, "flops": B * per}
        return {"bytes": B * (64 * 2 + 2 * 32 * 4) + 28 * learned_guess.NPARAM,
                "flops": B * (3 * per - 2 * 43 * 256)}
    if kind in ("setup", "batch"):
        nbytes = flops = 0.0
        its = 12 if kind == "batch" else 0
        sizes = range(case["lo"], case["hi"] + 1)
        for h in sizes:
            mol = _mol({"heavy": h, "molecule": case["molecule"], "basis": "sto-3g"}, 0)
            N, g = mol.nao_nr(), grids.atomic_grids(mol, 0).size
            e = direct.s8_size(N) * es
            nbytes += e * (1 + its) + g * (24 + es) + 4 * N * N * 8
            flops += roofline.eri_s8_flops(mol) + 14 * g * mol.natm ** 2 + its * (38 * N ** 3 + _xc_work(N, g, es)[1])
        k = case["count"] / len(sizes)
        return {"bytes": nbytes * k, "flops": flops * k}
    mol = _mol(case, 0)
    N = mol.nao_nr()
    n8 = direct.s8_size(N)
    if kind == "eri":
        return {"bytes": n8 * es, "flops": roofline.eri_s8_flops(mol)}
    if kind == "jk":
        return {"bytes": n8 * (es + 8) + 2 * N * N * es, "flops": 24 * n8}
    g = grids.atomic_grids(mol, case["level"]).size
    if kind == "xc":
        b, f = _xc_work(N, g, es)
        return {"bytes": b, "flops": f}
    if kind == "grad":
        return {"bytes": g * 32 + 4 * N * N * 8, "flops": 4 * roofline.eri_s8_flops(mol) + g * (4 * N * N + 60 * N)}
    if kind == "large":
        ge = 8 if case["gemm"].startswith("f64") else 4
        b, f = _xc_work(N, g, ge)
        return {"bytes": b + n8 * (8 if case["eri"] == "fp64" else 4), "flops": f + 12 * n8}
    b, f = _xc_work(N, g, 8)
    its = 14  # the benchmark's mean
    return {"bytes": its * n8 * 8, "flops": roofline.eri_s8_flops(mol) + its * (38 * N ** 3 + f)}


# ------------------------------------------------------------ 64-bit values ----
HERM = [(0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1), (2, 0, 0), (1, 1, 0), (1, 0, 1), (0, 2, 0), (0, 1, 1), (0, 0, 2)]
NHERM = (1, 4, 10)


def _pair_classes(mol, xyz):
    """Shell pairs by class: combined exponents, centres, Hermite expansion
    E[pair, primitive, component, Hermite index] and AO indices."""
    sh, out = _shells(mol), []
    dev = _device()
    for x in range(len(sh)):
        for y in range(x, len(sh)):
            la, at, ea, ca, aa = sh[x]
            lb, bt, eb, cb, ab = sh[y]
            i, j = torch.meshgrid(torch.arange(len(at), device=dev), torch.arange(len(bt), device=dev), indexing="ij")
            keep = (i >= j) if x == y else torch.ones_like(i, dtype=torch.bool)
            i, j = i[keep], j[keep]
            A, B = xyz[at[i]][:, None], xyz[bt[j]][:, None]
            ka, kb = ea.shape[1], eb.shape[1]
            a = ea[i][:, :, None].expand(-1, ka, kb).reshape(len(i), -1)
            b = eb[j][:, None, :].expand(-1, ka, kb).reshape(len(i), -1)
            c = (ca[i][:, :, None] * cb[j][:, None, :]).reshape(len(i), -1)
            p = a + b
            P = (a[..., None] * A + b[..., None] * B) / p[..., None]
            K = c * torch.exp(-a * b / p * ((A - B) ** 2).sum(-1))
            u, PA, PB = 0.5 / p, P - A, P - B
            zero = torch.zeros_like(K)
            comps = []
            for s in range(2 * la + 1):
                for t in range(2 * lb + 1):
                    h = {}
                    if la == 0:
                        h[0, 0, 0] = K
                    elif lb == 0:
                        h[0, 0, 0] = K * PA[..., s]
                        h[HERM[1 + s]] = K * u
                    else:
                        e = [tuple(int(v == w) for v in range(3)) for w in (s, t)]
                        h[0, 0, 0] = K * (PA[..., s] * PB[..., t] + (u if s == t else 0))
                        h[e[0]] = K * u * PB[..., t]
                        h[e[1]] = h.get(e[1], 0) * (1 if s == t else 0) + K * u * PA[..., s]
                        h[tuple(m + n for m, n in zip(*e))] = K * u * u
                    comps.append(torch.stack([h.get(q, zero) for q in HERM[:NHERM[la + lb]]], -1))
            ia = torch.stack([aa[i] + s for s in range(2 * la + 1) for _ in range(2 * lb + 1)], 1)
            ib = torch.stack([ab[j] + t for _ in range(2 * la + 1) for t in range(2 * lb + 1)], 1)
            out.append({"p": p, "P": P, "E": torch.stack(comps, 2), "l": la + lb, "ia": ia, "ib": ib, "a": a, "b": b,
                        "K": K, "PA": PA, "PB": PB, "la": la, "lb": lb})
    return out


def _boys(m, T):
    """F_0 .. F_m: the highest from the incomplete gamma function, the others downwards."""
    T = T.clamp(min=1e-13)
    a = torch.full_like(T, m + 0.5)
    F = [torch.special.gammainc(a, T) * math.gamma(m + 0.5) * 0.5 * T ** -(m + 0.5)]
    e = torch.exp(-T)
    for k in range(m, 0, -1):
        F.insert(0, (2 * T * F[0] + e) / (2 * k - 1))
    return F


def _hermite_coulomb(alpha, d, order, pref):
    F = _boys(order, alpha * (d[0] ** 2 + d[1] ** 2 + d[2] ** 2))
    memo = {(0, 0, 0, n): pref * (-2 * alpha) ** n * F[n] for n in range(order + 1)}

    def get(t, n):
        if t + (n,) in memo:
            return memo[t + (n,)]
        x = max(range(3), key=lambda k: t[k])
        lo = tuple(v - (k == x) for k, v in enumerate(t))
        r = d[x] * get(lo, n + 1)
        if lo[x] > 0:
            r = r + lo[x] * get(tuple(v - (k == x) for k, v in enumerate(lo)), n + 1)
        memo[t + (n,)] = r
        return r

    return lambda t: get(t, 0)


def _eri_block(bra, ket, lo, hi):
    """(pairs lo..hi of bra, components, pairs of ket, components) ERIs."""
    p, P, E = bra["p"][lo:hi], bra["P"][lo:hi], bra["E"][lo:hi]
    q, Q, G = ket["p"], ket["P"], ket["E"]
    (n, k), (m, kk) = p.shape, q.shape
    pf, qf = p.reshape(-1, 1), q.reshape(1, -1)
    d = [P[..., x].reshape(-1, 1) - Q[..., x].reshape(1, -1) for x in range(3)]
    R = _hermite_coulomb(pf * qf / (pf + qf), d, bra["l"] + ket["l"],
                         2 * math.pi ** 2.5 / (pf * qf * torch.sqrt(pf + qf)))
    hk = HERM[:NHERM[ket["l"]]]
    sign = torch.tensor([(-1.0) ** sum(h) for h in hk], dtype=F64, device=G.device)
    Gm = (G * sign).permute(0, 1, 3, 2).reshape(m, kk * len(hk), -1)
    out = 0
    for a, h in enumerate(HERM[:NHERM[bra["l"]]]):
        S = torch.stack([R(tuple(u + v for u, v in zip(h, g))) for g in hk], -1)          # (n k, m kk, hk)
        T = torch.bmm(S.reshape(n * k, m, -1).transpose(0, 1).contiguous(), Gm)           # (m, n k, comp)
        out = out + torch.einsum("nkc,mnkd->ncmd", E[..., a], T.reshape(m, n, k, -1))
    return out


def _tri(i, j):
    hi, lo = torch.maximum(i, j), torch.minimum(i, j)
    return hi * (hi + 1) // 2 + lo


def _chunks(bra, ket, most=1 << 22):
    step = max(1, most // (bra["p"].shape[1] * ket["p"].numel()))
    return [(a, min(a + step, len(bra["p"]))) for a in range(0, len(bra["p"]), step)]


def _eri_matrix(mol):
    """(pq|rs) as a symmetric matrix over packed AO pairs."""
    N = mol.nao_nr()
    n = N * (N + 1) // 2
    M = torch.empty(n, n, dtype=F64, device=_device())
    cl = _pair_classes(mol, _coords(mol))
    for x, bra in enumerate(cl):
        for ket in cl[:x + 1]:
            rows, cols = _tri(bra["ia"], bra["ib"]), _tri(ket["ia"], ket["ib"]).reshape(-1)
            for lo, hi in _chunks(bra, ket):
                r = rows[lo:hi].reshape(-1)
                B = _eri_block(bra, ket, lo, hi).reshape(len(r), len(cols))
                M[r[:, None], cols[None, :]] = B
                M[cols[:, None], r[None, :]] = B.T
    return M


def _s8(M):
    r, c = torch.tril_indices(len(M), len(M), device=M.device)
    return M[r, c]


def _overlap_1d(pa, pb, u):
    """S(i, j): one-dimensional overlaps of x^i, x^j over that of two s functions."""
    memo = {(0, 0): torch.ones_like(pa)}

    def S(i, j):
        if i < 0 or j < 0:
            return 0.0
        if (i, j) not in memo:
            if i > 0:
                memo[i, j] = pa * S(i - 1, j) + u * ((i - 1) * S(i - 2, j) + j * S(i - 1, j - 1))
            else:
                memo[i, j] = pb * S(i, j - 1) + u * (j - 1) * S(i, j - 2)
        return memo[i, j]

    return S


def _one_electron(mol, xyz, want_h=False):
    """Overlap and, if asked, H_core = T + V; differentiable in xyz."""
    N = mol.nao_nr()
    S = torch.zeros(N, N, dtype=F64, device=_device())
    H = torch.zeros_like(S)
    z = torch.tensor(mol.atom_charges().astype(np.float64), device=S.device)
    for c in _pair_classes(mol, xyz):
        p, b, rows, cols = c["p"], c["b"], c["ia"].reshape(-1), c["ib"].reshape(-1)
        s = ((math.pi / p) ** 1.5)[..., None] * c["E"][..., 0]
        S = _put(S, rows, cols, s.sum(1))
        if not want_h:
            continue
        # kinetic energy from one-dimensional overlaps
        u = 0.5 / p
        one = [_overlap_1d(c["PA"][..., x], c["PB"][..., x], u) for x in range(3)]
        t = []
        for ca in range(2 * c["la"] + 1):
            for cb in range(2 * c["lb"] + 1):
                i = [int(c["la"] == 1 and ca == x) for x in range(3)]
                j = [int(c["lb"] == 1 and cb == x) for x in range(3)]
                v = 0
                for x in range(3):
                    k = -2 * b * b * one[x](i[x], j[x] + 2) + b * (2 * j[x] + 1) * one[x](i[x], j[x])
                    for y in range(3):
                        if y != x:
                            k = k * one[y](i[y], j[y])
                    v = v + k
                t.append(c["K"] * (math.pi / p) ** 1.5 * v)
        h = torch.stack(t, 2)
        for a in range(mol.natm):
            d = [c["P"][..., x] - xyz[a, x] for x in range(3)]
            R = _hermite_coulomb(p, d, c["l"], 2 * math.pi / p)
            h = h - z[a] * sum(c["E"][..., k] * R(t)[..., None] for k, t in enumerate(HERM[:NHERM[c["l"]]]))
        H = _put(H, rows, cols, h.sum(1))
    return S, H


def _put(M, rows, cols, v):
    v = v.reshape(-1)
    M = M.index_put((rows, cols), v)
    return M.index_put((cols, rows), v)


def _jk(M, D):
    """J - hyb/2 K from the pair matrix, D symmetric."""
    N = len(D)
    ar = torch.arange(N, device=D.device)
    full = _tri(ar[:, None], ar[None, :])
    i, j = torch.tril_indices(N, N, device=D.device)
    J = (M @ (D[i, j] * (2 - (i == j).double())))[full]
    K = torch.stack([torch.einsum("qrs,qr->s", M[full[p]][:, full.reshape(-1)].reshape(N, N, N), D) for p in range(N)])
    return J - 0.5 * HYB * K


def _b3lyp(rho, norms):
    """Per point: energy density over rho, and its derivatives by rho and |grad rho|^2."""
    n = rho.detach().clamp(1e-9, 1e12).requires_grad_(True)
    s = norms.detach().clone().requires_grad_(True)
    slater = -0.75 * (3 / math.pi) ** (1 / 3) * n ** (4 / 3)
    # Becke's gradient correction, spin-compensated (a: one spin's density)
    a = n / 2
    chi = torch.sqrt(s / 4) * a ** (-4 / 3)
    b88 = slater - 2 * 0.0042 * a ** (4 / 3) * chi ** 2 / (1 + 6 * 0.0042 * chi * torch.asinh(chi))
    # VWN, Ceperley-Alder fit, paramagnetic
    A, x0, b, c = 0.0621813817379245 / 2, -0.10498, 3.72744, 12.9352
    x = torch.sqrt((3 / (4 * math.pi * n)) ** (1 / 3))
    X, X0, q = x * x + b * x + c, x0 * x0 + b * x0 + c, math.sqrt(4 * c - b * b)
    at = torch.atan(q / (2 * x + b))
    vwn = n * A * (torch.log(x * x / X) + 2 * b / q * at
                   - b * x0 / X0 * (torch.log((x - x0) ** 2 / X) + 2 * (b + 2 * x0) / q * at))
    # Lee-Yang-Parr, spin-compensated
    a_, b_, c_, d_ = 0.04918, 0.132, 0.2533, 0.349
    r = n ** (-1 / 3)
    P = 1 / (1 + d_ * r)
    delta = r * (c_ + d_ * P)
    cf = 0.3 * (3 * math.pi ** 2) ** (2 / 3)
    lyp = -a_ * (n * P + b_ * torch.exp(-c_ * r) * P * 0.25 * (
        4 * cf * n + s * n ** (-5 / 3) * ((60 - 14 * delta) / 36 - 11 / 6)))
    f = 0.08 * slater + 0.72 * b88 + 0.19 * vwn + 0.81 * lyp
    v, vs = torch.autograd.grad(f.sum(), (n, s))
    return (f / n).detach(), v, vs


def _xc(D, ao, w):
    y = ao[0] @ D
    rho = torch.stack([(y * ao[c]).sum(1) for c in range(4)])
    e, v, vs = _b3lyp(rho[0], 4 * (rho[1:] ** 2).sum(0) + 1e-20)
    coef = torch.cat([0.5 * v[None], 4 * vs * rho[1:]]) * w
    V = ao[0].T @ sum(coef[c][:, None] * ao[c] for c in range(4))
    return (rho[0] * w * e).sum(), V + V.T


def _gradient(mol, pts, w, C, e):
    """Derivative of the energy expression with the orbitals and the grid held fixed."""
    dev = _device()
    n = mol.nelectron // 2
    Co = torch.tensor(np.ascontiguousarray(C[:, :n]), device=dev)
    D = 2 * Co @ Co.T
    W = 2 * (Co * torch.tensor(e[:n], device=dev)) @ Co.T
    xyz = _coords(mol).requires_grad_(True)
    S, H = _one_electron(mol, xyz, True)
    z = torch.tensor(mol.atom_charges().astype(np.float64), device=dev)
    i, j = torch.tril_indices(mol.natm, mol.natm, -1, device=dev)
    ((D * H).sum() - (W * S).sum() + (z[i] * z[j] / (xyz[i] - xyz[j]).norm(dim=1)).sum()).backward()
    pts, w = torch.tensor(pts, device=dev), torch.tensor(w, device=dev)
    for a in range(0, len(w), 4096):
        ao = _aos(mol, xyz, pts[a:a + 4096])
        y = ao[0] @ D
        rho = torch.stack([(y * ao[c]).sum(1) for c in range(4)])
        norms = 4 * (rho[1:] ** 2).sum(0) + 1e-20
        _, v, vs = _b3lyp(rho[0], norms)
        (w[a:a + 4096] * (v * rho[0] + vs * norms)).sum().backward()
    ncl = len(_pair_classes(mol, xyz.detach()))
    for x in range(ncl):
        for y in range(x + 1):
            cl = _pair_classes(mol, xyz.detach())
            for lo, hi in _chunks(cl[x], cl[y], 1 << 21):
                c = _pair_classes(mol, xyz)
                bra, ket = c[x], c[y]
                p, q = bra["ia"][lo:hi, :, None, None], bra["ib"][lo:hi, :, None, None]
                r, s = ket["ia"], ket["ib"]
                gam = D[p, q] * D[r, s] - 0.25 * HYB * (D[p, r] * D[q, s] + D[p, s] * D[q, r])
                # both orders of a pair of different shells count; a pair of one shell holds all its components
                one = [torch.where(bra["ia"][lo:hi, :1] == bra["ib"][lo:hi, :1], 1.0, 2.0),
                       torch.where(ket["ia"][:, :1] == ket["ib"][:, :1], 1.0, 2.0)]
                gam = gam * one[0][:, :, None, None] * one[1]
                (0.5 * (1 if x == y else 2) * (gam * _eri_block(bra, ket, lo, hi)).sum()).backward()
    return xyz.grad


def _network(case, seed):
    X, Y, mask = _pair_rows(case, seed)
    w = torch.tensor(_weights(seed), device=X.device).double().requires_grad_(True)
    h = X.double()
    off = 0
    for k, (rows, cols) in enumerate([(learned_guess.NIN_PAD, 256), (256, 256), (256, 256),
                                      (256, learned_guess.NOUT_PAD)]):
        Wk = w[off:off + rows * cols].reshape(rows, cols)
        off += rows * cols
        if k == 0:  # the padded inputs take no part
            Wk = torch.cat([Wk[:43], Wk[43:].detach() * 0])
        h = h @ Wk + w[off:off + cols]
        off += cols
        if k < 3:
            h = torch.nn.functional.silu(h)
    if case["kind"] == "predict":
        return h.detach()
    loss = ((h - Y.double()) ** 2 * mask.double()).sum() / mask.double().sum()
    g, = torch.autograd.grad(loss, w)
    return {"loss": loss.detach().reshape(1), "grads": g}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("train", "predict"):
        return _network(case, seed)
    if kind == "eri":
        return _s8(_eri_matrix(_mol(case, seed)))
    if kind == "jk":
        v, idx, D = _sparse_eri(case, seed)
        v, D = v.double(), D.double()
        N = len(D)
        i, j, k, l = idx.long().unbind(1)
        J, K = torch.zeros(N * N, dtype=F64, device=v.device), torch.zeros(N * N, dtype=F64, device=v.device)
        for a, b, c, d in ((i, j, k, l), (j, i, k, l), (i, j, l, k), (j, i, l, k),
                           (k, l, i, j), (l, k, i, j), (k, l, j, i), (l, k, j, i)):
            J.index_add_(0, c * N + d, v * D[a, b])
            K.index_add_(0, a * N + d, v * D[b, c])
        return J - 0.5 * HYB * K
    if kind == "xc":
        D, ao, w = _xc_inputs(case, seed)
        return _xc(D.double(), ao.double(), w.double())
    if kind == "grad":
        s = prepare(case, seed)
        return _gradient(s["mol"], *s["args"])
    if kind == "large":
        mol = _mol(case, seed)
        D = torch.tensor(_density(mol), device=_device())
        pts, w = _becke(mol, grids.atomic_grids(mol, case["level"]))
        exc, V = _xc(D, _aos(mol, _coords(mol), pts), w)
        return {"Vxc": V, "dJK": _jk(_eri_matrix(mol), D), "exc": exc.reshape(1)}
    if kind == "setup" and case["count"] <= 256:
        out = {"eri": [], "weights": [], "S": [], "Hcore": [], "Linv": []}
        for z, r in _molecules(case, seed):
            mol = gto.Mole(list(zip(z.tolist(), r)), "sto-3g", unit="Bohr")
            N = mol.nao_nr()
            i, j = torch.tril_indices(N, N, device=_device())
            M = _eri_matrix(mol) / torch.outer(1 + (i == j).double(), 1 + (i == j).double())
            M.diagonal().mul_(0.5)
            S, H = _one_electron(mol, _coords(mol), True)
            out["eri"].append(_s8(M))
            out["weights"].append(_becke(mol, grids.atomic_grids(mol, 0))[1])
            out["S"].append(S.reshape(-1))
            out["Hcore"].append(H.reshape(-1))
            out["Linv"].append(torch.linalg.inv(torch.linalg.cholesky(S)).reshape(-1))
        return {**{k: torch.cat(v) for k, v in out.items()}, "dm": None}
    return None
