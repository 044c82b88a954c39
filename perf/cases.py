"""The work a user of this framework has it do, as cases that can be timed.

`listed()` gives the cases, `draw(rng)` more of the same ranges, `prepare` makes what a program has in hand before
the call, `run` is one pass through the public entry points, `work` the bytes and operations a pass cannot do
without, `tolerance` how far another correct implementation may be from this one.

A case names a path:

  predict    energies (and forces) of molecules resident on the device: `model.energies_and_forces`
  autograd   `model.forward` and `torch.autograd.grad`, the route of a program that differentiates the energy itself
  operators  the same with `fused=False`: the sequence of the registered operators that a saved model file calls
  lists      `model.predict` from host lists of per-molecule arrays: formatting, upload and prediction
  train      `model.build_Z_components` from host lists: Z^T Z and Z^T y over a training set with energies and forces
  solve      `ops.cholesky_solve_spd`: the regularised normal equations

and the molecules: `atoms_min` = `atoms_max` is one composition in displaced copies (a trajectory), otherwise the
atom counts are uniform between the two (a set of different molecules, zero-padded to the largest).  `cell` puts
them into periodic boxes.
"""
import math

import numpy as np
import torch

from qml_lightning_amd import ops
from qml_lightning_amd.models.hadamard_features import HadamardFeaturesModel
from qml_lightning_amd.models.random_features import RandomFourrierFeaturesModel
from qml_lightning_amd.representations.FCHL import FCHLCuda

SPECIES = {2: [1, 6], 3: [1, 6, 8], 4: [1, 6, 7, 8], 5: [1, 6, 7, 8, 9]}
HEAVY = {2: ([6], [1.0]), 3: ([6, 8], [0.7, 0.3]), 4: ([6, 7, 8], [0.72, 0.13, 0.15]),
         5: ([6, 7, 8, 9], [0.7, 0.12, 0.15, 0.03])}
NRS2, NRS3 = 24, 20                    # radial bins of the representation's defaults
ATOM_FEATURES = 4096 * 21 * 16384      # atoms x features of the largest listed SORF prediction


def _case(path, features, molecules, atoms, species, npcas, nstacks, ntransforms=1, forces=True, cell=False):
    return {"path": path, "features": features, "molecules": molecules, "atoms_min": atoms[0], "atoms_max": atoms[1],
            "species": species, "npcas": npcas, "nstacks": nstacks, "ntransforms": ntransforms, "forces": forces,
            "cell": cell}


def listed():
    return [
        # one C9H8O4-sized molecule: every step of a molecular dynamics run or a geometry optimisation
        dict(_case("predict", "sorf", 1, (21, 21), 3, 128, 128), name="one molecule"),
        # a hundred C6H6-sized molecules under a small model, differentiated by the caller
        dict(_case("autograd", "sorf", 100, (12, 12), 2, 64, 8), name="small batch, autograd"),
        # 4096 C9H8O4-sized molecules, 16384 features: the throughput of a trajectory
        dict(_case("predict", "sorf", 4096, (21, 21), 3, 128, 128), name="trajectory"),
        # screening: 8192 different molecules of 3 to 29 atoms, energies only
        dict(_case("predict", "sorf", 8192, (3, 29), 5, 128, 64, forces=False), name="screening energies"),
        # a wider model: 27 atoms, four elements, 256 components, 32768 features
        dict(_case("predict", "sorf", 1548, (27, 27), 4, 256, 128), name="wide model"),
        # random Fourier features at 32768 features
        dict(_case("predict", "rff", 4096, (21, 21), 3, 128, 256), name="fourier features"),
        # a saved model's operator sequence at the model class's default sizes, two transforms, different molecules
        dict(_case("operators", "sorf", 512, (3, 29), 4, 128, 32, ntransforms=2), name="operator sequence"),
        # a test set handed over as host lists, the model class's default sizes
        dict(_case("lists", "sorf", 2048, (3, 29), 4, 128, 32, ntransforms=2), name="test set from lists"),
        # snapshots of a periodic box: many neighbours per atom, few atoms
        dict(_case("predict", "sorf", 16, (96, 96), 3, 128, 64, cell=True), name="periodic boxes"),
        # the normal equations of 1000 C9H8O4-sized molecules with forces, 16384 features
        dict(_case("train", "sorf", 1000, (21, 21), 3, 128, 128), name="training set"),
        # a small training set of different molecules, random Fourier features
        dict(_case("train", "rff", 200, (3, 29), 4, 128, 64), name="small training set, fourier"),
        # the regression coefficients of a 16384-feature model
        {"path": "solve", "features": "sorf", "npcas": 128, "nstacks": 128, "name": "solve"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["predict", "predict", "predict", "autograd", "operators", "lists", "train", "solve"])
    npcas = rng.choice([64, 128, 128, 256])
    if path == "solve":
        nf = _log(rng, 512, 16384)
        npcas = rng.choice([64, 128])
        return {"path": path, "features": "sorf", "npcas": npcas, "nstacks": max(4, nf // npcas)}
    features = rng.choice(["sorf", "sorf", "rff"]) if path in ("predict", "autograd", "train") else "sorf"
    if features == "rff":
        npcas = rng.choice([64, 128])
    species = rng.choice([3, 4, 5] if npcas == 256 else [2, 3, 4, 5])     # two elements give 168 representation entries
    cell = path == "predict" and rng.random() < 0.25
    if cell:
        atoms = (_log(rng, 32, 128),) * 2
    elif rng.random() < 0.5:
        atoms = (rng.randint(6, 29),) * 2
    else:
        atoms = (3, rng.randint(12, 29))
    nstacks = _log(rng, 8, 128)
    ntransforms = rng.choice([1, 2]) if features == "sorf" else 1
    forces = True if path in ("autograd", "train") else rng.random() < 0.8
    hi = {"predict": 4096, "autograd": 1024, "operators": 768, "lists": 4096, "train": 600}[path]
    if cell:
        hi = 48
    molecules = _log(rng, 16 if path == "train" else 1, hi)
    case = _case(path, features, molecules, atoms, species, npcas, nstacks, ntransforms, forces, cell)
    # no dearer than the largest listed case of the path
    if path == "train":
        while _training_rows(case) * _features(case) ** 2 > 64000 * 8192 ** 2:
            case["molecules"] = max(16, case["molecules"] // 2)
            case["nstacks"] = max(8, case["nstacks"] // 2)
    else:
        most = ATOM_FEATURES // (8 if path == "operators" else 2 if features == "sorf" else 1)
        while case["molecules"] * case["atoms_max"] * _features(case) > most:
            case["molecules"] = max(1, case["molecules"] // 2)
    return case


# ---- molecules ------------------------------------------------------------------------------------------
def _geometries(rng, nmol, n, spacing, sites_per_edge, jitter, compact):
    """[nmol, n, 3]: n sites of a cubic grid, each displaced by at most `jitter` per component; taken at random, or
    from the middle outwards with some disorder (`compact`: the first k of them are a compact molecule too)."""
    m = sites_per_edge
    grid = np.stack(np.unravel_index(np.arange(m ** 3), (m, m, m)), 1).astype(np.float64)
    order = rng.random((nmol, m ** 3), dtype=np.float32)
    if compact:
        order += np.linalg.norm(grid - (m - 1) / 2.0, axis=1).astype(np.float32)
    sites = np.argsort(order, axis=1)[:, :n]
    return (grid[sites] + 0.5) * spacing + rng.uniform(-jitter, jitter, (nmol, n, 3))


def _molecules(case, seed):
    """Zero-padded coordinates [B,n,3] and charges [B,n], the atom counts [B], and the boxes [B,3,3] or None."""
    rng = np.random.default_rng(seed)
    B, lo, n, species = case["molecules"], case["atoms_min"], case["atoms_max"], case["species"]
    heavy, share = HEAVY[species]
    cells = None
    edge = int(math.ceil((2.0 * n) ** (1.0 / 3.0)))
    if case["cell"]:
        m = int(math.ceil((1.2 * n) ** (1.0 / 3.0)))
        X = _geometries(rng, B, n, 2.0, m, 0.4, False)
        cells = np.broadcast_to(np.eye(3) * 2.0 * m, (B, 3, 3)).copy()
    elif lo == n:
        base = _geometries(rng, 1, n, 1.75, edge, 0.3, True)
        X = base + rng.normal(0.0, 0.05, (B, n, 3))
    else:
        X = _geometries(rng, B, n, 1.75, edge, 0.3, True)
    counts = np.full(B, n) if lo == n else rng.integers(lo, n + 1, B)
    nheavy = np.maximum(1, np.ceil(counts / 2.2).astype(np.int64))
    kinds = rng.choice(heavy, (1 if lo == n else B, n), p=share)
    place = np.arange(n)[None, :]
    Q = np.where(place < nheavy[:, None], kinds, 1)
    Q = np.where(place < counts[:, None], Q, 0)
    X = np.where((place < counts[:, None])[:, :, None], X, 0.0)
    return X, Q.astype(np.int64), counts, cells


# ---- models ---------------------------------------------------------------------------------------------
def _model(case, seed):
    """A model with random weights: orthonormal projections, its own diagonals / random directions, normal alpha."""
    np.random.seed(seed % (1 << 31))
    elements = np.array(SPECIES[case["species"]])
    rep = FCHLCuda(species=elements)
    if case["features"] == "rff":
        m = RandomFourrierFeaturesModel(rep=rep, elements=elements, sigma=2.0, llambda=1e-5, npcas=case["npcas"],
                                        nstacks=case["nstacks"], nbatch_train=500)
    else:
        m = HadamardFeaturesModel(rep=rep, elements=elements, ntransforms=case["ntransforms"], sigma=2.0, llambda=1e-5,
                                  npcas=case["npcas"], nstacks=case["nstacks"], nbatch_train=500,
                                  fused=case["path"] != "operators")
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    R = rep.get_repsize()
    q, _ = torch.linalg.qr(torch.randn(len(elements), R, case["npcas"], device="cuda", dtype=torch.float64, generator=gen))
    m.reductors = q.float().contiguous()
    m.alpha = torch.randn(m.nfeatures(), device="cuda", dtype=torch.float64, generator=gen)
    m.is_trained = True
    return m


def prepare(case, seed):
    if case["path"] == "solve":
        F = _features(case)
        gen = torch.Generator(device="cuda")
        gen.manual_seed(seed)
        Z = torch.cos(6.3 * torch.rand(F + F // 2, F, device="cuda", dtype=torch.float64, generator=gen))
        A = Z.T @ Z
        A.diagonal().add_(1.0)
        b = Z.T @ torch.randn(Z.shape[0], 1, device="cuda", dtype=torch.float64, generator=gen)
        return {"path": "solve", "A": A, "b": b}
    model = _model(case, seed)
    X, Q, counts, cells = _molecules(case, seed)
    state = {"path": case["path"], "model": model, "forces": case["forces"]}
    if case["path"] in ("lists", "train"):
        state["X"] = [x[:k].copy() for x, k in zip(X, counts)]
        state["Q"] = [q[:k].copy() for q, k in zip(Q, counts)]
        state["n"] = int(counts.max())
        if case["path"] == "train":
            rng = np.random.default_rng(seed + 1)
            state["E"] = rng.normal(size=len(counts))
            state["F"] = [rng.normal(size=(k, 3)) for k in counts]
        return state
    boxes = {} if cells is None else {"cells": cells, "inv_cells": np.linalg.inv(cells)}
    data = model.format_data(X, Q, **boxes)
    state["args"] = [data[k] for k in ("coordinates", "charges", "atomIDs", "molIDs", "natom_counts", "cells", "inv_cells")]
    return state


def run(state):
    path = state["path"]
    if path == "solve":
        x, info = ops.cholesky_solve_spd(state["A"], state["b"])
        return {"x": x, "info": info}
    model = state["model"]
    if path == "lists":
        out = model.predict(state["X"], state["Q"], state["n"], forces=state["forces"])
        return {"energies": out[0], "forces": out[1]} if state["forces"] else {"energies": out}
    if path == "train":
        ztz, zty = model.build_Z_components(state["X"], state["Q"], E=state["E"], F=state["F"], print_info=False)
        return {"ztz": ztz, "zty": zty}
    X, rest = state["args"][0], state["args"][1:]
    if path == "predict":
        energies, forces = model.energies_and_forces(X, *rest, forces=state["forces"])
        return {"energies": energies, "forces": forces}
    if not state["forces"]:
        with torch.no_grad():
            return {"energies": model.forward(X, *rest)}
    X = X.detach().requires_grad_(True)
    energies = model.forward(X, *rest)
    forces, = torch.autograd.grad(-energies.sum(), X)
    return {"energies": energies.detach(), "forces": forces}


# ---- what a pass cannot do without ----------------------------------------------------------------------
def _features(case):
    return case["npcas"] * case["nstacks"]


def _mean_atoms(case):
    """Mean atom count and mean squared atom count of a molecule."""
    k = np.arange(case["atoms_min"], case["atoms_max"] + 1, dtype=np.float64)
    return float(k.mean()), float((k * k).mean())


def _training_rows(case):
    return case["molecules"] * (1.0 + 3.0 * _mean_atoms(case)[0])


def work(case):
    F, d = _features(case), case["npcas"]
    if case["path"] == "solve":
        return {"bytes": 8.0 * (F * F / 2.0 + 2.0 * F), "flops": F ** 3 / 3.0 + 2.0 * F * F}
    B, species, T = case["molecules"], case["species"], case["ntransforms"]
    R = species * NRS2 + species * (species + 1) * NRS3
    n1, n2 = _mean_atoms(case)
    A, both = B * n1, 2.0 if case["forces"] else 1.0
    nn = max(n1 - 1.0, 0.0)
    grad = 4.0 if case["forces"] else 1.0
    # per neighbour and radial bin, and per triple and radial bin: the exponential and its weighting
    rep = A * (nn * NRS2 * 4.0 + nn * (nn - 1.0) / 2.0 * NRS3 * 6.0) * both
    constants = 4.0 * species * (R * d + (d * F + F if case["features"] == "rff" else (T + 1) * F)) + 8.0 * F
    inputs = 4.0 * 4.0 * A
    if case["path"] == "train":
        M = _training_rows(case)
        per_row = 2.0 * d * F if case["features"] == "rff" else T * math.log2(d) * F
        rows = (A + 3.0 * B * n2) * (2.0 * R * d + per_row)
        return {"bytes": constants + 8.0 * (4.0 * A + B) + 8.0 * (F * F + F), "flops": rep + rows + M * F * (F + 1.0) + 2.0 * M * F}
    if case["features"] == "rff":
        per_atom = both * (2.0 * R * d + 2.0 * d * F) + 6.0 * F
    else:
        per_atom = both * (2.0 * R * d + T * math.log2(d) * F) + 6.0 * F
    return {"bytes": constants + inputs + 4.0 * B + (4.0 * 3.0 * A if grad > 1.0 else 0.0), "flops": rep + A * per_atom}


def tolerance(case):
    # the factorisation is fp64 throughout, of a matrix whose condition number is about 1e2 to 1e3; everything else
    # has fp32 representations, coefficients and sums in it (Z^T Z and Z^T y are fp64 sums of such rows)
    if case["path"] == "solve":
        return {"rel": 1e-10, "max": 1e-8}
    return {"rel": 1e-5, "max": 4e-4}
