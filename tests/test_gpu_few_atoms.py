"""Few atoms: the representation with its projection and the two backward are one launch each (64 or 128 components; up to 256 atoms
with 768 or 512 entries of the representation, 768 with half as many, 1536 with a quarter).  Energies and forces against the same model by the separate operators, which never take those
launches, at the edges of what does and where it no longer is taken; each case says which of the two it is.  Both are fp32 sums in another order: 2-norm errors against
fp64 are 5e-7 on either route, a fiftieth of the tolerance."""
import numpy as np
import pytest
import torch

from qml_lightning_amd import _lib, ops
from qml_lightning_amd.models.hadamard_features import HadamardFeaturesModel
from qml_lightning_amd.models.random_features import RandomFourrierFeaturesModel
from qml_lightning_amd.representations.FCHL import FCHLCuda
from tests import helpers
from tests.test_gpu_kernels import make_batch

pytestmark = pytest.mark.gpu
REL = 2.5e-5


def models(species, elements, npcas, nstacks, rff=False, **grids):
    out = []
    for separate in (False, True):
        np.random.seed(4)
        common = dict(rep=FCHLCuda(species=np.array(species), **grids), elements=np.array(elements), npcas=npcas, nstacks=nstacks,
                      separate_ops=separate)
        m = RandomFourrierFeaturesModel(sigma=1.0, **common) if rff else HadamardFeaturesModel(sigma=2.0, ntransforms=1, **common)
        gen = torch.Generator(device="cuda")
        gen.manual_seed(9)
        R = m.rep.get_repsize()
        m.reductors = torch.randn(len(elements), R, npcas, device="cuda", generator=gen) / R ** 0.5
        m.alpha = torch.randn(m.nfeatures(), device="cuda", dtype=torch.float64, generator=gen)
        m.is_trained = True
        out.append(m)
    return out


def check(species, elements, npcas, coords, charges, taken, nstacks=8, edge=None, **grids):
    one, other = models(species, elements, npcas, nstacks, **grids)
    X, Z, _, _, _ = make_batch(coords, charges)
    rep = one.rep
    prm = ops.make_params(rep.nspecies, rep.Rs2, rep.Rs3, rep.eta2, rep.eta3, rep.two_body_decay, rep.three_body_weight, rep.three_body_decay,
                          rep.rcut)
    assert _lib.lib().qmll_fchl19_projected_pays(sum(len(q) for q in charges), X.shape[1], prm, npcas) == taken
    assert one.reductors.data_ptr() % 16 == 0
    boxes = {} if edge is None else {"cells": np.tile(np.eye(3) * edge, (len(coords), 1, 1)), "inv_cells": np.tile(np.eye(3) / edge, (len(coords), 1, 1))}
    data = one.format_data(X, Z.astype(np.int64), **boxes)
    args = [data[k] for k in ("charges", "atomIDs", "molIDs", "natom_counts", "cells", "inv_cells")]
    energies, forces = one.energies_and_forces(data["coordinates"], *args)
    alone, _ = one.energies_and_forces(data["coordinates"], *args, forces=False)
    Y = data["coordinates"].detach().requires_grad_(True)
    e = other.forward(Y, *args)
    f, = torch.autograd.grad(-e.sum(), Y)
    for got, ref in ((energies, e), (alone, e), (forces, f)):
        assert torch.isfinite(got).all()
        assert (got - ref).norm() <= REL * ref.norm()


@pytest.mark.parametrize("npcas", [64, 128])
@pytest.mark.parametrize("natoms,molecules,taken", [(1, 3, 1), (2, 2, 1), (9, 1, 1), (21, 12, 1), (28, 9, 1), (32, 8, 0), (30, 5, 1), (16, 16, 1),
                                                    (43, 6, 0), (21, 13, 64)])           # (64: with 64 components)
def test_sizes(npcas, natoms, molecules, taken):
    rng = np.random.default_rng(natoms)
    coords, charges = helpers.fixed_composition_batch(rng.choice([1, 6, 8], natoms), molecules, natoms, box=max(4.0, 1.9 * natoms ** (1 / 3)))
    check([1, 6, 8], [1, 6, 8], npcas, coords, charges, taken if taken < 64 else npcas == 64)


@pytest.mark.parametrize("species,elements", [([6], [6]), ([1, 6], [6, 1]), ([1, 6, 8], [1, 6]), ([1, 6], [1, 6, 8]), ([1, 6, 7, 8], [1, 6, 7, 8]), ([1, 6, 7, 8, 9], [1, 6, 7, 8, 9])])
@pytest.mark.parametrize("npcas", [64, 128])
def test_lists_of_elements(species, elements, npcas):
    """The model's list in another order, shorter (atoms that it does not know have no gradient) and longer than the representation's."""
    rng = np.random.default_rng(len(species))
    coords, charges = helpers.fixed_composition_batch(rng.choice(species, 14), 4, 2, box=6.0)
    check(species, elements, npcas, coords, charges, len(species) < 5 or npcas == 64)


@pytest.mark.parametrize("species,npcas,natoms,molecules", [([1, 6, 8], 64, 21, 1), ([1, 6, 8], 128, 21, 12), ([1, 6], 64, 12, 100), ([1, 6, 8], 64, 20, 30)])
def test_random_fourier_features(species, npcas, natoms, molecules):
    """The same two launches, with the gradient in one part."""
    rng = np.random.default_rng(natoms)
    coords, charges = helpers.fixed_composition_batch(rng.choice(species, natoms), molecules, natoms, box=max(4.0, 1.9 * natoms ** (1 / 3)))
    check(species, species, npcas, coords, charges, 1, rff=True)


@pytest.mark.parametrize("species,npcas,natoms,molecules,taken", [
    ([1, 6], 64, 12, 128, 1), ([1, 6], 64, 12, 129, 0), ([1, 6], 64, 29, 9, 1), ([6], 128, 7, 200, 1), ([1, 6, 8], 64, 12, 64, 1),
    ([1, 6, 8], 64, 12, 65, 0), ([1, 6], 128, 24, 32, 1), ([1, 6, 8], 128, 20, 13, 0),
    # larger molecules: one wavefront forms a row, two or four share its triples on the way back
    ([1, 6, 8], 64, 33, 20, 1), ([1, 6], 64, 40, 15, 0), ([1, 6], 64, 40, 25, 1), ([6], 128, 46, 30, 1), ([1, 6], 64, 50, 20, 0)])
def test_more_atoms(species, npcas, natoms, molecules, taken):
    rng = np.random.default_rng(natoms)
    coords, charges = helpers.fixed_composition_batch(rng.choice(species, natoms), molecules, natoms, box=max(4.0, 1.9 * natoms ** (1 / 3)))
    check(species, species, npcas, coords, charges, taken)


def test_ragged_molecules_boxes_and_grids():
    coords, charges = helpers.ragged_batch(12, 2)
    known = [np.isin(q, [1, 6, 8]) for q in charges]
    check([1, 6, 8], [1, 6, 8], 64, [c[k] for c, k in zip(coords, known)], [q[k] for q, k in zip(charges, known)], 1)
    rng = np.random.default_rng(3)
    sites = [rng.uniform(0.0, 9.0, (24, 3)) for _ in range(4)]
    check([1, 6, 8], [1, 6, 8], 128, sites, [rng.choice([1, 6, 8], 24) for _ in sites], 1, edge=9.0)
    coords, charges = helpers.fixed_composition_batch(helpers.ASPIRIN, 2, 6)
    check([1, 6, 8], [1, 6, 8], 128, coords, charges, 1, nRs2=32, nRs3=17)
    check([1, 6], [1, 6], 64, coords, [np.where(q == 8, 6, q) for q in charges], 1, nRs2=7, nRs3=19)
