"""FCHL19 forward and backward with one and with several wavefronts per atom, at the sizes where the choice, the staging,
the chunks of the triple list and the private force copies change, against the fp64 oracle."""
import numpy as np
import pytest
import torch

from oracle import fchl19
from tests import helpers
from tests.test_gpu_kernels import REL_EF, REL_REP, CASES, close, gpu_prm, make_batch, oracle_prm, t32, ti32

pytestmark = pytest.mark.gpu


def check(coords, charges, species, copies, with_list, **kw):
    from qml_lightning_amd import ops
    prm = oracle_prm(species, **kw)
    X, Z, aid, mid, nat = make_batch(coords, charges)
    cnt, nl = fchl19.neighbours(X, nat, prm.rcut)
    ty = fchl19.element_types(Z, nat, prm.species)
    rep = fchl19.forward(X, ty, aid, mid, nl, cnt, prm)
    J = fchl19.jacobian(X, ty, aid, mid, nl, cnt, prm)
    g = np.random.default_rng(2).normal(size=rep.shape)
    v = np.einsum("mif,mijxf->mjx", g, J)
    B = len(coords)
    tile = lambda a: np.concatenate([a] * copies)       # noqa: E731
    mids = np.concatenate([mid + B * c for c in range(copies)])
    args = (t32(tile(X)), ti32(tile(ty)), None, None, ti32(tile(aid)), ti32(mids), ti32(tile(nat)), t32(prm.Rs2),
            t32(prm.Rs3), gpu_prm(prm))
    lists = dict(nlist=ti32(tile(nl)), nneigh=ti32(tile(cnt))) if with_list else {}
    got = ops.fchl_forward(*args, **lists)
    close(got[:B], rep, REL_REP, "rep")
    close(got[-B:], rep, REL_REP, "rep of the last copy")
    again = ops.fchl_forward(*args, **lists)
    assert torch.equal(got, again)                        # no atomics: the same bits
    gv = ops.fchl_vjp(t32(tile(g)), *args, **lists)
    close(gv[:B], v, REL_EF, "vjp")
    close(gv[-B:], v, REL_EF, "vjp of the last copy")


@pytest.mark.parametrize("with_list", [False, True])
@pytest.mark.parametrize("case", ["aspirin_c2", "ragged_c3", "flexible_c4", "big_molecule", "many_bins", "forty_bins", "sharp_radial",
                                  "short_cutoff"])
def test_one_wavefront_per_atom(case, with_list):
    (coords, charges), species, kw = CASES[case]()
    atoms = sum(len(q) for q in charges)
    check(coords, charges, species, 2100 // atoms + 1, with_list, **kw)


@pytest.mark.parametrize("copies", [1, 6, 40])
def test_more_neighbours_than_one_pass_stages(copies):
    """72 atoms, up to 60 neighbours: 8 and 4 wavefronts per atom, two or three chunks of the triple list."""
    (coords, charges), species, kw = CASES["many_atoms"]()
    check(coords, charges, species, copies, copies == 6, **kw)


def test_more_candidates_than_the_wavefronts_take_at_once():
    """300 atoms in a large box (few neighbours each): beyond 256 candidates with four wavefronts."""
    rng = np.random.default_rng(5)
    coords = [np.stack(np.unravel_index(np.arange(300), (7, 7, 7)), 1) * 3.1 + rng.uniform(-0.8, 0.8, (300, 3))]
    check(coords, [rng.choice([1, 6, 8], 300)], [1, 6, 8], 1, False, nRs2=5, nRs3=4)


@pytest.mark.parametrize("nspecies", [8, 9, 12])
def test_many_elements(nspecies):
    """The scan over the (type, wavefront) counts covers 64 of them; more take the two passes of one wavefront."""
    rng = np.random.default_rng(6)
    species = list(range(1, nspecies + 1))
    coords = [helpers.random_geometry(rng, 70, 12.0, 0.95)]
    check(coords, [rng.choice(species, 70)], species, 1, False, nRs2=4, nRs3=3)


@pytest.mark.parametrize("natoms", list(range(2, 18)) + [22, 32, 33, 34, 43, 54, 55, 63, 64, 65, 66])
def test_every_neighbour_count_has_its_force_copies(natoms):
    """All atoms within the cutoff of each other: nn = natoms - 1 neighbours, one and several wavefronts per atom."""
    rng = np.random.default_rng(natoms)
    coords = [helpers.random_geometry(rng, natoms, 3.45, 0.35)]
    charges = [rng.choice([1, 6], natoms)]
    for copies in (1, 2050 // natoms + 1):
        check(coords, charges, [1, 6], copies, False, nRs2=3, nRs3=3)
