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


@pytest.mark.parametrize("case", ["aspirin_c2", "ragged_c3", "flexible_c4"])
@pytest.mark.parametrize("copies", [1, 20])
def test_few_atoms(case, copies):
    """Up to 256 atoms and a few hundred: eight and four wavefronts forward, one and four backward by the number of triples."""
    (coords, charges), species, kw = CASES[case]()
    check(coords, charges, species, copies, copies == 1, **kw)


@pytest.mark.parametrize("natoms", list(range(2, 18)) + [22, 32, 33, 34, 43, 54, 55, 63, 64, 65, 66])
def test_every_neighbour_count_has_its_force_copies(natoms):
    """All atoms within the cutoff of each other: nn = natoms - 1 neighbours, one and several wavefronts per atom."""
    rng = np.random.default_rng(natoms)
    coords = [helpers.random_geometry(rng, natoms, 3.45, 0.35)]
    charges = [rng.choice([1, 6], natoms)]
    for copies in (1, 2050 // natoms + 1):
        check(coords, charges, [1, 6], copies, False, nRs2=3, nRs3=3)


class Padded:
    """Two small molecules of the given elements at the default grids, in batches padded to any capacity."""

    def __init__(self, species, natoms):
        rng = np.random.default_rng(8)
        self.prm = oracle_prm(species)
        coords = [helpers.random_geometry(rng, natoms, 6.0, 0.9), helpers.random_geometry(rng, 2, 3.0, 0.9)]
        self.X, Z, self.aid, self.mid, self.nat = make_batch(coords, [rng.choice(species, len(c)) for c in coords])
        cnt, nl = fchl19.neighbours(self.X, self.nat, self.prm.rcut)
        self.ty = fchl19.element_types(Z, self.nat, self.prm.species)
        args = (self.X, self.ty, self.aid, self.mid, nl, cnt, self.prm)
        self.rep = fchl19.forward(*args)
        self.g = np.random.default_rng(2).normal(size=self.rep.shape)
        self.v = np.einsum("mif,mijxf->mjx", self.g, fchl19.jacobian(*args))

    def __call__(self, op, capacity, *first):
        n = self.X.shape[1]

        def pad(a):
            return np.pad(a, [(0, 0), (0, capacity - n)] + [(0, 0)] * (a.ndim - 2), constant_values=0 if a.ndim == 3 else -1)
        return op(*[t32(pad(f)) for f in first], t32(pad(self.X)), ti32(pad(self.ty)), None, None, ti32(self.aid), ti32(self.mid),
                  ti32(self.nat), t32(self.prm.Rs2), t32(self.prm.Rs3), gpu_prm(self.prm))[:, :n]


@pytest.mark.parametrize("species,forward,backward", [([1, 6, 8], 1268, 1333), ([1, 6, 7, 8, 9], 1259, 1299)])
def test_capacities_up_to_the_limit_of_the_lds(species, forward, backward):
    """The largest capacities: smaller tables and compact force records before a refusal."""
    from qml_lightning_amd import ops
    batch = Padded(species, 19)
    for capacity in (forward - 170, forward):
        close(batch(ops.fchl_forward, capacity), batch.rep, REL_REP, "rep, capacity %d" % capacity)
    for capacity in (backward - 400, backward - 380, backward):
        close(batch(ops.fchl_vjp, capacity, batch.g), batch.v, REL_EF, "vjp, capacity %d" % capacity)
    for op, first in ((ops.fchl_forward, ()), (ops.fchl_vjp, (batch.g,))):
        with pytest.raises(RuntimeError, match="LDS"):
            batch(op, backward + 1, *first)


@pytest.mark.parametrize("nspecies,capacity", [(10, 70), (12, 64), (16, 300)])
def test_grids_too_large_for_more_wavefronts(nspecies, capacity):
    """Many elements at the default grids: the partial blocks leave room for four, two and one wavefronts forward, the force
    copies for four, four and two backward."""
    from qml_lightning_amd import ops
    batch = Padded(list(range(1, nspecies + 1)), 19)
    close(batch(ops.fchl_forward, capacity), batch.rep, REL_REP, "rep")
    close(batch(ops.fchl_vjp, capacity, batch.g), batch.v, REL_EF, "vjp")


def test_a_thousand_neighbours_and_few():
    """1200 atoms, listed one in the middle (some 650 neighbours: its force records take turns) and one at a corner."""
    from qml_lightning_amd import ops
    rng = np.random.default_rng(9)
    species = [1, 8]
    prm = oracle_prm(species, nRs2=2, nRs3=2)
    sites = np.stack(np.unravel_index(rng.permutation(1331)[:1200], (11, 11, 11)), 1) * 1.1
    X, Z, aid, mid, nat = make_batch([sites + rng.uniform(-0.15, 0.15, sites.shape)], [rng.choice(species, 1200)])
    r = np.linalg.norm(X[0] - X[0].mean(0), axis=1)
    aid, mid = np.array([r.argmin(), r.argmax()]), np.array([0, 0])
    cnt, nl = fchl19.neighbours(X, nat, prm.rcut)
    assert cnt[0, aid[0]] > 600 and cnt[0, aid[1]] < 250
    ty = fchl19.element_types(Z, nat, prm.species)
    rep = fchl19.forward(X, ty, aid, mid, nl, cnt, prm)
    g = np.random.default_rng(2).normal(size=rep.shape)
    J = fchl19.jacobian(X, ty, aid, mid, nl, cnt, prm)
    v = np.einsum("if,ijxf->jx", g[0, aid], J[0, aid])[None]
    args = (t32(X), ti32(ty), None, None, ti32(aid), ti32(mid), ti32(nat), t32(prm.Rs2), t32(prm.Rs3), gpu_prm(prm))
    close(ops.fchl_forward(*args)[0, aid], rep[0, aid], REL_REP, "rep")
    close(ops.fchl_vjp(t32(g), *args), v, REL_EF, "vjp")
