"""The radial bins of the three-body part: kernels for 17 to 20 of them take evenly spaced ones of ordinary cutoffs in groups of five (a
polynomial in the ratio of two weights) and any others one by one; both against the oracle on the same grid, and distances far beyond the cutoff from a
given list.  Tolerance: largest error over largest value, REL_REP; forces are sums of both signs over the bins, ten times that
(2-norm errors are 2e-7 to 6e-7 on either route)."""
import numpy as np
import pytest
import torch

from oracle import fchl19
from tests import helpers
from tests.test_gpu_kernels import REL_REP, close, gpu_prm, make_batch, oracle_prm, t32, ti32

pytestmark = pytest.mark.gpu

GRIDS = {
    "even": lambda n, rc: np.linspace(0.0, rc, n + 1)[1:],
    "descending": lambda n, rc: np.linspace(0.0, rc, n + 1)[1:][::-1],
    "shifted": lambda n, rc: np.linspace(0.7, 0.8 * rc, n),
    "quadratic": lambda n, rc: rc * (np.arange(1, n + 1) / n) ** 2,
    "one moved": lambda n, rc: np.linspace(0.0, rc, n + 1)[1:] + 1e-4 * (np.arange(n) == 9),
    "all equal": lambda n, rc: np.full(n, 2.0),
}


def check(natoms, molecules, nrs3, grid, seed, spread=1.0, **kw):
    from qml_lightning_amd import ops
    rng = np.random.default_rng(seed)
    species = [1, 6, 8]
    coords, charges = helpers.fixed_composition_batch(rng.choice(species, natoms), molecules, seed, box=max(6.0, 1.9 * natoms ** (1 / 3)))
    prm = oracle_prm(species, nRs3=nrs3, **kw)
    prm.Rs3 = GRIDS[grid](nrs3, prm.rcut).astype(np.float32).astype(np.float64)
    X, Z, aid, mid, nat = make_batch(coords, charges)
    types = fchl19.element_types(Z, nat, prm.species)
    nneigh, nlist = fchl19.neighbours(X, nat, prm.rcut)
    X = (X * spread).astype(np.float32).astype(np.float64)       # a stale list: distances that the cutoff would not let in
    ref = fchl19.forward(X, types, aid, mid, nlist, nneigh, prm)
    g = rng.normal(size=ref.shape).astype(np.float32)
    gref = fchl19.vjp(g.astype(np.float64), X, types, aid, mid, nlist, nneigh, prm)
    args = [t32(X), ti32(types), None, None, ti32(aid), ti32(mid), ti32(nat), t32(prm.Rs2), t32(prm.Rs3), gpu_prm(prm)]
    if spread != 1.0:
        args += [ti32(nlist), ti32(nneigh)]
    close(ops.fchl_forward(*args), ref, REL_REP, "representation")
    got = ops.fchl_vjp(t32(g), *args)
    assert torch.isfinite(got).all()
    close(got, gref, 10 * REL_REP, "gradient")


@pytest.mark.parametrize("grid", GRIDS)
@pytest.mark.parametrize("natoms,molecules", [(9, 3), (52, 1)])           # one wavefront per atom, several
def test_grids(grid, natoms, molecules):
    check(natoms, molecules, 20, grid, 11)


@pytest.mark.parametrize("nrs3", [17, 18, 19])
@pytest.mark.parametrize("natoms,molecules", [(14, 2), (50, 1)])
def test_bins_that_are_not_there(nrs3, natoms, molecules):
    """(17 of them, 0.35 A apart, are taken in groups where distances end at the cutoff, and one by one with a given list.)"""
    check(natoms, molecules, nrs3, "even", nrs3)


@pytest.mark.parametrize("natoms", [12, 50])
@pytest.mark.parametrize("kw", [dict(eta3=12.0), dict(rcut=9.0, eta3=4.0), dict(rcut=2.5)])
def test_weights_beyond_the_range_of_the_ratio(kw, natoms):
    check(natoms, 1, 20, "even", 5, **kw)


@pytest.mark.parametrize("spread", [1.3, 4.0])
@pytest.mark.parametrize("rcut", [6.0, 6.4, 8.0, 10.0])
def test_distances_beyond_the_cutoff(spread, rcut):
    check(30, 1, 20, "even", 3, spread=spread, rcut=rcut)


@pytest.mark.parametrize("natoms", [12, 66])
@pytest.mark.parametrize("share", [0.4, 0.7])
def test_bins_in_the_middle_of_the_range(natoms, share):
    """Distances far beyond all bins, where the ratio of two weights stops short."""
    GRIDS["middle"] = lambda n, rc: np.linspace(0.5 * (1 - share) * rc, 0.5 * (1 + share) * rc, n)
    check(natoms, 1, 20, "middle", 4, rcut=9.0)


@pytest.mark.parametrize("natoms", [12, 50, 66])
@pytest.mark.parametrize("nrs3,kw", [(20, dict(rcut=6.4)), (20, dict(rcut=6.5)), (17, dict(rcut=6.0)), (20, dict(rcut=8.0)), (20, dict(rcut=8.1)),
                                     (20, dict(rcut=8.2)), (17, dict(rcut=8.0)), (20, dict(rcut=10.0)),
                                     (20, dict(rcut=12.0)), (20, dict(rcut=12.3)), (17, dict(rcut=10.2)), (17, dict(rcut=10.5))])
def test_either_side_of_the_lines(nrs3, kw, natoms):
    """Cutoffs around those up to which the ratio of two weights has room (6.4 A where distances may be anything, else 8.1 A), beyond, where it
    stops short, and past 12.1 A (17 bins: 10.3), where bins are taken one by one."""
    check(natoms, 1, nrs3, "even", 7, **kw)


@pytest.mark.parametrize("size", [1e-12, 1e6])
def test_gradients_of_any_size(size):
    """The sums over a group reach 2^104 of its coefficients where the weight before them has underflown."""
    from qml_lightning_amd import ops
    rng = np.random.default_rng(2)
    coords, charges = helpers.fixed_composition_batch(rng.choice([1, 6, 8], 30), 1, 2, box=14.0)
    prm = oracle_prm([1, 6, 8], rcut=8.1)
    X, Z, aid, mid, nat = make_batch(coords, charges)
    types = fchl19.element_types(Z, nat, prm.species)
    args = [t32(X), ti32(types), None, None, ti32(aid), ti32(mid), ti32(nat), t32(prm.Rs2), t32(prm.Rs3), gpu_prm(prm)]
    g = torch.randn(X.shape[0], X.shape[1], prm.nspecies * prm.nRs2 + prm.nspecies * (prm.nspecies + 1) * prm.nRs3, device="cuda")
    ref = ops.fchl_vjp(g, *args)
    got = ops.fchl_vjp(g * size, *args) / size
    assert torch.isfinite(got).all() and (got - ref).norm() <= 1e-5 * ref.norm()
