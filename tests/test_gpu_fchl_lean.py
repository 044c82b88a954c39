"""FCHL19 with the number of elements known to the compiler (usual grids, one wavefront per atom) and with several wavefronts for
few atoms of the same grids, at the edges of what takes them: element counts, grid sizes, capacities, atoms without neighbours, elements that are absent or unknown, periodic boxes."""
import numpy as np
import pytest

from oracle import fchl19
from tests import helpers
from tests.test_gpu_kernels import REL_EF, REL_REP, close, gpu_prm, make_batch, oracle_prm, t32, ti32

pytestmark = pytest.mark.gpu

ATOMS = 2400                    # beyond this one wavefront per atom wherever its kernel holds the triples


def cube(rng, n, edge):
    m = int(np.ceil(n ** (1.0 / 3.0)))
    sites = np.stack(np.unravel_index(rng.permutation(m ** 3)[:n], (m, m, m)), 1)
    return (sites + 0.5) * (edge / m) + rng.uniform(-0.2, 0.2, (n, 3)) * edge / m


class Batch:
    """Molecules, repeated to at least `atoms` atoms, and what the oracle says of them."""

    def __init__(self, coords, charges, species, atoms=ATOMS, cell=None, **kw):
        self.prm = prm = oracle_prm(species, **kw)
        X, Z, aid, mid, nat = make_batch(coords, charges)
        B = len(coords)
        cells = icells = None
        if cell is not None:
            cells = np.broadcast_to(np.eye(3) * cell, (B, 3, 3)).astype(np.float32).astype(np.float64)
            icells = np.linalg.inv(cells).astype(np.float32).astype(np.float64)
        cnt, nl = fchl19.neighbours(X, nat, prm.rcut, cells, icells)
        ty = fchl19.element_types(Z, nat, prm.species)
        for m, i in zip(mid, aid):                      # neighbours of no known element are left out
            js = [j for j in nl[m, i, :cnt[m, i]] if ty[m, j] >= 0]
            nl[m, i], cnt[m, i] = js + [-1] * (nl.shape[2] - len(js)), len(js)
        self.oracle = (X, ty, aid, mid, nl, cnt, prm, cells, icells)
        self.B, k = B, atoms // len(aid) + 1
        tile = lambda a: np.concatenate([a] * k)       # noqa: E731
        box = (None, None) if cell is None else (t32(tile(cells)), t32(tile(icells)))
        self.tile = tile
        self.args = (t32(tile(X)), ti32(tile(ty)), *box, ti32(tile(aid)), ti32(np.concatenate([mid + B * c for c in range(k)])),
                     ti32(tile(nat)), t32(prm.Rs2), t32(prm.Rs3), gpu_prm(prm))

    def forward(self):
        from qml_lightning_amd import ops
        rep = fchl19.forward(*self.oracle)
        got = ops.fchl_forward(*self.args)
        close(got[:self.B], rep, REL_REP, "rep")
        close(got[-self.B:], rep, REL_REP, "rep of the last copy")

    def backward(self):
        from qml_lightning_amd import ops
        g = np.random.default_rng(2).normal(size=(self.B, self.oracle[0].shape[1], self.prm.repsize)).astype(np.float32)
        v = fchl19.vjp(g, *self.oracle)
        for scale in (1.0, -1.0):
            got = ops.fchl_vjp(t32(self.tile(g)), *self.args, scale=scale)
            close(got[:self.B], scale * v, REL_EF, "vjp")
            close(got[-self.B:], scale * v, REL_EF, "vjp of the last copy")


def batches():
    rng = np.random.default_rng(3)
    for ns in range(1, 7):                              # six take the general kernels
        species = [1, 6, 7, 8, 9, 16][:ns]
        n = 13
        yield "%d elements" % ns, ([helpers.random_geometry(rng, n, 5.0, 0.9)], [rng.choice(species, n)], species), {}
    for n in (2, 3, 45, 46):                            # 1024 triples are the most; two atoms have none
        yield "%d atoms" % n, ([cube(rng, n, 7.0 if n > 3 else 2.5)], [rng.choice([1, 6, 8], n)], [1, 6, 8]), {}
    for nrs2, nrs3 in ((32, 17), (1, 18), (24, 19), (32, 20), (33, 20), (24, 16), (24, 21)):
        c, q = helpers.fixed_composition_batch(helpers.ASPIRIN, 1, nrs2 + nrs3)
        yield "grids of %d and %d" % (nrs2, nrs3), (c, q, [1, 6, 8]), dict(nRs2=nrs2, nRs3=nrs3)
    far = np.array([[0, 0, 0], [1.1, 0, 0], [0, 1.2, 0.3], [40.0, 0, 0], [80.0, 0, 0], [81.0, 0, 0]])
    yield "lone atoms", ([far, far[:3], far[3:4]], [[8, 1, 1, 8, 1, 6], [6, 1, 1], [9]], [1, 6, 8, 9]), {}
    yield "absent and unknown elements", ([cube(rng, 12, 6.0)], [[9, 16, 1, 9, 1, 1, 16, 9, 9, 1, 9, 1]], [1, 6, 7, 8, 9]), {}
    # 10.5: beyond what the backward kernel's form about the middle of the grid takes
    c, q = helpers.fixed_composition_batch(helpers.ASPIRIN, 1, 8)
    yield "narrow bins", (c, q, [1, 6, 8]), dict(eta3=12.0)
    for nrs3 in (17, 19):                               # and more triples than the table of several wavefronts holds
        yield "box of 70, %d bins" % nrs3, ([cube(rng, 70, 10.0)], [rng.choice([1, 6, 8], 70)], [1, 6, 8]), dict(cell=10.0, nRs3=nrs3)
    for n in (32, 46, 64):                              # 64: several wavefronts
        yield "box of %d" % n, ([cube(rng, n, 9.0)], [rng.choice([1, 6, 8], n)], [1, 6, 8]), dict(cell=9.0)


ALL = {name: (a, kw) for name, a, kw in batches()}


@pytest.mark.parametrize("atoms", [1, 300, ATOMS])
@pytest.mark.parametrize("name", list(ALL))
def test_forward(name, atoms):
    a, kw = ALL[name]
    Batch(*a, atoms=atoms, **kw).forward()


@pytest.mark.parametrize("atoms", [1, 300, ATOMS])
@pytest.mark.parametrize("name", list(ALL))
def test_backward(name, atoms):
    a, kw = ALL[name]
    Batch(*a, atoms=atoms, **kw).backward()
