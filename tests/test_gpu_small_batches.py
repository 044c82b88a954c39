"""The kernels of small batches: SORF energies with the stacks in parts, and both small projections at the edges of their rule."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def dev():
    return torch.device("cuda:0")


def _model(A, ne, d, S, T, seed):
    g = torch.Generator(device="cpu").manual_seed(seed)
    types = torch.randint(0, ne + 1, (A,), generator=g).int()                 # the last of them is no element of the model
    x = torch.randn(A, d, generator=g)
    D = torch.sign(torch.rand(ne, T, S, d, generator=g) - 0.5)
    bias = torch.rand(ne, S * d, generator=g) * 6.28
    alpha = torch.randn(S * d, generator=g)
    return [t.to(dev()) for t in (types, x, D, bias, alpha)]


# one and several tiles, more parts than wavefront rounds of stacks (empty parts), both directions of the diagonal's fetch
@pytest.mark.parametrize("A,ne,d,S,T,nparts", [(1, 1, 64, 8, 1, 2), (21, 3, 128, 128, 1, 12), (50, 4, 256, 20, 1, 3), (33, 2, 128, 6, 1, 5),
                                               (21, 3, 64, 32, 2, 4), (130, 4, 256, 9, 2, 2)])
@pytest.mark.parametrize("grad", [True, False])
def test_parts_of_the_stacks_add_up(A, ne, d, S, T, nparts, grad):
    from qml_lightning_amd import _lib, ops
    from qml_lightning_amd.ops import _ptr, _stream
    L = _lib.lib()
    types, x, D, bias, alpha = _model(A, ne, d, S, T, A)
    ss, off = ops.sort_by_type(types, torch.arange(A, dtype=torch.int32, device=dev()), ne)
    bmax = bias.abs().max().reshape(1)

    def run(n):
        e = torch.zeros(n, A, device=dev())
        gx = torch.full((n, A, d), 3.0, device=dev()) if grad else None
        args = (_ptr(x), _ptr(off), _ptr(ss), _ptr(D), _ptr(bias), _ptr(alpha), _ptr(bmax), A, ne, d, S, T, 0.3)
        rc = L.qmll_sorf_energy_parts(*args, n, _ptr(e), A, _ptr(gx), _stream()) if n > 1 else \
            L.qmll_sorf_energy_sorted(*args, _ptr(e), _ptr(gx), _stream())
        assert rc == 0, _lib.last_error()
        return e.double().sum(0), None if gx is None else gx.double().sum(0)

    (e1, g1), (en, gn) = run(1), run(nparts)
    # the same features in another grouping: sums of S d terms of at most |alpha| norm each, rounded to fp32
    terms = float(alpha.abs().max()) * np.sqrt(2.0 / (S * d)) * np.sqrt(S * d) * 2.0 ** -24
    assert float((en - e1).abs().max()) <= 16 * terms * np.sqrt(S * d)
    if grad:
        assert float((gn - g1).abs().max()) <= 16 * terms * np.sqrt(S * d) * np.sqrt(d) * 0.3
        known = int(off[ne])
        assert (gn[known:] == 0).all()


# 32 columns of one, two and four atoms, 128 columns of four, 32 of eight, partial columns; with parts, and with more atoms than
# the small kernels take
@pytest.mark.parametrize("A,ne,R,d", [(1, 1, 168, 64), (30, 3, 312, 128), (200, 3, 312, 128), (700, 2, 168, 128), (1500, 3, 312, 128),
                                      (3000, 5, 720, 64), (600, 4, 496, 256), (40, 2, 168, 100), (4200, 3, 312, 128)])
@pytest.mark.parametrize("nparts", [1, 3])
def test_small_projections(A, ne, R, d, nparts):
    from qml_lightning_amd import _lib, ops
    from qml_lightning_amd.ops import _ptr, _stream
    L = _lib.lib()
    g = torch.Generator(device="cpu").manual_seed(R + A)
    types = torch.randint(0, ne + 1, (A,), generator=g).int().to(dev())
    ss, off = ops.sort_by_type(types, torch.arange(A, dtype=torch.int32, device=dev()), ne)
    known = int(off[ne])
    rep, U = torch.randn(A, R, generator=g).to(dev()), torch.randn(ne, R, d, generator=g).to(dev())
    gx = torch.randn(nparts, A, d, generator=g).to(dev())
    n = 1 if A % 3 else 3
    e = torch.randn(nparts, A, generator=g).to(dev())
    total, e_total = gx.double().sum(0), e.double().sum(0).view(-1, n).sum(1)
    x = torch.full((A, d), 9.0, device=dev())
    assert L.qmll_project_typed(_ptr(rep), _ptr(ss), _ptr(off), _ptr(U), None, A, ne, R, d, _ptr(x), _stream()) == 0
    g_rep = torch.full((A, R), 9.0, device=dev())
    energies = torch.empty(A // n, device=dev())
    rc = L.qmll_project_typed_backward_parts(_ptr(gx), nparts, _ptr(ss), _ptr(off), _ptr(U), None, _ptr(types), A, A, ne, R, d, _ptr(g_rep),
                                             _ptr(e), A // n, n, _ptr(energies), _stream())
    assert rc == 0, _lib.last_error()
    slots = ss[:known].long()
    for t in range(ne):
        a, b = int(off[t]), int(off[t + 1])
        rows, back = rep[slots[a:b]].double() @ U[t].double(), total[a:b] @ U[t].double().T
        # fp32 sums of R (d) products
        assert float((x[a:b] - rows).abs().max()) <= 4 * R ** 0.5 * 2.0 ** -24 * float(rows.abs().max()) if b > a else True
        assert float((g_rep[slots[a:b]] - back).abs().max()) <= 4 * (d + nparts) ** 0.5 * 2.0 ** -24 * float(back.abs().max()) if b > a else True
    unknown = (types >= ne).nonzero()[:, 0]
    assert (g_rep[unknown] == 0).all()
    assert float((energies - e_total).abs().max()) <= 4 * nparts * n * 2.0 ** -24 * float(e.abs().max())


@pytest.mark.parametrize("elements", [[1, 6, 8], [8, 1], [6, 1, 9, 8, 7, 16, 17, 2], [1, 6, 7, 8, 9, 16, 17, 2, 3]])
@pytest.mark.parametrize("atoms,pad", [(1, 0), (21, 0), (63, 1), (65, 0), (256, 0), (257, 0), (30, 40)])
def test_batch_prepared_beside_the_representation(elements, atoms, pad):
    """The one launch of few atoms against the separate kernels: up to 256 atoms, a model with its own element list (in another
    order, more elements than the launch sorts), padded slots, atoms listed in another order than they are stored."""
    _prepared_beside_the_representation([1, 6, 8], elements, atoms, pad, None)


@pytest.mark.parametrize("species", [[1], [6, 1], [1, 6, 8], [1, 6, 7, 8], [1, 6, 7, 8, 9], [1, 6, 7, 8, 9, 16]])
@pytest.mark.parametrize("elements", [None, [8, 1]])
@pytest.mark.parametrize("edge", [None, 6.5])
def test_batch_prepared_beside_the_representation_of_any_species(species, elements, edge):
    """A kernel for each number of the representation's elements (six take the separate kernels), free and in boxes."""
    for atoms in (1, 64, 250):
        _prepared_beside_the_representation(species, elements or species, atoms, 3, edge)


def _prepared_beside_the_representation(species, elements, atoms, pad, edge):
    import ctypes
    from qml_lightning_amd import _lib, ops
    from qml_lightning_amd.representations.FCHL import FCHLCuda
    rng = np.random.default_rng(atoms)
    rep = FCHLCuda(species=np.array(species))
    n = 21
    B = (atoms + n - 1) // n
    counts = np.minimum(n, atoms - n * np.arange(B))
    n += pad
    dev = torch.device("cuda:0")
    X = torch.tensor(rng.uniform(0, 6, (B, n, 3)), dtype=torch.float32, device=dev)
    Z = torch.tensor(np.where(np.arange(n) < counts[:, None], rng.choice(sorted({1, 6, 8, 16} | set(species)), (B, n)), 0), dtype=torch.float32, device=dev)
    order = rng.permutation(atoms)
    aid = torch.tensor(np.concatenate([np.arange(k) for k in counts])[order], dtype=torch.int32, device=dev)
    mid = torch.tensor(np.repeat(np.arange(B), counts)[order], dtype=torch.int32, device=dev)
    nat = torch.tensor(counts, dtype=torch.int32, device=dev)
    cell = icell = None
    if edge is not None:
        cell = torch.eye(3, device=dev).mul(edge).expand(B, 3, 3).contiguous()
        icell = torch.eye(3, device=dev).div(edge).expand(B, 3, 3).contiguous()
    msp = None if elements == species else torch.tensor(elements, dtype=torch.float32, device=dev)
    types, stypes, ss, off, zeroed = ops.prepare_batch(Z, nat, rep.species, aid, mid, msp, 5 * B * n)
    prm = ops.make_params(len(species), rep.Rs2, rep.Rs3, rep.eta2, rep.eta3, rep.two_body_decay, rep.three_body_weight,
                          rep.three_body_decay, rep.rcut)
    want = ops.fchl_forward(X, types, cell, icell, aid, mid, nat, rep.Rs2, rep.Rs3, prm)
    ne = len(elements)
    got = [torch.full_like(t, -7) for t in (types, stypes, ss, off)]
    zero = torch.full((5 * B * n,), 3.0, device=dev)
    r = torch.zeros_like(want)
    work = torch.empty(65536, dtype=torch.int32, device=dev)
    p = lambda t: ctypes.c_void_p(0 if t is None else t.data_ptr())       # noqa: E731
    _lib.check(_lib.lib().qmll_prepare_fchl19_forward(
        p(X), p(Z), p(rep.species), p(msp), ne, p(cell), p(icell), p(aid), p(mid), p(nat), atoms, B, n, p(rep.Rs2), p(rep.Rs3),
        ctypes.byref(prm), p(work), 4 * 65536, p(got[0]), p(got[1]) if msp is not None else None, p(got[2]), p(got[3]), p(zero),
        zero.numel(), p(r), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "qmll_prepare_fchl19_forward")
    assert torch.equal(got[0], types) and (msp is None or torch.equal(got[1], stypes))
    assert torch.equal(got[2], ss) and torch.equal(got[3], off)
    assert not zero.any()
    assert torch.equal(r, want)
