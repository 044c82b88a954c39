"""The matrix-core SORF kernel where its launch has two rounds of workgroups: whole tiles first, cut ones in the last round."""
import pytest
import torch

from qml_lightning_amd import _lib, ops

pytestmark = pytest.mark.gpu


def shares(A, ne, S, d, with_grad):
    """Shares of a call: its workspace holds a tile's part for each of them beside the forms, which do not depend on A."""
    L, atoms, resident = _lib.lib(), 32 if d == 256 else 64, 256 * (3 if with_grad and d >= 128 else 4)
    rounds = (S + 1) // 2
    nbytes = [int(L.qmll_sorf_matrix_workspace_bytes(a, ne, 1, S, d, with_grad)) for a in (1, A)]
    slot = 4 * atoms * (d + 1 if with_grad else 1)
    assert (nbytes[1] - nbytes[0]) % slot == 0
    return min((1 + ne) * rounds, resident) + (nbytes[1] - nbytes[0]) // slot


# d = 128 with the gradient, 768 workgroups resident; with 1536 shares: 863 tiles (less than an eighth of a tile a share would be left: equal
# shares), 864 (an eighth: eight parts a tile), 1346, 1536 (none left to cut), 1537 (two tiles each would be all but one), 1632 (an
# eighth again), 2400; the last tiles of the elements are not full.  With 128 stacks the first two have too few rounds for that, and 768 shares.
@pytest.mark.parametrize("S", [128, 256])
@pytest.mark.parametrize("tiles", [863, 864, 1346, 1536, 1537, 1632, 2400])
def test_whole_tiles_first(tiles, S):
    L, d, ne = _lib.lib(), 128, 2
    g = torch.Generator(device="cuda").manual_seed(tiles)
    first = tiles // 3
    counts = (64 * first - 5, 64 * (tiles - first) - 63)
    A = sum(counts)
    x = torch.randn(A, d, device="cuda", generator=g)
    D = torch.sign(torch.randn(ne, 1, S, d, device="cuda", generator=g))
    bias = 6.28 * torch.rand(ne, S * d, device="cuda", generator=g)
    alpha = torch.randn(S * d, device="cuda", generator=g)
    off = torch.tensor([0, counts[0], A], dtype=torch.int32, device="cuda")
    slots = torch.randperm(A, device="cuda", generator=g).int()
    bmax = bias.abs().max().reshape(1)
    assert L.qmll_sorf_matrix_pays(A, ne, 1, S, d, 1) and shares(A, ne, S, d, 1) == (768 if S == 128 and tiles < 1000 else 1536)
    e, gx = torch.zeros(A, device="cuda"), torch.full((A, d), 7.0, device="cuda")
    work = torch.empty(int(L.qmll_sorf_matrix_workspace_bytes(A, ne, 1, S, d, 1)), dtype=torch.uint8, device="cuda")
    common = (ops._ptr(x), ops._ptr(off), ops._ptr(slots), ops._ptr(D), ops._ptr(bias), ops._ptr(alpha))
    ops.check(L.qmll_sorf_energy_matrix(*common, A, ne, d, S, 1, 0.7, ops._ptr(work), work.numel(), ops._ptr(e), ops._ptr(gx), ops._stream()), "matrix")
    # the rows kernel, with the stacks in two parts
    p = 2
    ep, gp = torch.zeros(p, A, device="cuda"), torch.empty(p, A, d, device="cuda")
    ops.check(L.qmll_sorf_energy_parts(*common, ops._ptr(bmax), A, ne, d, S, 1, 0.7, p, ops._ptr(ep), A, ops._ptr(gp), ops._stream()), "rows")
    e_rows, gx_rows = ep.sum(0), gp.sum(0)
    # both within a few 1e-6 of fp64 (the bounds of the tests of either kernel): an entry left out or added twice is off by its own size
    assert float((e - e_rows).abs().max()) <= 1e-5 * float(e_rows.abs().max())
    assert float((gx - gx_rows).abs().max()) <= 1e-5 * float(gx_rows.abs().max())


# energies only, 1024 workgroups resident and 2048 shares: 1151 tiles leave less than an eighth of a tile a share, 1152 an eighth, 2049 next
# to nothing behind two tiles each, 2176 an eighth again; 1000 tiles have 1024 equal shares
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("tiles", [1000, 1151, 1152, 2048, 2049, 2176])
def test_energies_of_whole_tiles_first(tiles, d):
    L, S, ne, atoms = _lib.lib(), 128, 2, 32 if d == 256 else 64
    g = torch.Generator(device="cuda").manual_seed(tiles)
    first = tiles // 3
    counts = (atoms * first - 5, atoms * (tiles - first) - atoms + 1)
    A = sum(counts)
    x = torch.randn(A, d, device="cuda", generator=g)
    D = torch.randint(0, 2, (ne, 1, S, d), device="cuda", generator=g).float() * 2 - 1
    bias = 6.28 * torch.rand(ne, S * d, device="cuda", generator=g)
    alpha = torch.randn(S * d, device="cuda", generator=g)
    off = torch.tensor([0, counts[0], A], dtype=torch.int32, device="cuda")
    slots = torch.randperm(A, device="cuda", generator=g).int()
    assert L.qmll_sorf_matrix_pays(A, ne, 1, S, d, 0) and shares(A, ne, S, d, 0) == (1024 if tiles == 1000 else 2048)
    e, _ = ops.sorf_energy_sorted(x, off, slots, D, bias, alpha, 0.7, 1, A, with_grad=False)
    p = 2
    ep, gp = torch.zeros(p, A, device="cuda"), torch.empty(p, A, d, device="cuda")
    common = (ops._ptr(x), ops._ptr(off), ops._ptr(slots), ops._ptr(D), ops._ptr(bias), ops._ptr(alpha))
    ops.check(L.qmll_sorf_energy_parts(*common, ops._ptr(bias.abs().max().reshape(1)), A, ne, d, S, 1, 0.7, p, ops._ptr(ep), A, ops._ptr(gp),
                                       ops._stream()), "rows")
    assert float((e - ep.sum(0)).abs().max()) <= 1e-5 * float(e.abs().max())
