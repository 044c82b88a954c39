"""The matrix-core SORF kernel at 256 components, where the two halves of a vector lie in different lanes: a wavefront carries eight
atoms and a tile 32."""
import numpy as np
import pytest

from oracle import sorf
from qml_lightning_amd import _lib, ops
from tests import test_gpu_kernels as kernels
from tests.test_gpu_kernels import t32, ti32
from tests.test_gpu_sorf_shares import shares
from tests.test_gpu_sorf_limits import test_rows_around_the_limits as rows_around_the_limits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("A,T,S,scale", [(1, 1, 1, 1.0), (8, 2, 2, 1.0), (9, 1, 3, 1.0), (31, 2, 1, 1.0), (33, 1, 4, 1.0), (70, 2, 5, 1.0),
                                         (150, 1, 2, 1.0), (45, 1, 3, 3e4), (45, 2, 3, 2e3)])
def test_edges_of_the_tiles(monkeypatch, A, T, S, scale):
    """Partial wavefronts, tiles and rounds of stacks, rows of unknown elements, arguments of which whole revolutions come off, and the
    rows kernel where a diagonal is not +-1.  (The tolerance is that of the other sizes' test: an argument keeps 2^-24 of itself.)"""
    monkeypatch.setattr(_lib.lib(), "qmll_sorf_matrix_pays", lambda *a: 1)
    rng = np.random.default_rng(A + S)
    d, ne, norm = 256, 3, 2.0
    F = S * d
    types = np.sort(rng.integers(0, ne + 1, A))
    off = np.searchsorted(types, np.arange(ne + 1)).astype(np.int32)
    x = (rng.normal(size=(A, d)) * scale).astype(np.float32)
    D = np.where(rng.uniform(-1, 1, (ne, T, S, d)) > 0, 1.0, -1.0).astype(np.float32)
    b = rng.uniform(0, 2 * np.pi, (ne, F)).astype(np.float32)
    alpha = rng.normal(size=F).astype(np.float32)
    slots = rng.permutation(A).astype(np.int32)
    tol = 2e-5 * max(1.0, scale)
    for diagonal in (D, D * np.float32(1.5)):
        e_ref, g_ref = np.zeros(A), np.zeros((A, d))
        for a in range(int(off[ne])):
            t = types[a]
            c = sorf.sorf_coefficients(x[a][None, :].astype(np.float64), diagonal[t], norm).reshape(1, F)
            e_ref[slots[a]] = (np.sqrt(2.0 / F) * np.cos(c + b[t]) * alpha).sum()
            gc = -np.sqrt(2.0 / F) * np.sin(c + b[t]) * alpha
            g_ref[a] = sorf.sorf_adjoint(gc.reshape(1, S, d), diagonal[t], norm)[0]
        for grad in (True, False):
            e, gx = ops.sorf_energy_sorted(t32(x), ti32(off), ti32(slots), t32(diagonal), t32(b), t32(alpha), norm, T, A, with_grad=grad)
            assert np.abs(e.cpu().numpy() - e_ref).max() <= tol * max(1.0, np.abs(e_ref).max())
            if grad:
                assert np.abs(gx.cpu().numpy() - g_ref).max() <= tol * max(1.0, np.abs(g_ref).max())
                assert (gx[int(off[ne]):] == 0).all()


@pytest.mark.parametrize("mixed", [False, True])
def test_limits_of_the_arguments(monkeypatch, mixed):
    rows_around_the_limits(monkeypatch, 256, mixed)


def test_bounds_of_two_transforms(monkeypatch):
    kernels.test_sorf_matrix_kernel_bounds_the_arguments_of_two_transforms(monkeypatch, 256)


@pytest.mark.parametrize("steep", [False, True])
@pytest.mark.parametrize("T,S", [(1, 128), (2, 32)])
def test_as_exact_as_the_rows_kernel(monkeypatch, T, S, steep):
    kernels.test_sorf_matrix_kernel_is_as_exact_as_the_rows_kernel(monkeypatch, 256, T, S, steep)


# with the gradient 768 workgroups are resident; with 1536 shares: less than an eighth of a tile a share left, an eighth, next to nothing
# behind two tiles each, and whole tiles first again.  With 64 stacks the first three have too few rounds for that, and 768 shares
@pytest.mark.parametrize("S", [64, 256])
@pytest.mark.parametrize("tiles", [863, 864, 1537, 2400])
def test_whole_tiles_first(tiles, S):
    import torch
    L, d, ne = _lib.lib(), 256, 2
    g = torch.Generator(device="cuda").manual_seed(tiles)
    first = tiles // 3
    counts = (32 * first - 5, 32 * (tiles - first) - 31)
    A = sum(counts)
    x = torch.randn(A, d, device="cuda", generator=g)
    D = torch.randint(0, 2, (ne, 1, S, d), device="cuda", generator=g).float() * 2 - 1
    bias = 6.28 * torch.rand(ne, S * d, device="cuda", generator=g)
    alpha = torch.randn(S * d, device="cuda", generator=g)
    off = torch.tensor([0, counts[0], A], dtype=torch.int32, device="cuda")
    slots = torch.randperm(A, device="cuda", generator=g).int()
    assert L.qmll_sorf_matrix_pays(A, ne, 1, S, d, 1) and shares(A, ne, S, d, 1) == (768 if S == 64 and tiles < 2000 else 1536)
    e, gx = ops.sorf_energy_sorted(x, off, slots, D, bias, alpha, 0.7, 1, A)
    p = 2
    ep, gp = torch.zeros(p, A, device="cuda"), torch.empty(p, A, d, device="cuda")
    common = (ops._ptr(x), ops._ptr(off), ops._ptr(slots), ops._ptr(D), ops._ptr(bias), ops._ptr(alpha))
    ops.check(L.qmll_sorf_energy_parts(*common, ops._ptr(bias.abs().max().reshape(1)), A, ne, d, S, 1, 0.7, p, ops._ptr(ep), A, ops._ptr(gp),
                                       ops._stream()), "rows")
    # both within a few 1e-6 of fp64: an entry left out or added twice is off by its own size
    assert float((e - ep.sum(0)).abs().max()) <= 1e-5 * float(e.abs().max())
    assert float((gx - gp.sum(0)).abs().max()) <= 1e-5 * float(gx.abs().max())
