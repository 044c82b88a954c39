"""One transform on the matrix cores, with rows on either side of the sums between which all atoms share one power of two (128
revolutions; downwards where the bias is small) and up to which a stack leaves its arguments as they are (1500 radians)."""
import numpy as np
import pytest
import torch

from oracle import sorf
from qml_lightning_amd import _lib, ops
from tests.test_gpu_kernels import t32, ti32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("mixed", [False, True])       # all rows on one side, or one row in a wavefront beyond
def test_rows_around_the_limits(monkeypatch, d, mixed):
    monkeypatch.setattr(_lib.lib(), "qmll_sorf_matrix_pays", lambda *a: 1)
    rng = np.random.default_rng(d + mixed)
    ne, S, norm, A = 2, 5, 2.0, 40
    F = S * d
    D = np.where(rng.uniform(-1, 1, (ne, 1, S, d)) > 0, 1.0, -1.0).astype(np.float32)
    b = rng.uniform(0, 2 * np.pi, (ne, F)).astype(np.float32)
    alpha = rng.normal(size=F).astype(np.float32)
    off = np.array([0, 20, A], dtype=np.int32)
    shapes = rng.normal(size=(A, d))
    shapes[::3] *= np.eye(d)[rng.integers(d, size=len(shapes[::3]))] + 1e-3        # one large component: the argument is the sum
    for limit in (128.0, 1500.0 / (2 * np.pi)):
        for near in (0.98, 0.999, 1.001, 1.02):
            of = np.full(A, near)
            if mixed:
                of = np.where(np.arange(A) % 16 == 5, near, 0.01)
            # (sum |x| in revolutions, behind the kernel's factor norm / sqrt(d))
            x = (shapes / np.abs(shapes).sum(1, keepdims=True) * (of * limit)[:, None] * 2 * np.pi * np.sqrt(d) / norm).astype(np.float32)
            e_ref, g_ref, err = np.zeros(A), np.zeros((A, d)), np.zeros((A, 1))
            for a in range(A):
                t = int(a >= off[1])
                c = sorf.sorf_coefficients(x[a][None, :].astype(np.float64), D[t], norm).reshape(1, F)
                e_ref[a] = (np.sqrt(2.0 / F) * np.cos(c + b[t]) * alpha).sum()
                gc = -np.sqrt(2.0 / F) * np.sin(c + b[t]) * alpha
                g_ref[a] = sorf.sorf_adjoint(gc.reshape(1, S, d), D[t], norm)[0]
                # an argument is off by at most 2^-22 of the bound on it and the sine unit by 2^-20; features add up at worst
                bound = np.abs(x[a]).sum() * norm / np.sqrt(d) + 2 * np.pi
                err[a] = np.sqrt(2.0 / F) * np.abs(alpha).sum() * (bound * 2.0 ** -22 + 2.0 ** -20)
            for grad in (True, False):
                e, gx = ops.sorf_energy_sorted(t32(x), ti32(off), ti32(np.arange(A)), t32(D), t32(b), t32(alpha), norm, 1, A,
                                               with_grad=grad)
                assert (np.abs(e.cpu().numpy() - e_ref) <= err[:, 0]).all(), (limit, near)
                if grad:
                    assert (np.abs(gx.cpu().numpy() - g_ref) <= err * norm / np.sqrt(d)).all(), (limit, near)


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("steep", [False, True])
@pytest.mark.parametrize("size", [1e-2, 1e-3, 1e-4])
@pytest.mark.parametrize("alone", [False, True])       # all rows so small, or two of a wavefront
def test_small_arguments_without_bias(monkeypatch, d, steep, size, alone):
    """Where all arguments are small and no bias stands beside them the gradient follows x itself.  Entries of x keep 23 bits (rms
    0.7 x 2^-24) behind an atom's own power of two, where the rows kernel has fp32 sums: measured 0.9 to 1.25 of its error; entries cut
    off at 2^-33 revolutions were 1.3 to 60 times off."""
    S, n, norm = 16, 512, 1.5
    F = S * d
    g = torch.Generator(device="cuda").manual_seed(d)
    D = torch.randint(0, 2, (1, 1, S, d), device="cuda", generator=g).float() * 2 - 1
    alpha = torch.randn(F, device="cuda", generator=g)
    b = torch.zeros(1, F, device="cuda")
    b[0, d:2 * d] = np.pi                              # (whole halves of a revolution are the sign of alpha)
    x = torch.randn(n, d, device="cuda", generator=g)
    if steep:
        x = x * torch.logspace(0, -3, d, device="cuda")
    small = torch.ones(n, dtype=torch.bool, device="cuda")
    if alone:
        small = torch.arange(n, device="cuda") % 8 == 3
    x = torch.where(small[:, None], x * size, x)
    H = torch.tensor([[(-1.0) ** bin(i & j).count("1") for j in range(d)] for i in range(d)], dtype=torch.float64, device="cuda")
    c = (x.double()[:, None, :] * D[0, 0].double()) @ H / d ** 0.5
    weight = alpha.double().view(S, d) * (2.0 / F) ** 0.5
    gr = ((-torch.sin(c * norm + b.double().view(S, d)) * weight * norm) @ H / d ** 0.5 * D[0, 0].double()).sum(1)
    errors = {}
    for name in ("rows", "matrix"):
        monkeypatch.setattr(_lib.lib(), "qmll_sorf_matrix_pays", lambda *a: int(name == "matrix"))
        _, gx = ops.sorf_energy_sorted(x, ti32([0, n]), ti32(np.arange(n)), D, b, alpha, norm, 1, n)
        errors[name] = float(((gx.double() - gr)[small].norm() / gr[small].norm()))
    assert errors["matrix"] <= 1.5 * errors["rows"], errors


@pytest.mark.parametrize("d,S", [(128, 256), (128, 257), (64, 513), (256, 200)])      # 32768 entries, and more
@pytest.mark.parametrize("T", [1, 2])
def test_scale_of_many_coefficients(monkeypatch, d, S, T):
    """The largest alpha may be in any piece of it, and infinite ones do not count: the entries around it are tiny, and the answer is
    that of the rows kernel to a few 2^-24 of the sums."""
    monkeypatch.setattr(_lib.lib(), "qmll_sorf_matrix_pays", lambda *a: 1)
    n, ne, F = 40, 2, S * d
    g = torch.Generator(device="cuda").manual_seed(S)
    D = torch.randint(0, 2, (ne, T, S, d), device="cuda", generator=g).float() * 2 - 1
    b = 6.28 * torch.rand(ne, F, device="cuda", generator=g)
    x = torch.randn(n, d, device="cuda", generator=g)
    off, slots = ti32([0, 17, n]), ti32(np.arange(n))
    for at in (0, 8191, 8192, F // 2, F - 1):
        alpha = 1e-6 * torch.randn(F, device="cuda", generator=g)
        alpha[at] = 3e4
        got = {}
        for name in ("rows", "matrix"):
            monkeypatch.setattr(_lib.lib(), "qmll_sorf_matrix_pays", lambda *a: int(name == "matrix"))
            got[name] = ops.sorf_energy_sorted(x, off, slots, D, b, alpha, 1.5, T, n)
        for r, m in zip(got["rows"], got["matrix"]):
            assert torch.isfinite(m).all()
            assert (m - r).norm() <= 1e-5 * r.norm()


def test_few_atoms_of_many_stacks_stay_on_the_rows_kernel():
    """With the gradient and up to 128 components the line between the two kernels rises with the stacks, as the forms and the parts of a
    tile do."""
    pays = _lib.lib().qmll_sorf_matrix_pays
    for T, S, low, high in ((1, 128, 11600, 11900), (1, 512, 3600, 3800), (1, 2048, 970, 980), (2, 32, 18700, 18800), (2, 512, 1800, 1960)):
        assert not pays(low, 4, T, S, 128, 1) and pays(high, 4, T, S, 128, 1), (T, S)
    assert pays(1000, 4, 2, 200, 256, 1) and pays(12100, 4, 1, 128, 128, 0) and pays(3000, 4, 1, 512, 128, 0)
