"""The Cholesky factorisation's panels, whose columns follow the factorisation of a diagonal block step by step: one to four blocks in the
last panel, with and without columns beside it; the first pivot that is not positive in each block; the same bits each time.  Sizes that
are no whole blocks are solved in a copy with ones behind the matrix."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def problem(F, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    Z = torch.randn(F + F // 2, F, device="cuda", dtype=torch.float64, generator=gen)
    A = Z.T @ Z
    A.diagonal().add_(1.0)
    return A, A @ torch.randn(F, 1, device="cuda", dtype=torch.float64, generator=gen)


@pytest.mark.parametrize("F", [128 * blocks for blocks in (1, 2, 3, 4, 5, 6, 7, 8, 13)] + [2, 126, 130, 320, 510, 514, 1090])
def test_blocks_of_a_panel(F):
    from qml_lightning_amd import ops
    A, b = problem(F, F)
    kept = A.clone(), b.clone()
    x, info = ops.cholesky_solve_spd(A, b)
    assert int(info) == 0 and x.shape == b.shape
    assert torch.equal(A, kept[0]) and torch.equal(b, kept[1])
    # backward error of a Cholesky solve: at most 3 (F + 1) eps |A| |x| for each component, and far below it as a rule
    bound = 3.0 * (F + 1) * 2.0 ** -53 * (A.abs() @ x.abs())
    assert ((A @ x - b).abs() <= 0.25 * bound).all()
    again, _ = ops.cholesky_solve_spd(A, b)
    assert torch.equal(again, x)


@pytest.mark.parametrize("blocks,pivot", [(1, 77), (4, 5), (4, 130), (4, 300), (4, 511), (5, 200), (9, 640), (9, 900), (2.5, 319), (4.5, 40)])
def test_first_pivot_that_is_not_positive(blocks, pivot):
    from qml_lightning_amd import ops
    F = int(128 * blocks)
    A, b = problem(F, 3)
    A[pivot, pivot] = -1.0
    _, info = ops.cholesky_solve_spd(A, b)
    assert int(info) == pivot + 1


@pytest.mark.parametrize("F,offset", [(384, 1), (512, 1), (300, 1), (1090, 0)])
def test_in_place_in_a_wider_buffer(F, offset):
    """Rows 8 bytes past an aligned address: whole blocks are factored by a launch per step, the other sizes in their padded copy,
    whose factor ends up in the matrix."""
    from qml_lightning_amd import ops
    A, b = problem(F, F)
    wide = torch.full((F, F + 8), 7.0, device="cuda", dtype=torch.float64)
    view = wide[:, offset:offset + F]
    view.copy_(A)
    x, info = ops.cholesky_solve_spd(view, b, overwrite_a=True)
    assert int(info) == 0 and x.shape == b.shape
    assert ((A @ x - b).abs() <= 0.75 * (F + 1) * 2.0 ** -53 * (A.abs() @ x.abs())).all()
    U = torch.triu(view)
    bound = 2 * (F + 1) * 2.0 ** -53 * (U.abs().T @ U.abs())        # (F + 1) eps for the factorisation, as much for the product here
    assert ((U.T @ U - A).abs() <= bound).all()
    assert (wide[:, :offset] == 7.0).all() and (wide[:, offset + F:] == 7.0).all()


@pytest.mark.parametrize("F,beside", [(128, 2), (512, 2), (512, 8), (640, 2), (1152, 2), (1664, 6)])
def test_panels_in_a_wider_buffer(F, beside):
    """Whole blocks whose rows are longer than the matrix, aligned as the panels' launches need: tiles side by side then share lines of
    memory at their edges, and what is beside the matrix stays."""
    from qml_lightning_amd import ops
    A, b = problem(F, F)
    plain, _ = ops.cholesky_solve_spd(A, b)
    wide = torch.full((F, F + beside), 7.0, device="cuda", dtype=torch.float64)
    view = wide[:, :F]
    view.copy_(A)
    assert view.data_ptr() % 16 == 0
    x, info = ops.cholesky_solve_spd(view, b, overwrite_a=True)
    assert int(info) == 0 and torch.equal(x, plain)          # the same sums in the same order
    U = torch.triu(view)
    assert ((U.T @ U - A).abs() <= 2 * (F + 1) * 2.0 ** -53 * (U.abs().T @ U.abs())).all()
    assert (wide[:, F:] == 7.0).all()


@pytest.mark.parametrize("F", [130, 255, 514, 642])
def test_ragged_sizes_in_the_c_interface(F):
    """The last block of the launches per step and of the two triangular solves ends inside a tile, in rows of any alignment."""
    from qml_lightning_amd import _lib, ops
    A, b = problem(F, F)
    ld = F + 2 + F % 2                                  # even, as the interface asks for
    U = torch.zeros(F, ld, device="cuda", dtype=torch.float64)
    U[:, :F] = A
    L = _lib.lib()
    work = torch.empty(int(L.qmll_cholesky_workspace_bytes(F)) // 8 + 1, dtype=torch.float64, device="cuda")
    info = torch.zeros(1, dtype=torch.int32, device="cuda")
    x = b.clone()
    _lib.check(L.qmll_cholesky_f64(ops._ptr(U), F, ld, ops._ptr(work), ops._ptr(info), ops._stream()), "qmll_cholesky_f64")
    _lib.check(L.qmll_cholesky_solve_f64(ops._ptr(U), F, ld, ops._ptr(work), ops._ptr(x), ops._stream()), "qmll_cholesky_solve_f64")
    assert int(info) == 0
    assert ((A @ x - b).abs() <= 0.75 * (F + 1) * 2.0 ** -53 * (A.abs() @ x.abs())).all()


@pytest.mark.parametrize("F", [1024, 4096])
def test_sums_of_the_triangular_solves(F):
    """U with a unit diagonal and all entries of one sign, so that the products of a row add up: a running sum over F terms is off by some
    sqrt(F) roundings, four of a quarter of the terms by fewer.  The residual in long double."""
    import numpy as np
    from qml_lightning_amd import _lib, ops
    L = _lib.lib()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(F)
    U = torch.triu(torch.rand(F, F, device="cuda", dtype=torch.float64, generator=gen) / F, 1)
    U.diagonal().add_(1.0)
    A = U.T @ U
    x = torch.rand(F, device="cuda", dtype=torch.float64, generator=gen)
    work = torch.empty(int(L.qmll_cholesky_workspace_bytes(F)) // 8 + 1, dtype=torch.float64, device="cuda")
    info = torch.zeros(1, dtype=torch.int32, device="cuda")
    _lib.check(L.qmll_cholesky_f64(ops._ptr(A), F, F, ops._ptr(work), ops._ptr(info), ops._stream()), "qmll_cholesky_f64")
    assert int(info) == 0
    V = torch.triu(A)                                   # the factor as it was stored
    Vh = V.cpu().numpy().astype(np.longdouble)
    b = Vh.T @ (Vh @ x.cpu().numpy().astype(np.longdouble))
    bd = b.astype(np.float64)
    sol = torch.as_tensor(bd, device="cuda").clone()
    _lib.check(L.qmll_cholesky_solve_f64(ops._ptr(A), F, F, ops._ptr(work), ops._ptr(sol), ops._stream()), "qmll_cholesky_solve_f64")
    got = sol.cpu().numpy().astype(np.longdouble)
    residual = Vh.T @ (Vh @ got) - bd.astype(np.longdouble)
    # of either size 0.10 sqrt(F) eps, where one running sum per row or column gave 0.17
    assert np.linalg.norm(residual) <= 0.13 * F ** 0.5 * 2.0 ** -53 * np.linalg.norm(b)


@pytest.mark.parametrize("F", [704, 706])
def test_no_memory_for_the_padded_copy(monkeypatch, F):
    """A matrix that may be used up is factored in place where there is room for the workspace but not for a copy beside it, whichever of
    the two is asked for first."""
    from qml_lightning_amd import ops
    A, b = problem(F, F)
    kept = A.clone()
    n = (F + 127) // 128 * 128
    real, left = torch.empty, [8 * n * n + 1024]            # the copy alone fits, and so does the workspace

    def empty(*args, **kwargs):
        out = real(*args, **kwargs)
        left[0] -= out.numel() * out.element_size()
        if left[0] < 0:
            left[0] += out.numel() * out.element_size()
            raise torch.cuda.OutOfMemoryError("planted")
        return out
    monkeypatch.setattr(torch, "empty", empty)
    x, info = ops.cholesky_solve_spd(A, b, overwrite_a=True)
    assert int(info) == 0 and x.shape == b.shape
    assert ((kept @ x - b).abs() <= 0.75 * (F + 1) * 2.0 ** -53 * (kept.abs() @ x.abs())).all()
