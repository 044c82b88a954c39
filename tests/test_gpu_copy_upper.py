"""The copy of a symmetric matrix that the Cholesky solve works in: tiles of 128 x 128 on or above the diagonal, nothing else."""
import numpy as np
import pytest
import torch

from qml_lightning_amd import ops

pytestmark = pytest.mark.gpu


# one tile and its edges; odd sizes, odd row strides on either side and starts off 16 bytes take the way without pairs
@pytest.mark.parametrize("F,lda,ldu,oa,ou", [(1, 1, 2, 0, 0), (127, 128, 130, 0, 0), (128, 128, 128, 0, 0), (129, 130, 132, 0, 0),
                                             (300, 301, 300, 0, 0), (300, 300, 301, 0, 0), (300, 300, 300, 1, 0),
                                             (384, 384, 384, 0, 1), (385, 500, 386, 1, 1)])
def test_upper_tiles_are_copied_and_nothing_else_is_written(F, lda, ldu, oa, ou):
    A = torch.randn(oa + F * lda, dtype=torch.float64, device="cuda")
    U = torch.full((ou + F * ldu + 5,), 7.0, dtype=torch.float64, device="cuda")
    ops.check(ops._lib.lib().qmll_copy_upper_f64(ops._ptr(A[oa:]), lda, F, ops._ptr(U[ou:]), ldu, ops._stream()), "copy")
    want = torch.full_like(U, 7.0).cpu()
    rows = torch.arange(F) // 128
    upper = rows[None, :] >= rows[:, None]
    block = want[ou:ou + F * ldu].view(F, ldu)[:, :F]
    block[upper] = A[oa:].cpu().view(F, lda)[:, :F][upper]
    assert torch.equal(U.cpu(), want)


# a kept matrix in a wider buffer, also with an odd row stride; NaN in the tiles below the diagonal is never looked at
@pytest.mark.parametrize("F,W,at", [(300, 300, 0), (300, 700, 100), (300, 701, 3), (640, 643, 1)])
def test_solve_that_keeps_a_strided_matrix(F, W, at):
    rng = np.random.default_rng(F + W)
    Z = rng.normal(size=(2 * F, F))
    A = Z.T @ Z
    b = rng.normal(size=(F, 1))
    tile = np.arange(F) // 128
    held = np.where(tile[None, :] >= tile[:, None], A, np.nan)
    big = torch.full((F, W), 5.0, dtype=torch.float64, device="cuda")
    big[:, at:at + F] = torch.tensor(held, device="cuda")
    keep = big.clone()
    x, info = ops.cholesky_solve_spd(big[:, at:at + F], torch.tensor(b, device="cuda"))
    assert int(info.item()) == 0
    assert torch.equal(torch.nan_to_num(big, nan=-1.0), torch.nan_to_num(keep, nan=-1.0))
    # Cholesky is backward stable: |A x - b| <= c F^2 eps |A| |x|, entry by entry in norms (Higham, theorem 10.4; c of a few)
    got = x.cpu().numpy().reshape(F, 1)
    bound = 8 * F * F * np.finfo(np.float64).eps * np.abs(A).max() * np.abs(got).max()
    assert np.abs(A @ got - b).max() <= bound
