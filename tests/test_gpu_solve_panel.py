"""The Cholesky factorisation's panels, whose columns follow the factorisation of a diagonal block step by step: one to four blocks in the
last panel, with and without columns beside it; the first pivot that is not positive in each block; the same bits each time."""
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


@pytest.mark.parametrize("blocks", [1, 2, 3, 4, 5, 6, 7, 8, 13])
def test_blocks_of_a_panel(blocks):
    from qml_lightning_amd import ops
    F = 128 * blocks
    A, b = problem(F, blocks)
    x, info = ops.cholesky_solve_spd(A, b)
    assert int(info) == 0
    # backward error of a Cholesky solve: at most 3 (F + 1) eps |A| |x| for each component, and far below it as a rule
    bound = 3.0 * (F + 1) * 2.0 ** -53 * (A.abs() @ x.abs())
    assert ((A @ x - b).abs() <= 0.25 * bound).all()
    again, _ = ops.cholesky_solve_spd(A, b)
    assert torch.equal(again, x)


@pytest.mark.parametrize("blocks,pivot", [(1, 77), (4, 5), (4, 130), (4, 300), (4, 511), (5, 200), (9, 640), (9, 900)])
def test_first_pivot_that_is_not_positive(blocks, pivot):
    from qml_lightning_amd import ops
    F = 128 * blocks
    A, b = problem(F, 3)
    A[pivot, pivot] = -1.0
    _, info = ops.cholesky_solve_spd(A, b)
    assert int(info) == pivot + 1
