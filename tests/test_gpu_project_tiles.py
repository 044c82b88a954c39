"""Projections on the half-precision matrix cores at the edges of their tiles (64 rows for few atoms, 128 for more) and of the chunks
of the contraction."""
import pytest
import torch

from qml_lightning_amd import ops
from tests.test_gpu_kernels import close, dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R", [4, 28, 32, 36, 64, 100])        # one chunk of 32 entries, cut and whole; two; an odd number
@pytest.mark.parametrize("A", [4500, 33000])                   # tiles of 64 rows, of 128
@pytest.mark.parametrize("d", [128, 256])
def test_edges_of_tiles_and_chunks(R, A, d):
    g = torch.Generator(device=dev()).manual_seed(A + R)
    counts = [1, 63, 64, 65, 0, 127, 128, 129]
    counts.append(A - 37 - sum(counts))                        # and 37 rows of unknown elements
    ne = len(counts)
    types = torch.repeat_interleave(torch.arange(ne + 1, device=dev()), torch.tensor(counts + [37], device=dev()))
    types = types[torch.randperm(A, device=dev(), generator=g)].int()
    ss, off = ops.sort_by_type(types, torch.arange(A, device=dev(), dtype=torch.int32), ne)
    real, order = A - 37, ss.long()
    rep, gx = torch.randn(A, R, device=dev(), generator=g), torch.randn(A, d, device=dev(), generator=g)
    red = torch.randn(ne, R, d, device=dev(), generator=g) / R ** 0.5
    U = red.double()
    x, g_rep = ops.project_typed(rep, ss, off, red), ops.project_typed_backward(gx, ss, off, red, types, A)
    want, back = torch.empty(real, d, dtype=torch.float64, device=dev()), torch.zeros(A, R, dtype=torch.float64, device=dev())
    at = off.tolist()
    for t in range(ne):
        part = slice(at[t], at[t + 1])
        want[part] = rep[order[part]].double() @ U[t]
        back[order[part]] = gx[part].double() @ U[t].T.contiguous()
    # operands to 2^-23 of their binade, fp32 sums of at most 256 products: a few 2^-22 of the largest entry
    close(x[:real], want.cpu().numpy(), 2e-6, "x")
    close(g_rep, back.cpu().numpy(), 2e-6, "g_rep")
    assert (g_rep[types == ne] == 0).all()


@pytest.mark.parametrize("A", [4500, 33000])
def test_a_row_that_is_not_finite_stays_alone(A):
    """An infinity at a row's last entry, which lanes beyond the end of the row and of the tile read as well."""
    g = torch.Generator(device=dev()).manual_seed(A)
    R, d = 100, 128
    types = torch.zeros(A, dtype=torch.int32, device=dev())
    ss, off = ops.sort_by_type(types, torch.arange(A, device=dev(), dtype=torch.int32), 1)
    rep, red = torch.randn(A, R, device=dev(), generator=g), torch.randn(1, R, d, device=dev(), generator=g)
    clean = ops.project_typed(rep, ss, off, red)
    rep[A - 1, R - 1] = float("inf")
    x = ops.project_typed(rep, ss, off, red)
    # the rows beside it may take another power of two
    close(x[:A - 1], clean[:A - 1].double().cpu().numpy(), 2e-6, "the other rows")
    assert not torch.isfinite(x[A - 1]).any()
