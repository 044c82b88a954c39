"""Training rows of random Fourier features: atoms are taken in groups that share one sine and cosine per column."""
import numpy as np
import pytest

from oracle import sorf
from tests.test_gpu_kernels import close, dev, t32, ti32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("n", [5, 10, 15, 21])             # one to four blocks of 16 rows
@pytest.mark.parametrize("wide", [False, True])            # W in fp32 / fp64
def test_groups_of_atoms(d, n, wide):
    """Molecules of 0 to 9 atoms of an element (whole groups, remainders, none), two elements beside each other;
    70 columns: a cut block of columns."""
    import torch
    from qml_lightning_amd import ops
    rng = np.random.default_rng(d + n)
    F, counts = 70, [np.arange(10), np.array([3, 0, 1, 4, 0, 2, 5, 1, 8, 7])]
    nmol = len(counts[0])
    Ze, G, items = np.zeros((nmol, F)), np.zeros((nmol, n, 3, F)), []
    for k in counts[:1] if wide else counts:
        A, idx = int(k.sum()), np.repeat(np.arange(nmol), k).astype(np.int32)
        x, grad = rng.normal(size=(A, d)).astype(np.float32), rng.normal(size=(A, n, 3, d)).astype(np.float32)
        W, b = rng.normal(size=(d, F)) / 8.0, rng.uniform(0, 2 * np.pi, F)
        if not wide:
            W, b = W.astype(np.float32), b.astype(np.float32)
        W64, b64 = W.astype(np.float64), b.astype(np.float64)
        np.add.at(Ze, idx, np.sqrt(2.0 / F) * np.cos(x.astype(np.float64) @ W64 + b64))
        G += sorf.rff_derivative_features(x, grad, W64, b64, idx, nmol)
        items.append((x, grad, W, b, idx, np.concatenate([[0], np.cumsum(k)])))
    out = torch.zeros(nmol, n, 3, F, device=dev(), dtype=torch.float64)
    if wide:
        x, grad, W, b, idx, _ = items[0]
        ops.rff_derivative_features(t32(x), t32(grad), torch.tensor(W, device=dev()), torch.tensor(b, device=dev()), ti32(idx), out,
                                    molecule_major=True)
    else:
        energies = torch.empty(nmol, F, device=dev(), dtype=torch.float64)
        ops.rff_rows([(t32(x), t32(grad), t32(W), t32(b), ti32(seg)) for x, grad, W, b, _, seg in items], energies,
                     out.view(nmol * 3 * n, F), nmol, n, overwrite=True)
        close(energies, Ze, 1e-12, "energy rows")
    close(out, G, 1e-12, "force rows")          # (sums of d products of order one in fp64, as for the rows one by one)
