"""Training rows without those of padded slots: the rows that remain, Z^T Z and Z^T y equal those of the full rows, which
other tests pin to the fp64 oracle."""
import numpy as np
import pytest
import torch

from tests import helpers
from tests.test_gpu_kernels import close
from tests.test_gpu_model import build_rff_model, build_sorf_model

pytestmark = pytest.mark.gpu


def molecules(sizes, seed):
    """One molecule per size; a negative size -k is k atoms on a line, whose angles are degenerate."""
    rng = np.random.default_rng(seed)
    X, Q = [], []
    for k in sizes:
        if k < 0:
            axis = rng.normal(size=3)
            x = np.arange(-k)[:, None] * 1.2 * axis / np.linalg.norm(axis)
        else:
            x = helpers.random_geometry(rng, k, 1.7 * k ** (1 / 3) + 1.0, 0.95)
        X.append(x.astype(np.float32))
        Q.append(np.array(([6, 1, 8, 1, 1] * 20)[:abs(k)]))
    return X, Q, rng


@pytest.mark.parametrize("kind", ["sorf", "rff"])
@pytest.mark.parametrize("npcas", [64, 128])
@pytest.mark.parametrize("sizes,periodic", [((1, 2, -3, 3, 5), False), ((22, 23, 24, 7), False), ((29, -4, 1), False),
                                            ((9, 9, 9), False), ((11, 1, 6), True)])
def test_rows_left_out_change_nothing(kind, npcas, sizes, periodic):
    species = [1, 6, 8]
    X, Q, rng = molecules(sizes, 4)
    m = (build_sorf_model(species, npcas, 3) if kind == "sorf" else build_rff_model(species, npcas, 1))
    m = m[0] if isinstance(m, tuple) else m
    E, F = rng.normal(size=len(X)), [rng.normal(size=(len(q), 3)) for q in Q]
    kw = {}
    if periodic:
        cells = np.broadcast_to(np.eye(3) * 7.0, (len(X), 3, 3)).copy()
        kw = {"cells": cells, "inv_cells": np.linalg.inv(cells)}
    data = m.format_data(X, Q, E=E, F=F, **kw)
    full, y = m._batch_rows(data, True), m._targets(data, len(X), True, True)
    proj, targets = m._training_batch(data, True, True)
    rows = m._rows_from_projected(proj, True)
    # a row does not depend on which others there are: bit for bit, and fp64 sums of at most 300 rows in another order
    real = np.concatenate([np.arange(len(X))] + [len(X) + 3 * max(map(abs, sizes)) * i + np.arange(3 * abs(k)) for i, k in enumerate(sizes)])
    assert torch.equal(rows, full[real.tolist()]) and torch.equal(targets, y[real.tolist()])
    close(rows.T @ rows, (full.T @ full).cpu().numpy(), 1e-13, "Z^T Z")
    # forces alone: the energy rows stay as zeros
    m.nbatch_train = 3
    ztz, zty = m.build_Z_components(X, Q, E=None, F=F, print_info=False, **kw)
    G, yf = full[len(X):], y[len(X):]
    close(ztz, (G.T @ G).cpu().numpy(), 1e-13, "G^T G")
    close(zty, (G.T @ yf).cpu().numpy(), 1e-12, "G^T y")
