"""Preparation of a large batch, whose first workgroups count the types of the listed atoms for the sort."""
import numpy as np
import pytest
import torch

from qml_lightning_amd import ops
from tests.test_gpu_kernels import dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model_list", [None, [8.0, 1.0], [6.0, 9.0, 1.0]])
@pytest.mark.parametrize("listed", [4097, 8192, 20000])        # a cut workgroup of 256 atoms, whole ones, more than slots / 256
@pytest.mark.parametrize("shuffled", [False, True])
def test_equals_the_separate_kernels(listed, model_list, shuffled):
    rng = np.random.default_rng(listed)
    n = 23
    nmol = listed // 8
    counts = rng.integers(1, n + 1, size=nmol).astype(np.int32)
    Z = np.where(np.arange(n)[None] < counts[:, None], rng.choice([1.0, 6.0, 8.0, 7.0], size=(nmol, n)), 0.0)       # 7: in no list
    atoms = np.concatenate([np.arange(c) for c in counts])
    mols = np.repeat(np.arange(nmol), counts)
    order = rng.permutation(len(atoms)) if shuffled else np.arange(len(atoms))
    order = order[:listed]
    t = lambda a, kind: torch.tensor(a, device=dev(), dtype=kind)       # noqa: E731
    ai, mi = t(atoms[order], torch.int32), t(mols[order], torch.int32)
    Zt, ct = t(Z, torch.float32), t(counts, torch.int32)
    species = t([1.0, 6.0, 8.0], torch.float32)
    msp = t(model_list, torch.float32) if model_list else None
    types, stypes, ss, off, zero = ops.prepare_batch(Zt, ct, species, ai, mi, msp, 4 * nmol * n)
    X = torch.zeros(nmol, n, 3, device=dev())
    assert torch.equal(types, ops.element_types(X, Zt, ct, species))
    want = ops.element_types(X, Zt, ct, msp) if model_list else types
    assert torch.equal(stypes, want)
    want_ss, want_off = ops.sort_atoms_by_type(want, ai, mi, n, len(model_list or [1, 6, 8]))
    assert torch.equal(off, want_off)
    assert torch.equal(ss[:int(off[-1])], want_ss[:int(off[-1])])
    assert not zero.any()
