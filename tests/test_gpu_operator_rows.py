"""What the operator sequence does in few launches: the search for the atoms of all elements, and cosine features written
per molecule, against plain torch."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def dev():
    return torch.device("cuda:0")


@pytest.mark.parametrize("nslots", [1, 255, 256, 257, 5000])
@pytest.mark.parametrize("elements", [[1], [1, 6, 8], [8, 1, 6, 7, 9], list(range(1, 33)), list(range(1, 35)), [1, 6, 1]])
def test_rows_of_elements(nslots, elements):
    """One element, other orders, as many as the native search takes and more, an element listed twice."""
    from qml_lightning_amd.models.hadamard_features import element_rows
    rng = np.random.default_rng(nslots)
    Z = torch.tensor(rng.choice([0, 1, 6, 7, 16], nslots).reshape(1, -1), dtype=torch.float32, device=dev())
    rows, counts = element_rows(Z, torch.tensor(elements, dtype=torch.float32, device=dev()), torch.tensor(elements))
    want = [torch.nonzero(Z.view(-1) == e)[:, 0] for e in elements]
    assert counts == [len(w) for w in want]
    assert torch.equal(rows.long(), torch.cat(want))


def test_charges_are_truncated_in_their_own_type():
    """A float64 charge just below a whole one, which rounds up to it in float32, is the lower element's."""
    from qml_lightning_amd.models.hadamard_features import element_rows
    Z = torch.tensor([[6.0, 6.0 - 1e-9, 7.0 - 1e-9, 1.5, 0.0]], dtype=torch.float64, device=dev())
    rows, counts = element_rows(Z, torch.tensor([1.0, 5.0, 6.0], device=dev()), torch.tensor([1, 5, 6]))
    assert counts == [1, 1, 2] and rows.tolist() == [3, 1, 0, 2]


def test_species_elsewhere():
    """The list of elements need not be where the charges are."""
    from qml_lightning_amd.models.hadamard_features import element_rows
    Z = torch.tensor([[6.0, 1.0, 8.0, 1.0]], device=dev())
    rows, counts = element_rows(Z, torch.tensor([1.0, 6.0]), torch.tensor([1, 6]))
    assert counts == [2, 1] and rows.tolist() == [1, 3, 0]


def test_no_slots():
    from qml_lightning_amd.models.hadamard_features import element_rows
    rows, counts = element_rows(torch.zeros(0, 4, device=dev()), torch.tensor([1.0, 6.0], device=dev()), torch.tensor([1, 6]))
    assert counts == [0, 0] and rows.numel() == 0


@pytest.mark.parametrize("A,F,nmol,order", [(1, 4, 1, "up"), (7, 260, 5, "up"), (40, 64, 900, "up"), (300, 33, 3, "up"), (300, 128, 40, "mixed"),
                                            (300, 128, 40, "out"), (300, 128, 40, "below"), (16383, 8, 700, "up"), (16384, 8, 700, "up"),
                                            (16385, 8, 700, "up"), (16385, 8, 700, "mixed"), (16385, 8, 700, "below"), (600, 4096, 2050, "up")])
def test_cos_features_of_molecules(A, F, nmol, order):
    """Molecules without atoms, one and several columns per thread, the table by one workgroup and by many, and an index that is not
    ascending or leaves the range (its atoms are left out)."""
    gen = torch.Generator(device=dev()).manual_seed(A + F)
    c = torch.randn(A, F, device=dev(), generator=gen) * 2
    b = torch.rand(F, device=dev(), generator=gen) * 6
    idx = torch.randint(0, nmol, (A,), device=dev(), generator=gen)
    if order == "up":
        idx = idx.sort()[0]
    if order == "out":
        idx[::7] = nmol
    if order == "below":
        idx = idx.sort()[0]
        idx[::7] = -5                                      # and behind each a valid one, whose entries begin at 0
    torch.full((nmol, F), float("nan"), device=dev())              # what the result's memory may hold
    got = torch.ops.qml_lightning_sorf.get_cos_features(c, b, torch.tensor(nmol), idx.int())
    ok = (idx >= 0) & (idx < nmol)
    want = torch.zeros(nmol, F, device=dev(), dtype=torch.float64)
    want.index_add_(0, idx[ok], np.sqrt(2.0 / F) * torch.cos(c[ok].double() + b.double()))
    most = torch.bincount(idx[ok]).max().item()
    # 3.7e-7 of a cosine, a rounding per sum
    assert (got.double() - want).abs().max().item() < np.sqrt(2.0 / F) * most * (4e-7 + most * 6e-8)


def test_traced_model_on_other_batches():
    """torch.jit.trace records the search, not what it found in the example's batch."""
    from qml_lightning_amd.models.hadamard_features import HadamardFeaturesModel
    from qml_lightning_amd.representations.FCHL import FCHLCuda
    from tests import helpers
    elements = np.array([1, 6, 8])
    np.random.seed(0)
    m = HadamardFeaturesModel(rep=FCHLCuda(species=elements), elements=elements, ntransforms=1, sigma=2.0, npcas=32, nstacks=4, fused=False)
    gen = torch.Generator(device=dev()).manual_seed(1)
    m.reductors = torch.randn(m.reductors.shape, device=dev(), generator=gen) * 0.1
    m.alpha = torch.randn(m.nfeatures(), device=dev(), dtype=torch.float64, generator=gen)
    keys = ("charges", "atomIDs", "molIDs", "natom_counts", "cells", "inv_cells")

    def batch(seed):
        rng = np.random.default_rng(seed)
        X = np.stack([helpers.random_geometry(rng, 9, 5.0, 0.9) for _ in range(6)])
        Q = rng.choice(elements, (6, 9))
        Q[:, :3] = elements                                # (an element that the example lacks stays out of the trace)
        data = m.format_data(X, Q)
        return data["coordinates"].requires_grad_(True), [data[k] for k in keys]

    class Energies(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.model = m

        def forward(self, X, *rest):
            return self.model.forward(X, *rest)

    X, rest = batch(0)
    traced = torch.jit.trace(Energies(), (X, *rest), check_trace=False)
    for seed in (0, 1, 2):
        X, rest = batch(seed)
        got, want = traced(X, *rest), m.forward(X, *rest)
        assert torch.equal(got, want)
        g, w = (torch.autograd.grad(e.sum(), X)[0] for e in (got, want))
        assert (g - w).abs().max().item() <= 1e-5 * w.abs().max().item()       # forces are summed by atomics
