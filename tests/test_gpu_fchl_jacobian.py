"""The explicit Jacobian with one to four wavefronts per atom, with and without the table of triples."""
import numpy as np
import pytest
import torch

from oracle import fchl19
from tests.test_gpu_kernels import REL_REP, close, gpu_prm, make_batch, oracle_prm, t32, ti32

pytestmark = pytest.mark.gpu


# wavefronts that the launch takes: 4, 4, 4, 3, 2, 4 (no table), 1 (the rows of one wavefront fill what LDS there is)
@pytest.mark.parametrize("n,elements", [(1, 1), (2, 2), (12, 2), (29, 4), (29, 5), (45, 3), (6, 10)])
@pytest.mark.parametrize("with_list", [False, True])
def test_wavefronts_per_atom(monkeypatch, n, elements, with_list):
    from qml_lightning_amd import ops
    rng = np.random.default_rng(n + elements)
    species = [1, 6, 7, 8, 9, 14, 15, 16, 17, 35][:elements]
    sites = np.stack(np.unravel_index(rng.permutation(64)[:n], (4, 4, 4)), 1) * 1.6
    coords = [sites[:k] + rng.uniform(-0.3, 0.3, (k, 3)) for k in (n, max(1, n // 2))]
    X, Z, aid, mid, nat = make_batch(coords, [rng.choice(species, len(c)) for c in coords])
    prm = oracle_prm(species, rcut=4.0)             # (some atoms are no neighbours)
    cnt, nl = fchl19.neighbours(X, nat, prm.rcut)
    ty = fchl19.element_types(Z, nat, prm.species)
    args = (t32(X), ti32(ty), None, None, ti32(aid), ti32(mid), ti32(nat), t32(prm.Rs2), t32(prm.Rs3), gpu_prm(prm))
    lists = dict(nlist=ti32(nl), nneigh=ti32(cnt)) if with_list else {}
    rep, jac = ops.fchl_jacobian(*args, **lists)
    close(rep, fchl19.forward(X, ty, aid, mid, nl, cnt, prm), REL_REP, "rep")
    close(jac, fchl19.jacobian(X, ty, aid, mid, nl, cnt, prm), REL_REP, "jacobian")
    # every row of a listed atom, whatever the arrays held
    monkeypatch.setattr(torch, "empty", lambda *a, **k: torch.full(*a, float("nan"), **k))
    rep2, jac2 = ops.fchl_jacobian(*args, **lists, zero_fill=False)
    at = (torch.from_numpy(mid).long(), torch.from_numpy(aid).long())
    assert torch.equal(rep2[at], rep[at]) and torch.equal(jac2[at], jac[at])
