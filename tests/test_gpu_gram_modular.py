"""Z^T Z from exact integer products (csrc/gram_modular.hip) against sums in extended precision and against the fp64 kernel."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def dev():
    return torch.device("cuda:0")


def modular(Z, y=None, start=0.0):
    from qml_lightning_amd import _lib
    from qml_lightning_amd.ops import _ptr, _stream
    L = _lib.lib()
    M, F = Z.shape
    C = torch.full((F, F), start, dtype=torch.float64, device=dev())
    zy = torch.full((F,), start, dtype=torch.float64, device=dev()) if y is not None else None
    n = int(L.qmll_gram_modular_workspace_bytes(max(M, 768), F))     # what more rows need is enough for fewer
    ws = torch.full((n,), 77, dtype=torch.uint8, device=dev())        # whatever the workspace holds must not matter
    rc = L.qmll_gram_modular_f64(_ptr(Z), _ptr(y), M, F, _ptr(C), _ptr(zy), _ptr(ws), n, _stream())
    assert rc == 0, _lib.last_error()
    return C, zy


def fp64_kernel(Z, start=0.0):
    from qml_lightning_amd import _lib
    from qml_lightning_amd.ops import _ptr, _stream
    M, F = Z.shape
    C = torch.full((F, F), start, dtype=torch.float64, device=dev())
    rc = _lib.lib().qmll_gram_upper_f64(_ptr(Z), None, M, F, _ptr(C), None, _stream())
    assert rc == 0, _lib.last_error()
    return C


def upper(F):
    t = torch.arange(F) // 128
    return (t[:, None] <= t[None, :]).numpy()


def within_norms(C, Z, what):
    """Every entry within what the rounding of the columns to norm 2^53 .. 2^54 gives: the sum over the rows of independent
    errors of at most half a unit against the other column is normal with a standard deviation of 2^-53 sqrt(2/12) of the
    product of the norms at most; eight of these, and the rounding of the reference's and the result's own 53 bits."""
    ref = (Z.astype(np.longdouble).T @ Z.astype(np.longdouble))
    norm = np.sqrt(np.diagonal(ref))
    bound = 8 * 2.0 ** -53 * np.sqrt(2 / 12) * norm[:, None] * norm[None, :] + 2.0 ** -52 * np.abs(ref)
    off = np.abs(C - ref) / np.maximum(bound, np.finfo(np.longdouble).tiny)
    assert (off[upper(Z.shape[1])] <= 1.0).all(), (what, float(off[upper(Z.shape[1])].max()))


# one tile and less, one column more than a tile, several tiles, row counts around the stage of 64 and the pair of 128 rows,
# row ranges (few tiles, many rows)
@pytest.mark.parametrize("M,F", [(1, 5), (63, 24), (64, 256), (129, 257), (768, 300), (1000, 600), (4100, 130)])
def test_modular_gram_against_extended_precision(M, F):
    rng = np.random.default_rng(M + F)
    Z = rng.normal(size=(M, F)) * np.exp(2.0 * rng.normal(size=F))
    y = rng.normal(size=M)
    Zd, yd = torch.tensor(Z, device=dev()), torch.tensor(y, device=dev())
    C, zy = modular(Zd, yd)
    again, zy2 = modular(Zd, yd)
    assert torch.equal(C, again) and torch.equal(zy, zy2)
    assert (C.cpu().numpy()[~upper(F)] == 0).all()
    within_norms(C.cpu().numpy(), Z, "plain")
    ref = Z.astype(np.longdouble).T @ y
    assert (np.abs(zy.cpu().numpy() - ref) <= M * 2.0 ** -53 * (np.abs(Z).T @ np.abs(y))).all()     # a sum of M products
    onto, _ = modular(Zd, yd, 3.0)
    assert (onto.cpu().numpy()[~upper(F)] == 3.0).all()
    assert np.abs(onto.cpu().numpy() - 3.0 - C.cpu().numpy())[upper(F)].max() <= 2.0 ** -52 * (3.0 + C.abs().max().item())


def test_modular_gram_of_uneven_columns():
    """Columns of zeros, of one dominating entry (whose residues need their quotient corrected), of very small and very large
    numbers, of exact integers."""
    rng = np.random.default_rng(5)
    M, F = 900, 140
    Z = rng.normal(size=(M, F))
    Z[:, 3] = 0.0
    Z[:, 10:20] = 0.0
    Z[7, 10:20] = rng.normal(size=10)                    # one entry only
    Z[5, 20:40] *= 2.0 ** np.arange(20, 60, 2)           # one entry far above the others
    Z[:, 40:50] *= 1e-95
    Z[:, 50:60] *= 1e130
    Z[:, 60:70] = rng.integers(-40, 40, (M, 10))
    Z[:, 70:80] = 1.0                                    # equal entries
    Z[:, 80] = -Z[:, 81]
    C, _ = modular(torch.tensor(Z, device=dev()))
    C = C.cpu().numpy()
    within_norms(C, Z, "uneven")
    assert (C[3] == 0).all() and (C[:, 3] == 0).all()
    ints = np.r_[60:80]
    assert np.array_equal(C[np.ix_(ints, ints)], Z[:, ints].T @ Z[:, ints])      # whole numbers stay whole


@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf"), 1e160, 1e-170])
def test_columns_that_cannot_be_scaled_take_the_fp64_kernel(value):
    """NaN, infinities, squares that overflow or vanish: decided on the device, the result is the fp64 kernel's."""
    g = torch.Generator(device="cpu").manual_seed(11)
    Z = torch.randn(800, 384, dtype=torch.float64, generator=g).to(dev())
    if value == 1e-170:
        Z[:, 200] = 0.0
    Z[123, 200] = value
    C, _ = modular(Z, start=1.0)
    assert torch.equal(torch.nan_to_num(C, nan=0.5), torch.nan_to_num(fp64_kernel(Z, 1.0), nan=0.5))
    assert torch.equal(C.isnan(), fp64_kernel(Z, 1.0).isnan())


def uneven_rows(kind):
    """Rows whose columns have their large entries in different rows."""
    rng = np.random.default_rng(17)
    M, F = 800, 256
    Z = rng.normal(size=(M, F))
    if kind.startswith("lognormal"):
        return Z * np.exp(float(kind.split()[1]) * rng.normal(size=(M, F)))
    if kind == "own row":                         # one large entry per column, each in another row
        Z[np.arange(F), np.arange(F)] *= 1e6
        return Z
    Z[:M // 2, :F // 2] *= 1e-9                   # two halves of the columns, each large where the other is small
    Z[M // 2:, F // 2:] *= 1e-9
    return Z


@pytest.mark.parametrize("kind", ["lognormal 3", "lognormal 5", "own row", "halves"])
def test_gram_holds_the_bound_of_fp64_sums_entry_by_entry(kind):
    """A caller who has not said that the columns' norms are the measure gets every entry within M 2^-53 of the sum of its
    products' magnitudes (a sum of M products in any order: (M - 1) additions and one rounding of each product)."""
    from qml_lightning_amd import ops
    Z = uneven_rows(kind)
    M, F = Z.shape
    C = torch.zeros(F, F, dtype=torch.float64, device=dev())
    ops.gram(torch.tensor(Z, device=dev()), None, C, None)
    Zl = Z.astype(np.longdouble)
    off = np.abs(C.cpu().numpy() - Zl.T @ Zl) / (np.abs(Zl).T @ np.abs(Zl))
    assert off.max() <= M * 2.0 ** -53, (kind, float(off.max()))


@pytest.mark.parametrize("features", ["sorf", "rff"])
@pytest.mark.parametrize("with_energies,with_forces", [(True, True), (False, True), (True, False)])
def test_training_rows_lose_nothing_entry_by_entry(features, with_energies, with_forces):
    """What training relies on in saying so: on its rows the root mean square over the entries of the error relative to the sum of the
    products' magnitudes is no larger than that of the fp64 kernel, and none exceeds the bound of fp64 sums."""
    from qml_lightning_amd.models.hadamard_features import HadamardFeaturesModel
    from qml_lightning_amd.models.random_features import RandomFourrierFeaturesModel
    from qml_lightning_amd.representations.FCHL import FCHLCuda
    rng = np.random.default_rng(31)
    np.random.seed(31)
    elements = np.array([1, 6, 8])
    nmol = 60 if with_forces else 800
    counts = rng.integers(3, 10, nmol)
    grid = np.stack(np.meshgrid(*[np.arange(3)] * 3, indexing="ij"), -1).reshape(-1, 3) * 1.6
    X = [grid[rng.permutation(27)[:k]] + rng.uniform(-0.3, 0.3, (k, 3)) for k in counts]
    Q = [rng.choice(elements, k) for k in counts]
    E = rng.normal(size=nmol) if with_energies else None
    Fo = [rng.normal(size=(k, 3)) for k in counts] if with_forces else None
    cls = HadamardFeaturesModel if features == "sorf" else RandomFourrierFeaturesModel
    m = cls(rep=FCHLCuda(species=elements), elements=elements, sigma=2.0, llambda=1e-5, npcas=64, nstacks=8, nbatch_train=nmol)
    q, _ = torch.linalg.qr(torch.randn(3, m.rep.get_repsize(), 64, dtype=torch.float64, generator=torch.Generator().manual_seed(1)))
    m.reductors = q.float().contiguous().to(dev())
    data = m.format_data(X, Q, E=E, F=Fo)
    proj, _ = m._training_batch(data, with_energies, with_forces)
    rows = m._rows_from_projected(proj, with_forces, zero_energy_rows=not with_energies).contiguous()
    M, F = rows.shape
    assert M >= 768 and F == 512
    Z = rows.cpu().numpy().astype(np.longdouble)
    ref, mag = Z.T @ Z, np.abs(Z).T @ np.abs(Z)
    fp64 = fp64_kernel(rows).cpu().numpy()
    got = m.build_Z_components(X, Q, E=E, F=Fo, print_info=False)[0].cpu().numpy()
    u = upper(F)

    def errors(C):
        d = (np.abs(C - ref) / mag)[u].astype(np.float64)
        return np.sqrt((d * d).mean()), d.max()
    print(features, with_energies, with_forces, M, "rms, max: modular %.2e %.2e, fp64 %.2e %.2e" % (errors(got) + errors(fp64)))
    assert errors(got)[0] <= errors(fp64)[0]
    assert errors(got)[1] <= M * 2.0 ** -53


def test_modular_gram_in_a_graph_is_the_eager_result():
    g = torch.Generator(device="cpu").manual_seed(2)
    Z = torch.randn(1100, 300, dtype=torch.float64, generator=g).to(dev())
    from qml_lightning_amd import ops
    C = torch.zeros(300, 300, dtype=torch.float64, device=dev())
    ops.gram(Z, None, C, None, within_norms=True)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        ops.gram(Z, None, C.zero_(), None, within_norms=True)
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        C.zero_()
        ops.gram(Z, None, C, None, within_norms=True)
    for seed in range(3):
        Z.copy_(torch.randn(1100, 300, dtype=torch.float64, generator=g))
        graph.replay()
        torch.cuda.synchronize()
        ref = torch.zeros_like(C)
        ops.gram(Z, None, ref, None, within_norms=True)
        torch.cuda.synchronize()
        assert torch.equal(C, ref), seed


# below and above the row count from which the fp64 kernel takes a workspace of its own
@pytest.mark.parametrize("M,F", [(800, 300), (2100, 520)])
def test_gram_without_memory_for_its_workspace(monkeypatch, M, F):
    """Where the workspace of the integer products does not fit, the fp64 sums are taken, added to what is there, mirrored or not."""
    from qml_lightning_amd import ops
    g = torch.Generator(device="cpu").manual_seed(M)
    Z, y = torch.randn(M, F, dtype=torch.float64, generator=g).to(dev()), torch.randn(M, 1, dtype=torch.float64, generator=g).to(dev())

    def both(mirror, **kwargs):
        C, zy = torch.full((F, F), 2.0, dtype=torch.float64, device=dev()), torch.ones(F, 1, dtype=torch.float64, device=dev())
        ops.gram(Z, y, C, zy, mirror=mirror, **kwargs)
        return C, zy
    expect = [both(mirror) for mirror in (True, False)]
    real, refused = torch.empty, []

    def empty(*args, **kwargs):
        if kwargs.get("dtype") is torch.uint8:
            refused.append(args)
            raise torch.cuda.OutOfMemoryError("planted")
        return real(*args, **kwargs)
    monkeypatch.setattr(torch, "empty", empty)
    for mirror, (C, zy) in zip((True, False), expect):
        got, got_y = both(mirror, within_norms=True)
        assert torch.equal(got, C), mirror
        # Z^T y is added with atomics, 1 + M terms in any order: two such sums differ by twice the bound of either
        assert ((got_y - zy).abs() <= 2 * (M + 1) * 2.0 ** -53 * (1 + Z.abs().T @ y.abs())).all()
    assert len(refused) == 2


# 7168 features: the smallest matrix with a slab (3072 rows); 7296: its columns end within a tile of 256; 12288: 8192 rows;
# 19456: two slabs, of 12288 and 3072 rows
@pytest.mark.parametrize("F", [7168, 7296, 12288, 19456])
def test_factorisation_in_slabs(F):
    """The residual of the solve within the backward error of a factorisation of that size, the factor, and that of the general path (no
    workspace for slabs), in the measure of the diagonal, a pivot that is not positive and a NaN below the slab reported."""
    from qml_lightning_amd import _lib, ops
    L = _lib.lib()
    g = torch.Generator(device=dev()).manual_seed(9)
    Z = torch.randn(F + 300, F, dtype=torch.float64, device=dev(), generator=g) * 0.01
    Z *= torch.exp(torch.randn(F, dtype=torch.float64, device=dev(), generator=g))
    A = torch.zeros(F, F, dtype=torch.float64, device=dev())
    ops.gram(Z, None, A, None)
    del Z
    A.diagonal().add_(1e-3)
    b = torch.randn(F, 1, dtype=torch.float64, device=dev(), generator=g)
    assert L.qmll_cholesky_slabs_bytes(F) > 0 and L.qmll_cholesky_slabs_bytes(F - 1) == 0 and L.qmll_cholesky_slabs_bytes(7040) == 0
    x, info = ops.cholesky_solve_spd(A, b)
    assert int(info.item()) == 0
    # |A x - b| <= c n eps |A| |x| (a backward stable solve; c = 1 is far from what a random matrix shows)
    assert float((A @ x - b).norm()) <= F * 2.0 ** -53 * float(A.norm()) * float(x.norm())
    # fp64 sums: |U^T U - A| <= (n + 1) eps |U^T||U| entry by entry, and that is at most sqrt(a_ii a_jj) (Higham, theorem 10.3); the
    # integer products err by 2^-57 sqrt(n) sqrt(a_ii a_jj) at most
    work = torch.empty(int(L.qmll_cholesky_workspace_bytes(F)) // 8 + 1, dtype=torch.float64, device=dev())
    slabs = torch.empty(int(L.qmll_cholesky_slabs_bytes(F)), dtype=torch.uint8, device=dev())
    rows = torch.arange(0, F, 997, device=dev())
    scale = A.diagonal()[rows, None].sqrt() * A.diagonal()[None, :].sqrt()
    for s in (slabs, None):
        U = A.clone()
        info.zero_()
        ops.check(L.qmll_cholesky_slabs_f64(ops._ptr(U), F, F, ops._ptr(work), ops._ptr(s), ops._ptr(info), ops._stream()), "chol")
        assert int(info.item()) == 0
        U.triu_()
        assert float(((U[:, rows].T @ U - A[rows]).abs() / scale).max()) <= 2 * (F + 1) * 2.0 ** -53
        del U
    for row, col, value, expect in ((F - 2000, F - 2000, -1.0, F - 1999), (1000, F - 1500, float("nan"), None)):
        kept = A[row, col].item()
        A[row, col] = value
        A[col, row] = value
        _, info = ops.cholesky_solve_spd(A, b)
        assert int(info.item()) == expect if expect else int(info.item()) > 0
        A[row, col] = kept
        A[col, row] = kept


def test_solve_of_graded_systems_in_fp64_sums():
    """Columns that are coupled to one row each and otherwise only by 1e-8, and a right side over ten decades: with fp64 sums asked
    for, the residual stays entry by entry within that theorem's bound for a solve, (3 n + 1) 2^-53 |U|^T |U| |x|."""
    from qml_lightning_amd import ops
    F, n = 7168, 3000
    g = torch.Generator(device=dev()).manual_seed(1)
    A = torch.randn(F, F, dtype=torch.float64, device=dev(), generator=g) * 1e-8
    A = A + A.T
    i = torch.arange(n, device=dev())
    A[i, i + 4000] += 0.5
    A[i + 4000, i] += 0.5
    A.diagonal().copy_(torch.ones(F))
    b = torch.randn(F, 1, dtype=torch.float64, device=dev(), generator=g)
    b *= torch.exp(6.0 * torch.randn(F, 1, dtype=torch.float64, device=dev(), generator=g))
    x, info = ops.cholesky_solve_spd(A, b, within_norms=False)
    assert int(info.item()) == 0
    U = torch.linalg.cholesky(A, upper=True).abs()
    bound = ((3 * F + 1) * 2.0 ** -53 * (U.T @ (U @ x.abs())))[:, 0].cpu().numpy()
    An, xn, bn = A.cpu().numpy(), x[:, 0].cpu().numpy().astype(np.longdouble), b[:, 0].cpu().numpy()
    for lo in range(0, F, 512):
        r = np.abs(bn[lo:lo + 512] - An[lo:lo + 512].astype(np.longdouble) @ xn)
        assert (r <= bound[lo:lo + 512]).all(), (lo, float((r / bound[lo:lo + 512]).max()))


def test_solve_without_memory_for_slabs(monkeypatch):
    """Where the workspace of the slabs does not fit, the solve does without it."""
    from qml_lightning_amd import ops
    F = 7168
    g = torch.Generator(device=dev()).manual_seed(4)
    Z = torch.randn(F + 300, F, dtype=torch.float64, device=dev(), generator=g)
    A = torch.zeros(F, F, dtype=torch.float64, device=dev())
    ops.gram(Z, None, A, None)
    b = torch.randn(F, 1, dtype=torch.float64, device=dev(), generator=g)
    real, refused = torch.empty, []

    def empty(*args, **kwargs):
        if kwargs.get("dtype") is torch.uint8:
            refused.append(args)
            raise torch.cuda.OutOfMemoryError("planted")
        return real(*args, **kwargs)
    monkeypatch.setattr(torch, "empty", empty)
    x, info = ops.cholesky_solve_spd(A, b)
    assert refused and int(info.item()) == 0
    assert float((A @ x - b).norm()) <= F * 2.0 ** -53 * float(A.norm()) * float(x.norm())


# one launch of rows and two; edges of tiles; a column with an infinity, which takes the fp64 kernel
@pytest.mark.parametrize("M,F", [(768, 24), (2000, 300), (70000, 130)])
@pytest.mark.parametrize("infinite", [False, True])
def test_written_is_added_to_zeros(M, F, infinite):
    """ZTZ written over whatever it holds is what adding to zeros gives, bit for bit; and so through `ops.gram`, below the
    rows that the integer products take as well."""
    from qml_lightning_amd import _lib, ops
    from qml_lightning_amd.ops import _ptr, _stream
    g = torch.Generator(device=dev()).manual_seed(F)
    Z = torch.randn(M, F, dtype=torch.float64, device=dev(), generator=g)
    if infinite:
        Z[M // 2, F // 2] = float("inf")
    want, _ = modular(Z)
    C = torch.full((F, F), float("nan"), dtype=torch.float64, device=dev())
    n = int(_lib.lib().qmll_gram_modular_workspace_bytes(M, F))
    ws = torch.empty(n, dtype=torch.uint8, device=dev())
    assert _lib.lib().qmll_gram_modular_write_f64(_ptr(Z), None, M, F, _ptr(C), None, _ptr(ws), n, _stream()) == 0, _lib.last_error()
    up = upper(F)
    np.testing.assert_array_equal(C.cpu().numpy()[up], want.cpu().numpy()[up])
    for rows in (M, 200):
        y = torch.randn(rows, dtype=torch.float64, device=dev(), generator=g)
        got = [ops.gram(Z[:rows], y, torch.full((F, F), start, dtype=torch.float64, device=dev()),
                        torch.zeros(F, 1, dtype=torch.float64, device=dev()), within_norms=True, fresh=fresh)
               for start, fresh in ((0.0, False), (float("nan"), True))]
        for a, b in zip(*got):
            np.testing.assert_array_equal(a.cpu().numpy(), b.cpu().numpy())
