"""The chained diagonal recurrence (several steps per launch on row tiles with halos, the default on
SELL matrices) against the oracle and against single steps (a pinned step variant) on every element
layout: each scalar type and column width, the three matrix forms (one hopping value, a value table,
stored values), rows of 0 to 19 entries, ragged tiles, step counts with every remainder of the steps
per launch, site orders with small and large halos.  Runs are long enough (150 moments) that the
dispatch takes the chain for its plan's cost; shorter ones check that they do not need it.

Tolerances: the repository's parity bounds, 1e-10 (fp64, complex128) and 1e-4 (fp32, complex64) of
mu_0 against the oracle; twice that between two device forms."""
import numpy as np
import pytest
import scipy.sparse as sp

import abi
from pybinding_amd import generators

pytestmark = pytest.mark.gpu

TOL = {np.float64: 1e-10, np.complex128: 1e-10, np.float32: 1e-4, np.complex64: 1e-4}


def hilbert(h, n1, n2):
    inv = np.argsort(generators.honeycomb_cell_order(n1, n2))
    h = h[inv][:, inv].tocsr()
    h.sort_indices()
    return h


def scaled(h, dtype):
    h = (h * (2 / 10.0)).astype(dtype)
    h.sort_indices()
    return h


def lattice(form, n1=40, n2=24, dtype=np.float64):
    """honeycomb supercell with one hopping value, with three of them, or all different"""
    h = hilbert(generators.honeycomb_supercell(n1, n2, disorder=0.7, seed=4), n1, n2)
    rng = np.random.default_rng(8)
    if form != "uniform":
        up = sp.triu(h, 1).tocsr()
        up.data *= rng.choice([0.8, 1.0, 1.1], up.nnz) if form == "table" else rng.uniform(0.7, 1.1, up.nnz)
        phase = np.exp(1j * up.data) if np.dtype(dtype).kind == "c" and form == "stored" else 1
        up.data = up.data * phase
        h = (up + up.conj().T + sp.diags(h.diagonal())).tocsr()
    return scaled(h, dtype)


def starters(n, nvec, dtype, seed=3):
    rng = np.random.default_rng(seed)
    if np.dtype(dtype).kind == "c":
        return np.exp(2j * np.pi * rng.random((nvec, n))).astype(dtype)
    return (2 * rng.integers(0, 2, (nvec, n)) - 1).astype(dtype)


def run(h2, r0, moments, single=False):
    ctx = abi.Ctx(0)
    try:
        mat, blk = ctx.mat(h2, fmt=1), ctx.block(r0)
        if single:
            ctx.set_tile_width(h2.dtype, 64)
        return abi.moments_diagonal(mat, blk, moments)
    finally:
        ctx.close()


def check(oracle, h2, r0, moments):
    dtype = h2.dtype.type
    mu, ref = run(h2, r0, moments), oracle.diag_moments(h2, r0, moments)
    scale = np.abs(ref[:, :1])
    assert np.max(np.abs(mu - ref) / scale) <= TOL[dtype]
    single = run(h2, r0, moments, single=True)
    # in 32 bits both forms hold the same vectors (sums in double): at most the last rounding differs
    assert np.max(np.abs(mu - single) / scale) <= (2 * TOL[dtype] if TOL[dtype] < 1e-6 else 2.0 ** -22)


@pytest.mark.parametrize("dtype", [np.float64, np.float32, np.complex128, np.complex64])
@pytest.mark.parametrize("form", ["uniform", "table", "stored"])
@pytest.mark.parametrize("nvec", [1, 2, 3, 7, 16, 24])
def test_layouts(oracle, dtype, form, nvec):
    h2 = lattice(form, dtype=dtype)
    print("chain", np.dtype(dtype).name, form, nvec, flush=True)
    check(oracle, h2, starters(h2.shape[0], nvec, dtype), 158)


@pytest.mark.parametrize("moments", [2, 24, 150, 152, 154, 156, 158, 160, 162, 164, 166, 168, 170, 172])
def test_step_counts(oracle, moments):
    h2 = lattice("uniform", 17, 9)
    print("chain steps", moments, flush=True)
    check(oracle, h2, starters(h2.shape[0], 4, np.float64), moments)


@pytest.mark.parametrize("n1,n2", [(4, 4), (8, 4), (11, 3), (64, 32), (90, 70)])
def test_sizes(oracle, n1, n2):
    """one tile that holds the whole system, ragged last tiles, several tiles per CU"""
    h2 = lattice("uniform", n1, n2)
    print("chain size", h2.shape[0], flush=True)
    check(oracle, h2, starters(h2.shape[0], 5, np.float64), 150)


@pytest.mark.parametrize("dtype,n1,n2,nvec", [(np.float64, 64, 32, 33), (np.float64, 90, 70, 20), (np.complex128, 64, 32, 18),
                                              (np.float32, 90, 70, 64), (np.complex64, 24, 40, 40)])
def test_column_groups(oracle, dtype, n1, n2, nvec):
    """column groups side by side in one launch, all at once or in turns of which the last has fewer"""
    h2 = lattice("uniform", n1, n2, dtype)
    print("chain groups", np.dtype(dtype).name, h2.shape[0], nvec, flush=True)
    check(oracle, h2, starters(h2.shape[0], nvec, dtype), 158)


@pytest.mark.parametrize("dtype", [np.float64, np.float32, np.complex128])
@pytest.mark.parametrize("width", [5, 8, 19])
def test_long_rows(oracle, dtype, width):
    """rows of up to `width` off-diagonal entries near the diagonal, some rows empty"""
    n = 1500
    rng = np.random.default_rng(width)
    up = sp.random(n, n, density=0.0, format="lil")
    for d in range(1, width // 2 + 1):
        v = rng.uniform(0.1, 0.3, n - d) * (rng.random(n - d) < 0.9)
        v[700:720] = 0
        up += sp.diags(v, d, shape=(n, n))
    up = sp.csr_matrix(up)
    up.eliminate_zeros()
    h = (up + up.T).tocsr()
    h2 = (h * (2 / abs(h).sum(axis=1).max())).astype(dtype)  # a scaled Hamiltonian: spectrum in [-2, 2]
    h2.sort_indices()
    print("chain width", width, np.dtype(dtype).name, flush=True)
    check(oracle, h2, starters(n, 6, dtype), 154)


def test_orders(oracle):
    """row-major and random site orders (halos too large for a chain: single steps) agree"""
    n1, n2 = 96, 80
    h = generators.honeycomb_supercell(n1, n2, disorder=0.7, seed=4)
    r0 = starters(h.shape[0], 4, np.float64)
    for q in (np.arange(h.shape[0]), np.random.default_rng(1).permutation(h.shape[0])):
        h2 = scaled(h[q][:, q].tocsr(), np.float64)
        print("chain order", q[:3], flush=True)
        check(oracle, h2, np.ascontiguousarray(r0[:, q]), 150)


def test_repeats_and_graph_replays_are_bitwise():
    h2 = lattice("table")
    r0 = starters(h2.shape[0], 9, np.float64)
    ctx = abi.Ctx(0)
    try:
        mat, blk = ctx.mat(h2, fmt=1), ctx.block(r0)
        first = abi.moments_diagonal(mat, blk, 166)
        assert np.array_equal(abi.moments_diagonal(mat, blk, 166), first)
        ctx.set_graph_policy(2)
        for _ in range(3):
            assert np.array_equal(abi.moments_diagonal(mat, blk, 166), first)
            other = ctx.block(starters(h2.shape[0], 3, np.float64, seed=9))
            abi.moments_diagonal(mat, other, 10)
            other.close()
    finally:
        ctx.close()


@pytest.mark.parametrize("dtype", [np.float64, np.float32, np.complex128])
@pytest.mark.parametrize("form", ["uniform", "table", "stored"])
@pytest.mark.parametrize("nvec", [1, 2, 3, 4, 10])
def test_batches(oracle, dtype, form, nvec):
    """systems of 2 to 4140 sites in one batch, each with its own hopping values: the chained form
    (graph and stream launches) against the oracle and the walkers (a pinned partition)"""
    h2s = [lattice(form, n1, n2, dtype=dtype) * dtype(f) for n1, n2, f in
           ((1, 1, 1), (4, 2, 0.9), (8, 4, 0.8), (11, 3, 0.7), (19, 17, 1), (46, 45, 0.6))]
    r0 = [starters(h.shape[0], nvec, dtype, seed=i) for i, h in enumerate(h2s)]
    M = 130
    print("chain batch", np.dtype(dtype).name, form, nvec, flush=True)
    ctx = abi.Ctx(0)
    try:
        b = abi.Batch(ctx, h2s)
        b.starters(np.concatenate(r0, axis=1))
        out = {}
        for mode in (False, True, True):
            b.run(M, mode)
            out.setdefault("chain", b.fetch(M))
            assert np.array_equal(b.fetch(M), out["chain"])
        b.set_partition(64)
        b.run(M, False)
        out["walkers"] = b.fetch(M)
    finally:
        ctx.close()
    for s, (h, r) in enumerate(zip(h2s, r0)):
        ref = oracle.diag_moments(h, r, M)
        scale = np.abs(ref[:, :1])
        assert np.max(np.abs(out["chain"][s] - ref) / scale) <= TOL[dtype], s
        assert np.max(np.abs(out["chain"][s] - out["walkers"][s]) / scale) <= 2 * TOL[dtype], s


def pinned(ctx, dtype):
    ctx.set_tile_width(dtype, 64)  # turns the chained form off


@pytest.mark.parametrize("dtype", [np.float64, np.float32, np.complex128, np.complex64])
@pytest.mark.parametrize("form", ["uniform", "table", "stored"])
def test_dots_and_marks(oracle, dtype, form):
    """<beta|op T_n|alpha> and (T_n alpha)[dest] on one vector: against the oracle and single steps"""
    h2 = lattice(form, dtype=dtype)
    n, M = h2.shape[0], 163
    rng = np.random.default_rng(2)
    alpha = starters(n, 3, dtype)[1:2]
    beta = rng.standard_normal(n).astype(dtype) * dtype(1 if np.dtype(dtype).kind != "c" else 1 + 0.5j)
    op = sp.diags([rng.uniform(0.5, 1.5, n), rng.uniform(0.5, 1.5, n - 7)], [0, 7]).tocsr().astype(dtype)
    dest = [0, 5, n - 1, n // 2, 5]
    print("chain dots", np.dtype(dtype).name, form, flush=True)
    ctx = abi.Ctx(0)
    try:
        mat, blk = ctx.mat(h2, fmt=1), ctx.block(alpha)
        out = [(abi.moments_generic(mat, blk, M, beta, o), abi.moments_multi_unit(mat, blk, M, dest)) for o in (None, op)]
        pinned(ctx, dtype)
        single = [(abi.moments_generic(mat, blk, M, beta, o), abi.moments_multi_unit(mat, blk, M, dest)) for o in (None, op)]
    finally:
        ctx.close()
    norm = np.linalg.norm(alpha) * np.linalg.norm(beta) * 2
    for (mu, units), (mu1, units1), o in zip(out, single, (None, op)):
        ref = oracle.offdiag_moments(h2, alpha[0], M, "generic", beta=beta, op=o)
        assert np.max(np.abs(mu - ref)) <= TOL[dtype] * norm
        assert np.max(np.abs(mu - mu1)) <= 2 * TOL[dtype] * norm
        ref = oracle.offdiag_moments(h2, alpha[0], M, "multi_unit", dest=dest)
        assert np.max(np.abs(units - ref)) <= TOL[dtype] * np.linalg.norm(alpha)
        assert np.max(np.abs(units - units1)) <= 2 * TOL[dtype] * np.linalg.norm(alpha)


@pytest.mark.parametrize("dtype", [np.float64, np.float32, np.complex128, np.complex64])
@pytest.mark.parametrize("nvec", [1, 2, 4, 9])
def test_kubo_panels(dtype, nvec):
    """the panels of the Kubo moments from chained sweeps (the right operator applied inside them) against
    single steps, with operators of the Hamiltonian's pattern, of more neighbours than it has (outside the
    first ring: single steps) and with longer rows"""
    h2 = lattice("stored", 24, 20, dtype=dtype)
    n, M = h2.shape[0], 90
    x = np.random.default_rng(5).uniform(-1, 1, n)
    v = h2.copy()
    v.data = (h2.data * (np.repeat(x, np.diff(h2.indptr)) - x[h2.indices])).astype(dtype)
    far = sp.csr_matrix((v @ v).astype(dtype))
    local = (v + sp.diags(x).astype(dtype)).tocsr().astype(dtype)
    for left, right in ((v, v), (v, far), (far, local)):
        left.sort_indices()
        right.sort_indices()
        print("chain kubo", np.dtype(dtype).name, nvec, right.nnz, flush=True)
        ctx = abi.Ctx(0)
        try:
            mat, vl, vr = ctx.mat(h2, fmt=1), ctx.mat(left, fmt=1), ctx.mat(right, fmt=1)
            blk = ctx.block(starters(n, nvec, dtype))
            mu = abi.kubo_moments(mat, vl, vr, blk, M)
            pinned(ctx, dtype)
            ref = abi.kubo_moments(mat, vl, vr, blk, M)
        finally:
            ctx.close()
        assert np.max(np.abs(mu - ref)) <= 2 * TOL[dtype] * np.max(np.abs(ref))


@pytest.mark.parametrize("dtype", [np.float64, np.float32, np.complex64])
@pytest.mark.parametrize("form", ["uniform", "stored"])
def test_row_order(oracle, dtype, form):
    """tiles in another row order than the matrix's (kpmx_mat_set_row_order): diagonal moments, dots and
    marked rows of a randomly ordered matrix whose tiles follow the lattice"""
    h = lattice(form, dtype=dtype)
    n, M = h.shape[0], 162
    q = np.random.default_rng(6).permutation(n)  # row i of the shuffled matrix is lattice row q[i]
    h2 = h[q][:, q].tocsr()
    h2.sort_indices()
    r0 = starters(n, 5, dtype)
    one = np.ascontiguousarray(r0[:1])
    beta, dest = starters(n, 1, dtype, seed=8)[0], [0, 3, n - 1]
    print("chain row order", np.dtype(dtype).name, form, flush=True)
    ctx = abi.Ctx(0)
    try:
        mat, blk, blk1 = ctx.mat(h2, fmt=1), ctx.block(r0), ctx.block(one)
        with pytest.raises(RuntimeError, match="not a permutation"):
            mat.set_row_order(np.zeros(n, dtype=np.int32))
        calls = (lambda: abi.moments_diagonal(mat, blk, M), lambda: abi.moments_generic(mat, blk1, M, beta),
                 lambda: abi.moments_multi_unit(mat, blk1, M, dest))
        single = [f() for f in calls]
        mat.set_row_order(q)
        out = [f() for f in calls]
        mat.set_row_order(None)
        assert all(np.array_equal(f(), s) for f, s in zip(calls, single))
    finally:
        ctx.close()
    ref = oracle.diag_moments(h2, r0, M)
    assert np.max(np.abs(out[0] - ref) / np.abs(ref[:, :1])) <= TOL[dtype]
    for a, b, scale in zip(out, single, (n, n, 1)):
        assert np.max(np.abs(a - b)) <= scale * (2 * TOL[dtype] if TOL[dtype] < 1e-6 else 2.0 ** -20)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("form", ["uniform", "stored"])
@pytest.mark.parametrize("nvec,checkpoint", [(1, 16), (3, 2), (8, 3), (9, 64), (16, 74), (16, 73), (20, 37), (33, 16), (5, 0)])
def test_adjoint(form, dtype, nvec, checkpoint):
    """Forward and backward passes in launches of several steps against single steps, with the
    checkpoints near the ends of the run.  Tolerance: 75 steps forward and back that round
    differently in fp64, 75 x 4 x 2^-53 < 1e-13 and a hundredfold for what cancels; in fp32 the
    vectors are equal and only double sums are taken in another order."""
    h2 = lattice(form, dtype=dtype)
    moments = 150
    w = np.random.default_rng(6).standard_normal(moments)
    out = []
    for single in (False, True):
        ctx = abi.Ctx(0)
        mat, blk = ctx.mat(h2, fmt=1), ctx.block(starters(h2.shape[0], nvec, dtype))
        if single:
            ctx.set_tile_width(dtype, 64)
        print("chain adjoint", np.dtype(dtype).name, form, nvec, checkpoint, single, flush=True)
        out.append(abi.adjoint_diagonal(mat, blk, moments, w, checkpoint))
        ctx.close()
    (grad, mu), (ref, mu_ref) = out
    assert np.max(np.abs(grad - ref)) <= 1e-11 * np.max(np.abs(ref))
    scale = np.abs(mu_ref[:, :1])
    assert np.max(np.abs(mu - mu_ref) / scale) <= (1e-11 if dtype == np.float64 else 2.0 ** -22)
