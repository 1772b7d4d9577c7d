"""Objects that a chained run leaves something with (plans, captured graphs) used again under other
conditions: the results are those of a fresh object, bit for bit."""
import numpy as np
import pytest

import abi
from pybinding_amd import generators
from pybinding_amd.batch import kpm_batch
from test_gpu_chain import lattice, starters

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,counts", [(np.float64, (20, 32, 17)), (np.complex128, (9, 16)), (np.float32, (33, 64)),
                                          (np.float64, (1, 4, 3, 1))])
def test_batch_with_other_vector_counts(dtype, counts):
    """the replayed graph of a batch belongs to its number of vectors (more of them than before fill the
    same padded block)"""
    hs = [generators.square_flake(60, 70, disorder=1.0, seed=1, dtype=dtype),
          generators.square_flake(31, 44, disorder=1.0, seed=2, dtype=dtype)]
    ranges, M = [(-4.6, 4.6)] * 2, 130

    def fresh(nvec):
        kb = kpm_batch(hs, ranges)
        mu = kb.moments(M, nvec, use_graph=False)
        kb.close()
        return mu

    kb = kpm_batch(hs, ranges)
    for nvec in counts:
        print("batch of", nvec, np.dtype(dtype).name, flush=True)
        ref = fresh(nvec)
        for repeat in range(3):
            assert np.array_equal(kb.moments(M, nvec), ref)
    kb.set_tile_width(16)  # column tiles: 20 vectors in tiles of 16 and 4, then 30 in 16 and 14
    for nvec in (20, 30):
        tiled = kb.moments(M, nvec, use_graph=False)
        for repeat in range(2):
            assert np.array_equal(kb.moments(M, nvec), tiled)
    kb.close()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_row_order_between_graph_replays(dtype):
    """a row order frees the plans that a captured run reads: the next run is captured anew"""
    h = lattice("uniform", dtype=dtype)
    q = np.random.default_rng(6).permutation(h.shape[0])
    h2 = h[q][:, q].tocsr()
    h2.sort_indices()
    r0, M = starters(h.shape[0], 5, dtype), 162

    def fresh(order):
        ctx = abi.Ctx(0)
        mat = ctx.mat(h2, fmt=1)
        if order is not None:
            mat.set_row_order(order)
        mu = abi.moments_diagonal(mat, ctx.block(r0), M)
        ctx.close()
        return mu

    ctx = abi.Ctx(0)
    ctx.set_graph_policy(2)
    mat, blk = ctx.mat(h2, fmt=1), ctx.block(r0)
    other = h.shape[0] - 1 - q
    for i, order in enumerate((None, q, other, None, q)):
        print("row order", np.dtype(dtype).name, None if order is None else order[:3], flush=True)
        if i:
            mat.set_row_order(order)
        ref = fresh(order)
        for repeat in range(3):
            assert np.array_equal(abi.moments_diagonal(mat, blk, M), ref)
    ctx.close()
