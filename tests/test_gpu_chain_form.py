"""The inputs of test_gpu_chain.py run in the form that they are there for: the chained one, except for
runs too short to pay for a plan, systems of fewer than 64 rows and large systems without compact tiles.
Diagonal runs are asked for their form (one-vector collections and Kubo panels use the plans of blocks of
their width); batches and gradients have no such question, but sum in another order than single steps,
which shows in the last bits of their float64 results."""
import numpy as np
import pytest

import abi
from pybinding_amd import generators
from test_gpu_chain import lattice, scaled, starters

pytestmark = pytest.mark.gpu


def steps(h2, nvec, moments):
    ctx = abi.Ctx(0)
    try:
        return abi.diagonal_form(ctx.mat(h2, fmt=1), nvec, moments)[0]
    finally:
        ctx.close()


@pytest.mark.parametrize("dtype", [np.float64, np.float32, np.complex128, np.complex64])
@pytest.mark.parametrize("form", ["uniform", "table", "stored"])
def test_layouts(dtype, form):
    h2 = lattice(form, dtype=dtype)
    for nvec in (1, 2, 3, 7, 16, 24):
        print("form of", np.dtype(dtype).name, form, nvec, flush=True)
        assert steps(h2, nvec, 158) > 1, nvec
    assert steps(h2, 1, 2 * 162) > 1  # dots and marked rows


def test_lengths_sizes_and_orders():
    for moments in range(150, 174, 2):
        assert steps(lattice("uniform", 17, 9), 4, moments) > 1, moments
    for moments in (2, 24):
        assert steps(lattice("uniform", 17, 9), 4, moments) == 1
    for n1, n2 in ((8, 4), (11, 3), (64, 32), (90, 70)):
        assert steps(lattice("uniform", n1, n2), 5, 150) > 1, (n1, n2)
    assert steps(lattice("uniform", 4, 4), 5, 150) == 1  # 32 rows
    for dtype, n1, n2, nvec in ((np.float64, 64, 32, 33), (np.float64, 90, 70, 20), (np.complex128, 64, 32, 18),
                                (np.float32, 90, 70, 64), (np.complex64, 24, 40, 40)):
        assert steps(lattice("uniform", n1, n2, dtype), nvec, 158) > 1, (dtype, n1, n2, nvec)
    # random order: a tile of a small system still holds the rows within a few steps; of 205 k rows, tiles
    # have 130 or more, a distance of two 10 times as many, and 8 columns fit 900
    for n1, n2, nvec, chained in ((96, 80, 4, True), (512, 200, 8, False)):
        h = generators.honeycomb_supercell(n1, n2, disorder=0.7, seed=4)
        q = np.random.default_rng(1).permutation(h.shape[0])
        assert (steps(scaled(h[q][:, q].tocsr(), np.float64), nvec, 1030) > 1) == chained


@pytest.mark.parametrize("form", ["uniform", "table", "stored"])
def test_batches(form):
    h2s = [lattice(form, n1, n2) * f for n1, n2, f in ((8, 4, 0.8), (19, 17, 1), (46, 45, 0.6))]
    n = sum(h.shape[0] for h in h2s)
    for nvec in (1, 4, 10):
        print("batch form of", form, nvec, flush=True)
        ctx = abi.Ctx(0)
        b = abi.Batch(ctx, h2s)
        b.starters(np.random.default_rng(3).standard_normal((nvec, n)))
        b.run(130, False)
        chained = b.fetch(130)
        b.set_partition(64)
        b.run(130, False)
        assert not np.array_equal(chained, b.fetch(130))
        ctx.close()


@pytest.mark.parametrize("nvec,checkpoint", [(1, 16), (9, 64), (16, 74), (16, 73), (20, 37), (33, 37), (3, 0)])
def test_gradients(nvec, checkpoint):
    """forward and backward each: a tape of the chained form run backward in single steps and the reverse"""
    h2 = lattice("stored")
    r0, moments = np.random.default_rng(4).standard_normal((nvec, h2.shape[0])), 150
    w = np.random.default_rng(6).standard_normal(moments)

    def run(forward_single, backward_single):
        ctx = abi.Ctx(0)
        mat, blk = ctx.mat(h2, fmt=1), ctx.block(r0)
        if forward_single:
            ctx.set_tile_width(np.float64, 64)
        tape = abi.Tape(mat, blk, moments, checkpoint)
        if backward_single:
            ctx.set_tile_width(np.float64, 64)
        grad = tape.backward(w)
        tape.close()
        ctx.close()
        return grad

    print("gradient form of", nvec, checkpoint, flush=True)
    single, backward = run(True, True), run(False, True)
    if checkpoint:  # tapes that keep every vector are made in single steps
        assert not np.array_equal(single, backward)
    assert not np.array_equal(backward, run(False, False))
