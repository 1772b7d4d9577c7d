"""Checks of the engine's dispatch on a HIP runtime without a device (host_runtime.cpp), one per function:
which kernels a call launches, what it keeps in graphs and what it does without memory.  Results are
not looked at (no kernel runs).  `python host_dispatch.py LIBRARY NAME` runs one of them in a process of
its own, where that runtime takes the place of the real one; test_host_dispatch.py runs them all."""
import ctypes
import os
import sys
from collections import Counter

import numpy as np
import scipy.sparse as sp

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path[:0] = [os.path.dirname(HERE), HERE]

CHECKS = {}


def check(f):
    CHECKS[f.__name__] = f
    return f


class Runtime:
    def __init__(self, path):
        self.lib = ctypes.CDLL(path, mode=ctypes.RTLD_GLOBAL)
        self.lib.host_runtime_log.restype = ctypes.c_char_p
        self.lib.host_runtime_used.restype = ctypes.c_size_t

    def launches(self):
        """Kernel names and their counts since the last call."""
        return Counter(self.lib.host_runtime_log().decode().split())

    def of(self, f, *args):
        self.launches()
        f(*args)
        return self.launches()

    def captures(self):
        return self.lib.host_runtime_captures()

    def spare(self, nbytes):
        """Leaves `nbytes` of device memory (None: plenty)."""
        self.lib.host_runtime_limit(ctypes.c_size_t(self.lib.host_runtime_used() + nbytes if nbytes is not None else 8 << 30))

    def growth(self, sampled, of_all):
        """Local rows that each distance adds to a tile, in the sampled and in all tiles."""
        self.lib.host_runtime_growth(int(sampled), int(of_all))

    def cost(self, kernel, us):
        self.lib.host_runtime_cost(kernel.encode(), ctypes.c_double(us))


def chain(n, dtype=np.float64, width=2):
    """a matrix of `width` off-diagonal entries per row (a ring with neighbours at 1, 2, ...), one value"""
    rows = np.repeat(np.arange(n), width)
    step = np.tile([s for k in range(1, width // 2 + 1) for s in (k, -k)], n)
    h = sp.csr_matrix((np.full(n * width, 0.3), (rows, (rows + step) % n)), shape=(n, n)).astype(dtype)
    h.sort_indices()
    return h


def block(n, nvec, dtype=np.float64):
    return np.ones((nvec, n), dtype=dtype)


def chained(launches):
    return launches["k_chain"]


def stepped(launches):
    return sum(c for k, c in launches.items() if k.startswith("k_step"))


@check
def batch_graph_is_captured_for_its_vectors(rt):
    """A batch replays a graph only for the vectors it was captured with: each run launches every column
    group (of 8 fp64, 4 complex128 vectors)."""
    import abi
    for dtype, counts, cols in ((np.float64, (20, 32, 17, 32), 8), (np.complex128, (9, 16), 4), (np.float64, (33, 64), 8)):
        ctx = abi.Ctx(0)
        b = abi.Batch(ctx, [chain(3000, dtype), chain(5000, dtype)])
        M = 258
        runs = []
        for nvec in counts:
            b.starters(block(8000, nvec, dtype))
            plain = rt.of(b.run, M, False)
            assert chained(plain) and chained(plain) % -(-nvec // cols) == 0
            graph = rt.of(b.run, M, True)
            assert rt.of(b.run, M, True) == graph  # a replay
            runs.append((nvec, chained(graph), chained(plain)))
        assert all(g == p for _, g, p in runs), runs
        ctx.close()


@check
def batch_graph_is_captured_for_its_plan(rt):
    """1 and 4 vectors share a padded block, but not the plan: also where the partial sums of both reach
    their limit and the buffer does not grow"""
    import abi
    ctx = abi.Ctx(0)
    b = abi.Batch(ctx, [chain(150000), chain(150000)])
    M = 1 << 18
    before = rt.captures()
    for nvec in (1, 4):
        b.starters(block(300000, nvec))
        b.run(M, True)
    assert rt.captures() - before == 2
    ctx.close()


@check
def row_order_drops_captured_runs(rt):
    """A row order frees the plans that a captured run's launches read: the run is captured again"""
    import abi
    n = 6000
    ctx = abi.Ctx(0)
    ctx.set_graph_policy(2)
    mat, blk = ctx.mat(chain(n), fmt=1), ctx.block(block(n, 4))
    for i, order in enumerate((None, np.arange(n)[::-1], None)):
        if i:
            mat.set_row_order(order)
        before = rt.captures()
        for repeat in range(3):
            assert chained(rt.of(abi.moments_diagonal, mat, blk, 258))
        assert rt.captures() - before == 1, i
    ctx.close()


@check
def tuning_is_of_its_matrix_and_width(rt):
    """Where the autotuner finds the chained form slower, that matrix's blocks of that width leave it; other
    matrices and widths on the context do not"""
    import abi
    for two_step in (100, 1):  # us of an LDS two-step launch: single steps or the two-step form win
        ctx = abi.Ctx(0)
        n, M = 20000, 258
        tuned, other = ctx.mat(chain(n), fmt=1), ctx.mat(chain(n), fmt=1)
        blk, narrow = ctx.block(block(n, 16)), ctx.block(block(n, 4))
        for kernel, us in (("", 0), ("k_step", 4), ("k_step2_lds", two_step), ("k_chain", 1000)):
            rt.cost(kernel, us)
        abi.autotune_diagonal(tuned, blk)
        run = rt.of(abi.moments_diagonal, tuned, blk, M)
        assert not chained(run) and stepped(run)
        assert bool(run["k_step2_lds"]) == (two_step == 1)
        for mat, b in ((tuned, narrow), (other, blk), (other, narrow)):
            run = rt.of(abi.moments_diagonal, mat, b, M)
            assert chained(run) and not stepped(run), run
        rt.cost("k_chain", 1)
        abi.autotune_diagonal(tuned, blk)  # the next tuning decides anew
        assert chained(rt.of(abi.moments_diagonal, tuned, blk, M))
        ctx.close()


@check
def tuning_times_what_runs(rt):
    """The autotuner compares whole starter tiles: all column groups of the chained form, side by side as
    they run, and the padded columns of single steps"""
    import abi
    n, M = 3000, 514
    # 32 vectors: two column tiles a step, or four groups in one launch of 12 steps; 3: a block of 4
    for nvec, launch in ((32, 60), (3, 60)):
        ctx = abi.Ctx(0)
        ctx.set_autotune_two_step(False)
        mat, blk = ctx.mat(chain(n), fmt=1), ctx.block(block(n, nvec))
        for kernel, us in (("", 0), ("k_step", 5.5), ("k_chain", launch), ("k_chain_", 0)):
            rt.cost(kernel, us)
        abi.autotune_diagonal(mat, blk)
        steps, _ = abi.diagonal_form(mat, nvec, M)
        assert steps == 12, (nvec, steps)  # 5 us a step, against 11 and 5.5
        rt.cost("k_chain", 12 * (12 if nvec == 32 else 6))
        abi.autotune_diagonal(mat, blk)
        assert abi.diagonal_form(mat, nvec, M)[0] == 1
        ctx.close()


def flake(side=25, dtype="float64"):
    import pybinding_amd as pb
    from pybinding_amd.repository import graphene
    return pb.Model(graphene.monolayer(), pb.rectangle(side, side), *([pb.force_double_precision()] if dtype == "float64" else []))


@check
def sites_without_a_chain_decide_for_their_width_only(rt):
    """An LDOS of many sites for which no plan fits keeps the light cone, and that of one site still takes
    the chained form, in either order of the calls"""
    import pybinding_amd as pb
    rt.growth(600, 600)  # two distances exceed a tile of 8 columns, not one of a single column
    energy = np.linspace(-3, 3, 20)
    for dtype in ("float64", "float32"):
        for calls in ((1, 32, 1, 32), (32, 1, 32, 1)):
            kpm = pb.kpm(flake(dtype=dtype), energy_range=(-9, 9), silent=True)
            for sites in calls:
                run = rt.of(kpm.impl.calc_ldos_indices, energy, 0.05, list(range(100, 100 + sites)))
                assert bool(chained(run)) == (sites == 1) and bool(stepped(run)) == (sites > 1), (dtype, calls, sites, run)


@check
def memory_for_single_steps_is_enough(rt):
    """Under every limit on device memory with which a call succeeds on single steps (a pinned tile width, the
    light cone) it succeeds where the chained form is the default: plans and their vectors are given up"""
    import abi
    import pybinding_amd as pb
    n, M = 30000, 258
    h = chain(n)
    w = np.ones(M)

    def on_context(call):
        def run(single):
            ctx = abi.Ctx(0)
            try:
                if single:
                    ctx.set_tile_width(np.float64, 16)
                mats = [ctx.mat(h, fmt=1) for _ in range(3)]
                blocks = {v: ctx.block(block(n, v)) for v in (1, 4, 16)}
                call(ctx, mats, blocks)
            finally:
                ctx.close()
        return run

    def ldos(single):
        kpm = pb.kpm(model, energy_range=(-9, 9), silent=True, **(dict(site_order="bfs") if single else {}))
        kpm.impl.calc_ldos_indices(np.linspace(-3, 3, 20), 0.05, [100])
        kpm.impl.calc_greens_vector(5, [6, 7], np.linspace(-3, 3, 20), 0.05)

    model = flake(20, "float32")
    calls = {
        "diagonal": on_context(lambda c, m, b: abi.moments_diagonal(m[0], b[16], M)),
        "generic": on_context(lambda c, m, b: abi.moments_generic(m[0], b[4], M, np.ones(n))),
        "generic after diagonal": on_context(lambda c, m, b: (abi.moments_diagonal(m[0], b[1], M),
                                                              abi.moments_generic(m[0], b[4], M, np.ones(n)))),
        "multi_unit": on_context(lambda c, m, b: abi.moments_multi_unit(m[0], b[1], M, [1, 2, 3])),
        "kubo": on_context(lambda c, m, b: abi.kubo_moments(m[0], m[1], m[2], b[1], 100)),
        "gradient": on_context(lambda c, m, b: abi.adjoint_diagonal(m[0], b[16], M, w, 64)),
        "autotune": on_context(lambda c, m, b: abi.autotune_diagonal(m[0], b[4])),
        "ldos": ldos,
    }

    def fits(call, single, limit):
        rt.lib.host_runtime_limit(ctypes.c_size_t(limit))
        try:
            rt.launches()
            call(single)
            return True
        except RuntimeError as e:
            assert "hipMalloc" in str(e) or "do not fit" in str(e), e
            return False

    for name, call in calls.items():
        rt.lib.host_runtime_limit(ctypes.c_size_t(8 << 30))
        assert fits(call, True, 8 << 30) and not chained(rt.launches()), name
        assert fits(call, False, 8 << 30) and chained(rt.launches()), name
        low, high = 0, 8 << 30  # the least memory for single steps
        while high - low > 4096:
            mid = (low + high) // 2
            low, high = (low, mid) if fits(call, True, mid) else (mid, high)
        for extra in [0] + [int(2e5 * 1.35 ** k) for k in range(14)]:
            if fits(call, True, high + extra):
                assert fits(call, False, high + extra), (name, high, extra)


@check
def kubo_panels_take_the_chain_where_it_pays(rt):
    """Panels of the chain's widest rows where not many groups of small vectors run one after another, and
    of single columns for up to two vectors, for four on small systems and in fp64 on large ones; other
    groups advance all their vectors in single steps"""
    import abi
    M = 160
    for dtype, n, forms in ((np.float32, 20000, {1: 1, 2: 1, 3: 1, 8: 0, 16: 1, 64: 1}), (np.float32, 40000, {2: 1, 4: 0}),
                            (np.float64, 20000, {4: 1, 8: 1, 64: 1}), (np.float64, 5000, {64: 0}),
                            (np.float64, 60000, {2: 1, 4: 0}), (np.float64, 400000, {4: 1}),
                            (np.complex64, 40000, {2: 1, 4: 0, 8: 1}), (np.complex64, 5000, {4: 1, 32: 0}),
                            (np.complex64, 400000, {4: 0}), (np.complex128, 20000, {1: 1, 2: 1, 4: 1, 8: 1, 16: 0, 32: 0}),
                            (np.complex128, 120000, {16: 1})):
        h = chain(n, dtype)
        ctx = abi.Ctx(0)
        mat, v = ctx.mat(h, fmt=1), ctx.mat(h, fmt=1)
        for nvec, form in forms.items():
            run = rt.of(abi.kubo_moments, mat, v, v, ctx.block(block(n, nvec, dtype)), M)
            # single launches beside the chain: the left operator, and the right one on a group's last vector
            assert bool(chained(run)) == bool(form) and (stepped(run) < M) == bool(form), (dtype, n, nvec, run)
        ctx.close()


@check
def short_batch_runs_keep_the_walkers(rt):
    """A batch builds a plan for runs long enough to pay for it in their first pass, by its rows and vectors"""
    import abi
    for systems, size, nvec, forms in ((2, 500000, 8, {40: 0, 60: 1}), (2, 500000, 4, {60: 0, 100: 1}), (10, 2000, 4, {60: 0, 80: 1})):
        ctx = abi.Ctx(0)
        b = abi.Batch(ctx, [chain(size)] * systems)
        b.starters(block(size * systems, nvec))
        for M, form in forms.items():
            run = rt.of(b.run, M, False)
            assert bool(chained(run)) == bool(form), (size, nvec, M, run)
        ctx.close()


@check
def close_checkpoints_keep_single_reverse_steps(rt):
    """The backward pass leaves the chained form where its launches end at checkpoints after too few steps"""
    import abi
    n, M = 20000, 258
    for dtype, nvec, forms in ((np.float64, 16, {2: 0, 4: 0, 6: 0, 16: 1, 64: 1}), (np.float32, 16, {2: 0, 3: 0, 4: 1, 64: 1}),
                               (np.float64, 1, {2: 0, 3: 1, 64: 1}), (np.float32, 3, {2: 0, 3: 1, 64: 1})):
        ctx = abi.Ctx(0)
        mat, blk = ctx.mat(chain(n, dtype), fmt=1), ctx.block(block(n, nvec, dtype))
        for interval, form in forms.items():
            tape = abi.Tape(mat, blk, M, interval)
            run = rt.of(tape.backward, np.ones(M))
            single = sum(c for k, c in run.items() if k.startswith("k_adjoint") and "chain" not in k)
            assert bool(run["k_chain_adjoint"]) == bool(form) and (single < 5) == bool(form), (dtype, nvec, interval, run)
            tape.close()
        ctx.close()


@check
def plans_are_weighed_as_they_come_out(rt):
    """A plan whose tiles were halved and left with fewer steps per launch than its samples promised is
    taken only if it still promises to be faster than single steps (here: halos that grow by `growth` rows
    a step in a fifth of the system, between the samples)"""
    import abi
    n, M = 1000000, 1026
    h = chain(n)
    for growth, steps in ((30, 12), (300, 4), (500, 1)):
        rt.growth(30, 30)
        rt.lib.host_runtime_region(n // 5, growth)
        ctx = abi.Ctx(0)
        form = abi.diagonal_form(ctx.mat(h, fmt=1), 1, M)
        assert form[0] == steps, (growth, form)
        ctx.close()


if __name__ == "__main__":
    CHECKS[sys.argv[2]](Runtime(sys.argv[1]))
