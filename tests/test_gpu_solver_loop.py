"""The solver loop's shortcuts leave its results alone: V-cycles replayed from a
recorded graph, V-cycles launched before the norm is known, totals written to
pinned memory.  A solve in which they run is compared, bit for bit, with the
same context's first solve after the graph was dropped and with a fresh
context, on repeats with eager work in between, and after the matrix, the format
and the stream have changed under a recorded graph.  Sizes on both sides of the
tail's 8192 rows."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

GRIDS = [(16, 16, 16), (32, 32, 16), (40, 24, 32), (64, 48, 32)]


def _context(hip, dims, kappa):
    ctx = hip.Context(0)
    ctx.generate(*dims, levels=3, kappa=kappa)
    ctx.prepare(hip.HPCGX_PREC_FP32)
    ctx.prepare(hip.HPCGX_PREC_FP16)
    return ctx


def _solve(hip, ctx, variant, tol, iters=12):
    n = ctx.info(0)["n"]
    b, x = ctx.vec(0, np.random.default_rng(3).random(n) - 0.5), ctx.vec(0)
    out = ctx.cg(b, x, max_iter=iters, tol=tol, variant=variant, history=True)
    got = out["hist"], x.download()
    b.free()
    x.free()
    return got


def _equal(a, b):
    np.testing.assert_array_equal(a[0], b[0])
    np.testing.assert_array_equal(a[1], b[1])


@pytest.mark.parametrize("dims", GRIDS)
@pytest.mark.parametrize("tol", [0.0, 1e-30, 1e-4])
@pytest.mark.parametrize("op", ["hpcg", "kappa"])
def test_solves_repeat(hip, dims, tol, op):
    n = int(np.prod(dims))
    kappa = np.exp(0.5 * np.random.default_rng(1).standard_normal(n)) if op == "kappa" else None
    ctx = _context(hip, dims, kappa)
    for variant in (hip.HPCGX_CG_FP64, hip.HPCGX_CG_MIXED_FP32, hip.HPCGX_CG_MIXED_FP16):
        first = _solve(hip, ctx, variant, tol)
        r = ctx.vec(0, np.random.default_rng(4).random(n))
        z = ctx.vec(0)
        for _ in range(3):
            ctx.mg(0, r, z)  # eager work on the same levels
            ctx.dot(r, z)
            _equal(_solve(hip, ctx, variant, tol), first)
        _equal(_solve(hip, _context(hip, dims, kappa), variant, tol), first)


def test_two_iterations_then_more(hip):
    """A solve too short to record, then one that records, then one that replays."""
    a, b = _context(hip, (40, 24, 32), None), _context(hip, (40, 24, 32), None)
    for iters in (1, 2, 9, 9):
        _equal(_solve(hip, a, hip.HPCGX_CG_FP64, 0.0, iters), _solve(hip, b, hip.HPCGX_CG_FP64, 0.0, iters))


def test_changes_under_a_recorded_graph(hip):
    dims = (40, 24, 32)
    n = int(np.prod(dims))
    variants = (hip.HPCGX_CG_FP64, hip.HPCGX_CG_MIXED_FP32, hip.HPCGX_CG_MIXED_FP16)
    used = _context(hip, dims, None)
    for v in variants:
        _solve(hip, used, v, 0.0)
    stream = torch.cuda.Stream()
    d = 26.0 + np.random.default_rng(2).random(n)

    def diagonal(ctx):
        ctx.set_diagonal(0, d)

    def explicit(ctx):
        ctx.set_column_format(hip.HPCGX_COLS_EXPLICIT)

    def other_stream(ctx):
        ctx.set_stream(stream.cuda_stream)

    def other_problem(ctx):
        ctx.generate(48, 32, 24, levels=3, kappa=np.linspace(1.0, 2.0, 48 * 32 * 24))
        ctx.prepare(hip.HPCGX_PREC_FP32)
        ctx.prepare(hip.HPCGX_PREC_FP16)

    done = []
    for change in (diagonal, explicit, other_stream, other_problem):
        done.append(change)
        change(used)
        fresh = _context(hip, dims, None)
        for c in done:
            c(fresh)
        for v in variants:
            want = _solve(hip, fresh, v, 0.0)
            _equal(_solve(hip, used, v, 0.0), want)
            _equal(_solve(hip, used, v, 0.0), want)


def test_dot_answers(hip):
    """Totals that are NaN, infinite and zero reach the host too."""
    ctx = hip.Context(0)
    ctx.generate(24, 16, 16, levels=1)
    n = ctx.info(0)["n"]
    x = np.random.default_rng(6).random(n)
    for bad, want in ((np.nan, np.isnan), (np.inf, np.isposinf), (0.0, lambda v: v > 0)):
        y = x.copy()
        y[n // 2] = bad
        dx, dy, dw = ctx.vec(0, x), ctx.vec(0, y), ctx.vec(0)
        assert want(ctx.dot(dx, dy))
        assert want(ctx.waxpby_dot(1.0, dy, 0.0, dx, dw))
        assert want(ctx.dot_noalloc(dx, dy))
    zero = ctx.vec(0)
    assert ctx.dot(zero, zero) == 0.0
