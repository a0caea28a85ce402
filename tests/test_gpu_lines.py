"""Colour steps that share a launch (classes that differ in x alone by whole grid
lines, classes that differ in z alone by whole columns) give the bits of the
oracle's steps: lines shorter and longer than a wave, up to and past a
workgroup, columns up to and past a workgroup's planes, odd extents (which take
the steps apart), blocks with padding, kappa, every precision; V-cycles into
vectors that hold NaN; and solves, whose r.z partials then come from a pass of
their own, against the same solve with explicit columns."""
import numpy as np
import pytest

from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

GRIDS = [(10, 40, 40), (26, 26, 26), (40, 26, 30), (62, 14, 18), (64, 20, 14), (66, 16, 18), (96, 16, 12), (130, 10, 14),
         (200, 8, 12), (256, 8, 10), (258, 6, 8), (510, 6, 8), (512, 6, 8), (514, 6, 8), (34, 34, 13), (33, 34, 14),
         (34, 33, 14), (20, 6, 128), (20, 6, 130), (4, 18, 254)]


@pytest.mark.parametrize("dims", GRIDS)
@pytest.mark.parametrize("op", ["hpcg", "kappa"])
def test_steps_bitexact(hip, dims, op):
    n = int(np.prod(dims))
    levels = 2 if all(d % 2 == 0 for d in dims) else 1
    g = np.random.default_rng(n)
    kappa = np.exp(0.5 * g.standard_normal(n)) if op == "kappa" else None
    ctx = hip.Context(0)
    ctx.generate(*dims, levels=levels, kappa=kappa)
    P = po.Problem(*dims, levels=levels, kappa=kappa)
    x, r = g.random(n) - 0.5, g.random(n) - 0.5
    dr, dx = ctx.vec(0, r), ctx.vec(0, x)
    ctx.symgs(0, dr, dx)
    np.testing.assert_array_equal(dx.download(), P.symgs(r, x))
    nan = ctx.vec(0, np.full(n, np.nan))
    ctx.mg(0, dr, nan)
    np.testing.assert_array_equal(nan.download(), P.mg(r))
    for prec, name in ((hip.HPCGX_PREC_FP32, "mg_f32"), (hip.HPCGX_PREC_FP16, "mg_f16")):
        ctx.prepare(prec)
        ctx.mg_mixed(prec, dr, dx)
        np.testing.assert_array_equal(dx.download(), getattr(P, name)(r.astype(np.float32)).astype(np.float64))


@pytest.mark.parametrize("dims", [(26, 26, 26), (66, 16, 18), (130, 10, 14), (34, 34, 14)])
def test_solve_matches_steps_apart(hip, dims):
    n = int(np.prod(dims))
    out = []
    for fmt in (hip.HPCGX_COLS_COMPACT, hip.HPCGX_COLS_EXPLICIT):
        ctx = hip.Context(0)
        ctx.generate(*dims, levels=2)
        ctx.set_column_format(fmt)
        b, x = ctx.vec(0, np.random.default_rng(5).random(n)), ctx.vec(0)
        out.append((ctx.cg(b, x, max_iter=10, history=True)["hist"], x.download()))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    np.testing.assert_array_equal(out[0][1], out[1][1])
