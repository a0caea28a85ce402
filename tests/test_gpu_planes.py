"""Grids of one plane above the size that one workgroup takes: some colour blocks
have no rows, on the finest level or on a coarse one.  Bit-exact against the
oracle, every call that sweeps."""
import numpy as np
import pytest

from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,levels", [((128, 128, 1), 1), ((128, 1, 128), 1), ((1, 128, 128), 1), ((130, 66, 1), 1),
                                         ((200, 200, 2), 2)])
@pytest.mark.parametrize("op", ["hpcg", "kappa"])
def test_empty_blocks(hip, dims, levels, op):
    n = int(np.prod(dims))
    g = np.random.default_rng(n)
    kappa = np.exp(0.5 * g.standard_normal(n)) if op == "kappa" else None
    ctx = hip.Context(0)
    ctx.generate(*dims, levels=levels, kappa=kappa)
    P = po.Problem(*dims, levels=levels, kappa=kappa)
    for l in range(levels):
        nl = ctx.info(l)["n"]
        x, r = g.random(nl) - 0.5, g.random(nl) - 0.5
        dr, dx = ctx.vec(l, r), ctx.vec(l, x)
        ctx.symgs(l, dr, dx)
        np.testing.assert_array_equal(dx.download(), P.level(l).symgs(r, x))
    r = g.random(n) - 0.5
    dr, dx = ctx.vec(0, r), ctx.vec(0, np.full(n, np.nan))
    ctx.mg(0, dr, dx)
    np.testing.assert_array_equal(dx.download(), P.mg(r))
    for prec, name in ((hip.HPCGX_PREC_FP32, "mg_f32"), (hip.HPCGX_PREC_FP16, "mg_f16")):
        ctx.prepare(prec)
        ctx.mg_mixed(prec, dr, dx)
        np.testing.assert_array_equal(dx.download(), getattr(P, name)(r.astype(np.float32)).astype(np.float64))
    out = []
    for fmt in (hip.HPCGX_COLS_COMPACT, hip.HPCGX_COLS_EXPLICIT):
        ctx.set_column_format(fmt)
        db, ds = ctx.vec(0, r), ctx.vec(0)
        out.append((ctx.cg(db, ds, max_iter=8, history=True)["hist"], ds.download()))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    np.testing.assert_array_equal(out[0][1], out[1][1])
