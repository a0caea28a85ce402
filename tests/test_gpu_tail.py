"""The one-workgroup tail of the V-cycle gives the bits of the oracle's
level-by-level V-cycle: on grids at and around its row limit (8192 padded
rows), entered at level 0 or at a coarse level, on one-slice and padded
levels, in every precision, and for a smoothing step alone (general rows:
test_gpu_general)."""
import numpy as np
import pytest

from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

GRIDS = [((2, 2, 2), 1), ((4, 4, 4), 2), ((8, 8, 8), 4), ((16, 16, 16), 4), ((24, 8, 16), 3), ((24, 16, 16), 2),
         ((32, 16, 16), 4), ((20, 20, 20), 2), ((32, 24, 16), 4), ((40, 24, 16), 4), ((5, 7, 9), 1), ((6, 10, 14), 2)]


@pytest.mark.parametrize("dims,levels", GRIDS)
@pytest.mark.parametrize("kappa", [False, True])
def test_tail_bitexact(hip, dims, levels, kappa):
    n = int(np.prod(dims))
    g = np.random.default_rng(n)
    k = np.exp(0.5 * g.standard_normal(n)) if kappa else None
    ctx = hip.Context(0)
    ctx.generate(*dims, levels=levels, kappa=k)
    P = po.Problem(*dims, levels=levels, kappa=k)
    x, r = g.random(n) - 0.5, g.random(n) - 0.5
    for fmt in (hip.HPCGX_COLS_COMPACT, hip.HPCGX_COLS_EXPLICIT):
        ctx.set_column_format(fmt)
        dr, dx = ctx.vec(0, r), ctx.vec(0, x)
        ctx.symgs(0, dr, dx)
        np.testing.assert_array_equal(dx.download(), P.symgs(r, x))
        ctx.mg(0, dr, dx)
        np.testing.assert_array_equal(dx.download(), P.mg(r))
        for prec, name in ((hip.HPCGX_PREC_FP32, "mg_f32"), (hip.HPCGX_PREC_FP16, "mg_f16")):
            ctx.prepare(prec)
            ctx.mg_mixed(prec, dr, dx)
            np.testing.assert_array_equal(dx.download(), getattr(P, name)(r.astype(np.float32)).astype(np.float64))
