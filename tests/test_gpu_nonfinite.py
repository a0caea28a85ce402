"""NaN and infinities in a vector reach the rows that couple to them and no
others: every call on compact columns equals the oracle's, which goes through a row's
entries alone.  (A slot without an entry, a neighbour outside the grid, names some
other row of the level.)  Each value form, with the special entries on faces,
edges, corners and inside; grids that take row runs, lines and columns, single
steps and the tail, odd extents, padding."""
import numpy as np
import pytest

from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

GRIDS = [((16, 16, 16), 3), ((66, 16, 18), 2), ((64, 32, 20), 2), ((33, 17, 31), 1), ((128, 128, 66), 2)]


def _make(hip, dims, levels, op):
    n = int(np.prod(dims))
    kappa = None if op == "hpcg" else np.exp(0.5 * np.random.default_rng(n).standard_normal(n))
    ctx = hip.Context(0)
    ctx.generate(*dims, levels=levels, kappa=kappa)
    P = po.Problem(*dims, levels=levels, kappa=kappa)
    if op == "stored":  # the kappa matrix as rows: no field to read the values from
        up = hip.Context(0)
        for l in range(levels):
            d = tuple(v >> l for v in dims)
            f2c = None
            if l + 1 < levels:
                k, j, i = np.meshgrid(*(np.arange(v // 2) for v in d[::-1]), indexing="ij")
                f2c = ((2 * k * d[1] + 2 * j) * d[0] + 2 * i).reshape(-1).astype(np.int32)
            up.upload_level(l, d, *ctx.export_level(l), f2c)
        ctx = up
    return ctx, P


def _places(dims):
    x, y, z = dims
    mid = (x // 2, y // 2, z // 2)
    for p in [(mid[0], mid[1], 0), (mid[0], 0, mid[2]), (0, mid[1], mid[2]), (x - 1, mid[1], z - 1), (x - 1, y - 1, z - 1),
              mid]:
        yield (p[2] * y + p[1]) * x + p[0]


def _same(got, want, what):
    nan = np.isnan(want)
    np.testing.assert_array_equal(np.isnan(got), nan, err_msg=what)
    np.testing.assert_array_equal(got[~nan], want[~nan], err_msg=what)


@pytest.mark.parametrize("dims,levels", GRIDS)
@pytest.mark.parametrize("op", ["hpcg", "kappa", "stored"])
def test_stays_where_it_couples(hip, dims, levels, op):
    ctx, P = _make(hip, dims, levels, op)
    n = int(np.prod(dims))
    g = np.random.default_rng(3)
    x0, r = g.random(n) - 0.5, g.random(n) - 0.5
    dr, dx, dy = ctx.vec(0, r), ctx.vec(0), ctx.vec(0)
    for k, at in enumerate(_places(dims)):
        x = x0.copy()
        x[at] = (np.nan, np.inf)[k % 2]
        dx.upload(x)
        ctx.spmv(0, dx, dy)
        _same(dy.download(), P.spmv(x), f"spmv {at}")
        if levels > 1:
            dc = ctx.vec(1)
            ctx.restrict(0, dr, dx, dc)
            _same(dc.download(), P.restrict(r, P.spmv(x)), f"restrict {at}")
            dc.free()
        ctx.symgs(0, dr, dx)
        _same(dx.download(), P.symgs(r, x), f"symgs {at}")
        if k % 3 or n > 1 << 19:
            continue
        rn = r.copy()
        rn[at] = np.nan
        dx.upload(rn)
        ctx.mg(0, dx, dy)
        _same(dy.download(), P.mg(rn), f"mg {at}")
        for prec, name in ((hip.HPCGX_PREC_FP32, "mg_f32"), (hip.HPCGX_PREC_FP16, "mg_f16")):
            ctx.prepare(prec)
            ctx.mg_mixed(prec, dx, dy)
            _same(dy.download(), getattr(P, name)(rn.astype(np.float32)).astype(np.float64), f"{name} {at}")
