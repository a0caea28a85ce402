"""Steps by row runs and by single-wave workgroups give the bits of the stored
values: grids whose colour blocks lie around the sizes where the launch shape
changes (2^17 rows: two rows per lane; 2^18: 256 threads a workgroup), with an
odd number of slices, padding and unequal blocks."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# rows of the largest block: 131072, 140608 (2197 slices), 140556 (unequal), 262080 (4095 slices), 262144
GRIDS = [((128, 64, 128), 2), ((104, 104, 104), 2), ((105, 103, 101), 1), ((126, 128, 130), 1), ((128, 128, 128), 1)]


@pytest.mark.parametrize("dims,levels", GRIDS)
@pytest.mark.parametrize("op", ["hpcg", "kappa"])
def test_steps_bitexact(hip, dims, levels, op):
    n = int(np.prod(dims))
    g = np.random.default_rng(n)
    ctx = hip.Context(0)
    ctx.generate(*dims, levels=levels, kappa=np.exp(0.5 * g.standard_normal(n)) if op == "kappa" else None)
    x, r = g.random(n) - 0.5, g.random(n)
    got = {}
    for fmt in (hip.HPCGX_COLS_EXPLICIT, hip.HPCGX_COLS_COMPACT):
        ctx.set_column_format(fmt)
        dx, dr, dy = ctx.vec(0, x), ctx.vec(0, r), ctx.vec(0)
        out = []
        ctx.spmv(0, dx, dy)
        out.append(dy.download())
        ctx.symgs(0, dr, dx)
        out.append(dx.download())
        ctx.mg(0, dr, dy)
        out.append(dy.download())
        for prec in (hip.HPCGX_PREC_FP32, hip.HPCGX_PREC_FP16):
            ctx.prepare(prec)
            ctx.mg_mixed(prec, dr, dy)
            out.append(dy.download())
        got[fmt] = out
        for v in (dx, dr, dy):
            v.free()
    ctx.close()
    for a, b in zip(got[hip.HPCGX_COLS_EXPLICIT], got[hip.HPCGX_COLS_COMPACT]):
        np.testing.assert_array_equal(a.view(np.int64), b.view(np.int64))
