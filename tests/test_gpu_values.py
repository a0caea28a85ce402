"""The value forms give the bits of the stored values.

With compact columns a stencil level whose stored entries are one value per
slot is read as 27 values and a row mask, and a generated kappa level as its
kappa field and the mask; with explicit columns every kernel reads the stored
value array.  Each form is compared with the stored values bit for bit: on
grids with padding, one-wide and odd extents, boundary rows in every slice,
with diagonals replaced (one value, then many), and on levels that only nearly
have a form (one entry changed, an entry of -0) and must fall back.  Signed
zeros, infinities and NaN are compared on stored values with compact columns:
a neighbour outside the grid is a zero entry that names the row itself with
explicit columns and may name another with compact ones, and 0 * inf tells the
two apart."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _kappa(n, seed=1):
    return np.exp(0.5 * np.random.default_rng(seed).standard_normal(n))


def _generate(dims, levels, kappa=None):
    def make(hip):
        ctx = hip.Context(0)
        ctx.generate(*dims, levels=levels, kappa=kappa)
        return ctx
    return make


def _upload(dims, change):
    """The HPCG matrix as uploaded rows, one entry changed."""
    def make(hip):
        src = hip.Context(0)
        src.generate(*dims, levels=1)
        nr, cols, vals = src.export_level(0)
        change(vals)
        ctx = hip.Context(0)
        ctx.upload_level(0, dims, nr, cols, vals)
        return ctx
    return make


def _set(i, j, v):
    def change(vals):
        vals[i, j] = v
    return change


def _diagonal(value):
    def make(hip):
        ctx = hip.Context(0)
        ctx.generate(12, 8, 16, levels=3)
        for l in range(3):
            n = ctx.info(l)["n"]
            ctx.set_diagonal(l, np.full(n, 31.0) if value is None else 26.0 + value * np.arange(n))
        return ctx
    return make


_zeros = _kappa(8 * 8 * 8)
_zeros[100:102] = 0.0  # two neighbouring cells: their coupling is -0

CASES = {
    "hpcg_16": _generate((16, 16, 16), 4),
    "hpcg_2": _generate((2, 2, 2), 1),
    "hpcg_1x1x1": _generate((1, 1, 1), 1),
    "hpcg_1x5x7": _generate((1, 5, 7), 1),
    "hpcg_33x17x9": _generate((33, 17, 9), 1),
    "hpcg_130x6x10": _generate((130, 6, 10), 2),
    "hpcg_256x256x8_strips": _generate((256, 256, 8), 4),
    "hpcg_one_new_diagonal": _diagonal(None),
    "hpcg_many_diagonals": _diagonal(0.5),
    "hpcg_uploaded": _upload((9, 8, 7), lambda vals: None),
    "hpcg_entry_changed": _upload((9, 8, 7), _set(200, 3, -1.5)),
    "hpcg_entry_negative_zero": _upload((9, 8, 7), _set(200, 3, -0.0)),
    "hpcg_entry_zero": _upload((9, 8, 7), _set(200, 3, 0.0)),
    "kappa_16": _generate((16, 16, 16), 4, _kappa(4096)),
    "kappa_one": _generate((16, 8, 8), 3, np.full(1024, 1.75)),
    "kappa_7x5x9": _generate((7, 5, 9), 1, _kappa(315)),
    "kappa_66x10x6": _generate((66, 10, 6), 2, _kappa(3960)),
    "kappa_zero_coupling": _generate((8, 8, 8), 2, _zeros),
}


def _vectors(n):
    g = np.random.default_rng(7)
    yield "random", g.random(n) - 0.5, g.random(n)


def _special(n):
    g = np.random.default_rng(8)
    x, r = g.random(n) - 0.5, g.random(n)
    x[::5] = -0.0
    x[n // 2], r[n // 3] = np.inf, np.nan
    x[n // 4] = -1e308
    return x, r


def _run(hip, ctx, fmt):
    ctx.set_column_format(fmt)
    n, levels = ctx.info(0)["n"], ctx.info(0)["levels"]
    precisions = [("fp32", hip.HPCGX_PREC_FP32), ("fp16", hip.HPCGX_PREC_FP16)]
    for _, prec in precisions:
        ctx.prepare(prec)
    out = {}
    for kind, x, r in _vectors(n):
        dx, dr, dy = ctx.vec(0, x), ctx.vec(0, r), ctx.vec(0)
        ctx.spmv(0, dx, dy)
        out[kind, "spmv"] = dy.download()
        ctx.symgs(0, dr, dx)
        out[kind, "symgs"] = dx.download()
        if levels > 1:
            dc = ctx.vec(1)
            ctx.restrict(0, dr, dx, dc)
            out[kind, "restrict"] = dc.download()
        ctx.mg(0, dr, dy)
        out[kind, "mg"] = dy.download()
        for name, prec in precisions:
            ctx.mg_mixed(prec, dr, dy)
            out[kind, name] = dy.download()
    db, ds = ctx.vec(0, np.ones(n)), ctx.vec(0)
    out["cg", "hist"] = ctx.cg(db, ds, max_iter=6, history=True)["hist"]
    out["cg", "x"] = ds.download()
    return out


def _same(got, want, what):
    nan = np.isnan(want)
    np.testing.assert_array_equal(np.isnan(got), nan, err_msg=what)
    np.testing.assert_array_equal(got[~nan].view(np.int64), want[~nan].view(np.int64), err_msg=what)


@pytest.mark.parametrize("case", sorted(CASES))
def test_value_forms_same_bits(hip, case):
    ctx = CASES[case](hip)
    stored = _run(hip, ctx, hip.HPCGX_COLS_EXPLICIT)
    formed = _run(hip, ctx, hip.HPCGX_COLS_COMPACT)
    for key, want in stored.items():
        _same(formed[key], want, str(key))


@pytest.mark.parametrize("dims", [(16, 16, 16), (33, 17, 9), (130, 6, 10), (7, 5, 9)])
def test_field_form_special_values(hip, dims):
    """The kappa matrix generated (field) and uploaded (stored values).  The
    product alone: a smoothing step on a vector that holds an infinity is not
    one value (a zero entry may name a row that the same step updates)."""
    n = int(np.prod(dims))
    made = _generate(dims, 1, _kappa(n))(hip)
    sent = hip.Context(0)
    sent.upload_level(0, dims, *made.export_level(0))
    x, _ = _special(n)
    got = []
    for ctx in (made, sent):
        dx, dy = ctx.vec(0, x), ctx.vec(0)
        ctx.spmv(0, dx, dy)
        got.append(dy.download())
    _same(got[0], got[1], "spmv")


@pytest.mark.parametrize("dims", [(16, 16, 16), (33, 17, 9), (130, 6, 10), (7, 5, 9)])
def test_slot_form_special_values(hip, dims):
    """The HPCG matrix, and with one entry of one row changed (stored values):
    the product is the same on every other row."""
    n = int(np.prod(dims))
    row = n // 7
    made = _upload(dims, lambda vals: None)(hip)
    sent = _upload(dims, _set(row, 0, -1.5))(hip)
    x, _ = _special(n)
    got = []
    for ctx in (made, sent):
        dx, dy = ctx.vec(0, x), ctx.vec(0)
        ctx.spmv(0, dx, dy)
        got.append(np.delete(dy.download(), row))
    _same(got[0], got[1], "spmv")


def test_diagonal_replaced_under_a_form(hip):
    """The benchmark's own check rewrites the diagonal of a level in use
    (TestCG.cpp:68-79) and puts it back: each state gives the bits of the
    stored values."""
    ctx = hip.Context(0)
    ctx.generate(16, 8, 12, levels=2)
    n = ctx.info(0)["n"]
    ctx.set_column_format(hip.HPCGX_COLS_COMPACT)
    first = _run(hip, ctx, hip.HPCGX_COLS_COMPACT)
    for d in (np.where(np.arange(n) < 9, 26.0 * (np.arange(n) + 2) * 1e6, 26.0e6), np.full(n, 26.0)):
        ctx.set_column_format(hip.HPCGX_COLS_COMPACT)
        ctx.set_diagonal(0, d)
        formed = _run(hip, ctx, hip.HPCGX_COLS_COMPACT)
        stored = _run(hip, ctx, hip.HPCGX_COLS_EXPLICIT)
        for key, want in stored.items():
            np.testing.assert_array_equal(formed[key], want, err_msg=str(key))
    for key, want in first.items():
        np.testing.assert_array_equal(stored[key], want, err_msg=str(key))
