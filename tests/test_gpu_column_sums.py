"""Sum-to-shape gradients over leading dims (bias gradients) at the sizes where the column kernel changes form: one column
group or many, odd numbers of columns, one chunk of rows or several, remainders of its unrolled loads, rows further apart
than their length, gradients overwritten or added to -- and terms that are not finite."""
import numpy as np
import pytest

from newch_amd import hip, hipmem

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    return hip.Kernels()


def dev(a):
    return hipmem.DeviceBuffer.from_numpy(a)


def run(K, op, which, rows, cols, g, a, b, gr, old, acc):
    """The gradient of operand `which` of a[rows, cols] op b[cols] (or a[cols] op b[rows, cols]), kept over the columns;
    g's rows start gr floats apart."""
    full, kept = (cols, 1), (0, 1)
    sa, sb = (kept, full) if which == 0 else (full, kept)
    G = np.full((rows, gr), np.nan, np.float32)
    G[:, :cols] = g
    n = K.binary_bwd_workspace((rows, cols), kept)
    ws = np.full(n + 8, 0x55, np.uint8)
    dg, da, db, dgx, dws = dev(G), dev(a), dev(b), dev(np.append(old, np.float32(77))), dev(ws)
    K.binary_bwd(op, which, (rows, cols), dg.ptr, (gr, 1), da.ptr, sa, db.ptr, sb, dgx.ptr, kept, dws.ptr, n,
                 accumulate=acc)
    assert (dws.to_numpy(np.uint8, n + 8)[n:] == 0x55).all(), "wrote past the workspace"
    out = dgx.to_numpy(np.float32, cols + 1)
    assert out[cols] == 77, "wrote past the gradient"
    return out[:cols]


def terms(op, which, g, a, b):
    g, a, b = (v.astype(np.float64) for v in (g, a, b))
    if op in ("add", "sub"):
        return g if op == "add" or which == 0 else -g
    if op == "mul":
        return g * (b if which == 0 else a)
    return g / b if which == 0 else -(g * a) / (b * b)


@pytest.mark.parametrize("cols", [1, 2, 3, 31, 32, 33, 64, 1000, 1001])
@pytest.mark.parametrize("rows", [2, 63, 64, 65, 511, 513, 2048, 2049, 5000])
@pytest.mark.parametrize("op,which,pad,acc", [("add", 1, 0, False), ("sub", 1, 1, True), ("mul", 1, 0, True),
                                              ("mul", 0, 3, False), ("div", 1, 1, False), ("div", 0, 0, True)])
def test_column_sums(K, rows, cols, op, which, pad, acc):
    rng = np.random.default_rng(rows * 1000 + cols)
    g = rng.standard_normal((rows, cols)).astype(np.float32)
    wide, one = rng.standard_normal((rows, cols)).astype(np.float32), rng.uniform(0.5, 2, cols).astype(np.float32)
    if op == "div" and which == 0:
        wide = np.abs(wide) + np.float32(0.5)
    a, b = (one, wide) if which == 0 else (wide, one)
    old = rng.standard_normal(cols).astype(np.float32)
    got = run(K, op, which, rows, cols, g, a, b, cols + pad, old, acc)
    t = terms(op, which, g, a, b)
    start = old.astype(np.float64) if acc else np.zeros(cols)
    want, size = start + t.sum(0), np.abs(start) + np.abs(t).sum(0)
    # fp64 sums of up to 5000 terms of a few roundings each, then one rounding to fp32
    assert (np.abs(got - want) <= 2.0 ** -24 * np.abs(want) + 2.0 ** -38 * size).all()


def test_column_sums_not_finite(K):
    """x / 0, 0 / 0, infinities and NaN give what the terms' own division gives."""
    rows, cols = 70, 8
    rng = np.random.default_rng(1)
    g = rng.standard_normal((rows, cols)).astype(np.float32)
    a = np.abs(rng.standard_normal((rows, cols))).astype(np.float32)
    g[:, 1] = 0
    g[:, 2] = np.abs(g[:, 2])
    a[7, 3] = np.inf
    b = np.array([0, 0, 0, 1, np.inf, np.nan, 1e-30, 1e-42], np.float32)
    got = run(K, "div", 1, rows, cols, g, a, b, cols, np.zeros(cols, np.float32), False)
    with np.errstate(all="ignore"):
        want = terms("div", 1, g, a, b).sum(0).astype(np.float32)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    np.testing.assert_allclose(got[ok], want[ok], rtol=2.0 ** -22)


@pytest.mark.parametrize("rows,cols", [(63, 1 << 17), (95, (1 << 17) + 1), (97, (1 << 17) - 1), (255, 1 << 17), (257, (1 << 17) + 3),
                                       (1024, 5), (1025, 5), (1025, 2049), (2049, 40)])
@pytest.mark.parametrize("op,which", [("add", 1), ("div", 1), ("div", 0)])
def test_column_sums_at_the_choice(K, rows, cols, op, which):
    """Sizes on both sides of the line between a lane a column and the column kernel, and of its first split."""
    test_column_sums(K, rows, cols, op, which, 0, True)
