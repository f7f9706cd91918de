"""LayerNorm at the widths where the kernels change form -- a wave or a team of waves per row, how many registers hold it,
rows of whole aligned float4s or not -- at any alignment, forward and backward, against float64."""
import numpy as np
import pytest

from newch_amd import hip, hipmem

pytestmark = pytest.mark.gpu

WIDTHS = [1, 2, 3, 5, 7, 255, 257, 511, 513, 767, 768, 769, 1023, 1024, 1025, 1028, 2048, 2049, 3071, 3073, 4096, 4097, 6144,
          6145, 8191, 8192, 8193, 12288, 12289]
EPS = 1e-5
# A result of one fp32 rounding has 6e-8 of its size; the chains here -- (x - mean) rstd gamma + beta, and the gradient's
# difference of three such terms -- are within 8 roundings of the largest term in each.
TOL = 8 * 2.0 ** -24


@pytest.fixture(scope="module")
def K():
    return hip.Kernels()


def placed(a, off):
    """`a` on the device, `off` floats into a buffer of guard values (77)."""
    flat = np.full(a.size + off + 4, 77, np.float32)
    flat[off:off + a.size] = a.ravel()
    return hipmem.DeviceBuffer.from_numpy(flat)


def read(buf, shape, off):
    n = int(np.prod(shape))
    flat = buf.to_numpy(np.float32, n + off + 4)
    assert (flat[:off] == 77).all() and (flat[off + n:] == 77).all(), "wrote outside"
    return flat[off:off + n].reshape(shape).astype(np.float64)


def near(got, want, scale, roundings=1.0):
    assert np.isfinite(got).all()
    assert (np.abs(got - want) <= roundings * TOL * scale).all(), np.abs(got - want).max() / np.max(scale)


@pytest.mark.parametrize("D", WIDTHS)
@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("acc,affine", [(False, True), (True, False)])
def test_layer_norm_any_width(K, D, off, acc, affine):
    rows = 67 if D < 3000 else 9
    rng = np.random.default_rng(D + off)
    x, g, old = ((rng.standard_normal((rows, D)) * 2).astype(np.float32) for _ in range(3))
    w, b = ((rng.standard_normal(D) * 0.1 + i).astype(np.float32) for i in (1, 0))
    gw0, gb0 = (rng.standard_normal(D).astype(np.float32) for _ in range(2))
    dx, dg, dw, db, dgw, dgb = (placed(a, off) for a in (x, g, w, b, gw0, gb0))
    dy, dgx, dst = placed(np.zeros_like(x), off), placed(old, off), placed(np.zeros((rows, 2)), 0)
    p = 4 * off
    n = K.layer_norm_bwd_workspace(rows, D)
    ws = hipmem.DeviceBuffer.from_numpy(np.full(n + 8, 0x55, np.uint8))
    wp, bp = (dw.ptr + p, db.ptr + p) if affine else (None, None)
    K.layer_norm_fwd(rows, D, dx.ptr + p, wp, bp, EPS, dy.ptr + p, dst.ptr)
    K.layer_norm_bwd(rows, D, dx.ptr + p, wp, dst.ptr, dg.ptr + p, dgx.ptr + p, dgw.ptr + p, dgb.ptr + p, ws.ptr, n,
                     accumulate=acc)
    assert (ws.to_numpy(np.uint8, n + 8)[n:] == 0x55).all(), "wrote past the workspace"

    X, G = x.astype(np.float64), g.astype(np.float64)
    W = w.astype(np.float64) if affine else np.ones(D)
    B = b.astype(np.float64) if affine else np.zeros(D)
    mean = X.mean(1, keepdims=True)
    rstd = 1 / np.sqrt(X.var(1, keepdims=True) + EPS)
    st = read(dst, (rows, 2), 0)
    near(st[:, :1], mean, np.abs(mean))
    near(st[:, 1:], rstd, rstd)
    # from here on with the statistics as stored: the kernels' own inputs
    mean, rstd = st[:, :1], st[:, 1:]
    xh = (X - mean) * rstd
    near(read(dy, (rows, D), off), xh * W + B, np.abs(xh * W) + np.abs(B) + 1e-30)
    gh = G * W
    mg, mgx = gh.mean(1, keepdims=True), (gh * xh).mean(1, keepdims=True)
    size = rstd * (np.abs(gh) + np.abs(gh).mean(1, keepdims=True) + np.abs(xh) * np.abs(gh * xh).mean(1, keepdims=True))
    o = old if acc else np.zeros_like(old)
    near(read(dgx, (rows, D), off), o + rstd * (gh - mg - xh * mgx), size + np.abs(o))
    # the column sums: each product rounded up to three times, at most 9 rows of a wave summed in fp32
    near(read(dgw, (D,), off), gw0 + (G * xh).sum(0), np.abs(gw0) + np.abs(G * xh).sum(0), 2)
    near(read(dgb, (D,), off), gb0 + G.sum(0), np.abs(gb0) + np.abs(G).sum(0), 2)


@pytest.mark.parametrize("D", [257, 2049, 8192])
def test_layer_norm_partial_outputs(K, D):
    """gx alone, and the column gradients alone, equal the full call's."""
    rows = 33
    rng = np.random.default_rng(D)
    x, g = ((rng.standard_normal((rows, D))).astype(np.float32) for _ in range(2))
    w = rng.standard_normal(D).astype(np.float32)
    dx, dg, dw, st = placed(x, 0), placed(g, 0), placed(w, 0), placed(np.zeros((rows, 2)), 0)
    y = placed(x, 0)
    K.layer_norm_fwd(rows, D, dx.ptr, dw.ptr, None, EPS, y.ptr, st.ptr)
    n = K.layer_norm_bwd_workspace(rows, D)
    ws = hipmem.DeviceBuffer.from_numpy(np.zeros(n, np.uint8))

    def run(gx, cols):
        bufs = [placed(np.zeros_like(x), 0), placed(np.zeros(D), 0), placed(np.zeros(D), 0)]
        K.layer_norm_bwd(rows, D, dx.ptr, dw.ptr, st.ptr, dg.ptr, bufs[0].ptr if gx else None,
                         *(b.ptr if cols else None for b in bufs[1:]), ws.ptr, n, accumulate=False)
        return [read(b, s, 0) for b, s in zip(bufs, ((rows, D), (D,), (D,)))]

    full, only_x, only_c = run(True, True), run(True, False), run(False, True)
    np.testing.assert_array_equal(only_x[0], full[0])
    np.testing.assert_array_equal(only_c[1], full[1])
    np.testing.assert_array_equal(only_c[2], full[2])


# constant rows: the lowest and the largest float, a mask's -1e9, a large one, the smallest normal
EXTREMES = [np.finfo(np.float32).min, np.finfo(np.float32).max, -1e9, 1e30, np.finfo(np.float32).tiny]


@pytest.mark.parametrize("D", [3, 5, 255, 257, 513, 767, 769, 1023, 1028, 2044, 2049, 3001, 4100, 6146, 8188, 8193, 12287])
@pytest.mark.parametrize("acc", [False, True])
def test_layer_norm_bwd_of_extreme_rows(K, D, acc):
    """Rows of one value whose mean times rstd leaves the fp32 range: xhat is 0 in all of the row, and the gradient finite,
    whatever the places past the row's end hold."""
    rng = np.random.default_rng(D)
    x = np.repeat(np.float32(EXTREMES)[:, None], D, axis=1)
    x = np.concatenate([x, rng.standard_normal((3, D)).astype(np.float32)])
    rows = len(x)
    g, old = (rng.standard_normal((rows, D)).astype(np.float32) for _ in range(2))
    w = (1 + 0.1 * rng.standard_normal(D)).astype(np.float32)
    dx, dg, dw, dgx = placed(x, 0), placed(g, 0), placed(w, 0), placed(old, 0)
    y, dst = placed(x, 0), placed(np.zeros((rows, 2)), 0)
    dgw, dgb = placed(np.zeros(D), 0), placed(np.zeros(D), 0)
    n = K.layer_norm_bwd_workspace(rows, D)
    ws = hipmem.DeviceBuffer.from_numpy(np.zeros(n, np.uint8))
    print(f"layer_norm extreme rows {rows}x{D} acc={acc}", flush=True)
    K.layer_norm_fwd(rows, D, dx.ptr, dw.ptr, None, EPS, y.ptr, dst.ptr)
    K.layer_norm_bwd(rows, D, dx.ptr, dw.ptr, dst.ptr, dg.ptr, dgx.ptr, dgw.ptr, dgb.ptr, ws.ptr, n, accumulate=acc)
    st = read(dst, (rows, 2), 0)
    mean, rstd = st[:, :1], st[:, 1:]
    assert (mean[:len(EXTREMES), 0].astype(np.float32) == x[:len(EXTREMES), 0]).all()
    G, gh, xh = g.astype(np.float64), g.astype(np.float64) * w, (x - mean) * rstd
    mg, mgx = gh.mean(1, keepdims=True), (gh * xh).mean(1, keepdims=True)
    size = rstd * (np.abs(gh) + np.abs(gh).mean(1, keepdims=True) + np.abs(xh) * np.abs(gh * xh).mean(1, keepdims=True))
    o = old if acc else np.zeros_like(old)
    near(read(dgx, (rows, D), 0), o + rstd * (gh - mg - xh * mgx), size + np.abs(o))
    near(read(dgw, (D,), 0), (G * xh).sum(0), np.abs(G * xh).sum(0), 2)
    near(read(dgb, (D,), 0), G.sum(0), np.abs(G).sum(0), 2)
