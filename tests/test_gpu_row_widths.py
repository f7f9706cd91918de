"""Row kernels at the widths where they change form -- a wave or a workgroup per row, how many registers hold it -- with
rows of 4-byte alignment and rows that hold infinities, NaN and the lowest floats, against fp64 and the oracle."""
import numpy as np
import pytest

from newch_amd import hip, hipmem
from oracle import pyoracle as O
from tests.test_gpu_parity import assert_bits, assert_close64, ce_prob

pytestmark = pytest.mark.gpu

GUARD = np.float32(777.0)
WIDTHS = [5, 255, 257, 513, 1023, 1025, 1028, 2047, 2052, 4095, 4097, 6145, 8191, 8196, 12289, 16383, 16385, 24577,
          32767, 32769, 49153, 65535, 65537]


@pytest.fixture(scope="module")
def K():
    return hip.Kernels()


class Off:
    """A float array on the device, `off` floats into its buffer, guard values on both sides."""

    def __init__(self, a, off):
        a = np.asarray(a, np.float32)
        self.shape, self.n, self.off = a.shape, a.size, off
        flat = np.full(a.size + off + 4, GUARD, np.float32)
        flat[off:off + a.size] = a.ravel()
        self.buf = hipmem.DeviceBuffer.from_numpy(flat)
        self.ptr = self.buf.ptr + 4 * off

    def read(self):
        flat = self.buf.to_numpy(np.float32, self.n + self.off + 4)
        assert (flat[:self.off] == GUARD).all() and (flat[self.off + self.n:] == GUARD).all(), "wrote outside"
        return flat[self.off:self.off + self.n].reshape(self.shape)


def logits(rng, rows, C):
    x = (rng.standard_normal((rows, C)) * 3).astype(np.float32)
    x[0, C - 1] = x[0].max() + 1  # the maximum in the row's last, short piece
    x[1, C // 2] = -np.inf
    x[2] = np.finfo(np.float32).min  # a row of the lowest float
    return x


@pytest.mark.parametrize("C", WIDTHS)
@pytest.mark.parametrize("log_form", [False, True])
def test_softmax_widths(K, C, log_form):
    rng = np.random.default_rng(C + log_form)
    rows = 6
    x, g = logits(rng, rows, C), rng.standard_normal((rows, C)).astype(np.float32)
    off = C % 3
    print(f"softmax {rows}x{C} log={log_form} offset {off}", flush=True)
    X, Y, G = Off(x, off), Off(np.zeros_like(x), off), Off(g, off)
    K.softmax_fwd(log_form, rows, C, X.ptr, Y.ptr)
    hipmem.synchronize()
    y = Y.read()
    x64 = x.astype(np.float64)
    e = np.exp(x64 - x64.max(1, keepdims=True))
    p = e / e.sum(1, keepdims=True)
    with np.errstate(divide="ignore"):
        want = np.log(p) if log_form else p
    assert_close64(y, want, 1.0 if log_form else 0.0, "fwd")
    G64 = g.astype(np.float64)
    if log_form:
        grad, sc = G64 - p * G64.sum(1, keepdims=True), np.abs(G64) + p * np.abs(G64).sum(1, keepdims=True)
    else:
        grad = p * (G64 - (G64 * p).sum(1, keepdims=True))
        sc = p * (np.abs(G64) + (np.abs(G64) * p).sum(1, keepdims=True))
    for acc in (False, True):
        old = rng.standard_normal((rows, C)).astype(np.float32)
        GI = Off(old, off)
        K.softmax_bwd(log_form, rows, C, Y.ptr, G.ptr, GI.ptr, accumulate=acc)
        hipmem.synchronize()
        assert_close64(GI.read(), grad + (old if acc else 0), sc + (np.abs(old) if acc else 0), f"bwd acc={acc}")


@pytest.mark.parametrize("C", [257, 1023, 1025, 4097, 16385, 50001])
def test_softmax_special_rows(K, C):
    """NaN first (the row is NaN), NaN later, all -inf, +inf: the reference's NaN pattern."""
    rng = np.random.default_rng(C)
    x = rng.standard_normal((5, C)).astype(np.float32)
    x[0, 0], x[1, C - 1], x[2], x[3, 7] = np.nan, np.nan, -np.inf, np.inf
    for log_form in (False, True):
        X, Y = Off(x, 1), Off(np.zeros_like(x), 1)
        K.softmax_fwd(log_form, 5, C, X.ptr, Y.ptr)
        hipmem.synchronize()
        y, ref = Y.read(), O.softmax_fwd(x, log_form)
        assert (np.isnan(y) == np.isnan(ref)).all(), f"NaN pattern, log={log_form}"
        assert_close64(y[4], ref[4].astype(np.float64), 1.0 if log_form else 0.0, "plain row")


@pytest.mark.parametrize("C", WIDTHS + [4, 6, 1024, 50257])
def test_cross_entropy_widths(K, C):
    rng = np.random.default_rng(3 * C)
    rows, off = 7, C % 2
    x = logits(rng, rows, C)
    lab = rng.integers(0, C, rows).astype(np.int32)
    lab[0], lab[1], lab[3] = C - 1, 0, C - 1  # labels in a row's last and first piece
    print(f"cross entropy {rows}x{C} offset {off}", flush=True)
    X, S = Off(x, off), hipmem.DeviceBuffer(8 * rows)
    L = hipmem.DeviceBuffer.from_numpy(lab)
    loss, bad = hipmem.DeviceBuffer(4), hipmem.DeviceBuffer(8)
    nws = K.loss_workspace(rows, C)
    ws = hipmem.DeviceBuffer(nws)
    K.cross_entropy_fwd(rows, C, X.ptr, L.ptr, S.ptr, loss.ptr, bad.ptr, ws.ptr, nws)
    hipmem.synchronize()
    assert bad.to_numpy(np.uint64, 1)[0] == np.uint64(0xFFFFFFFFFFFFFFFF)
    # the terms as log(sum exp(x - m)) - (x_label - m): m + log(sum) would lose the log beside the lowest float
    d = x.astype(np.float64) - x.astype(np.float64).max(1, keepdims=True)
    terms = np.log(np.exp(d).sum(1)) - d[np.arange(rows), lab]
    assert_close64(loss.to_numpy(np.float32, 1)[0], terms.mean(), np.abs(terms).sum() / rows ** 1.5, "loss")
    prob = ce_prob(x, S.to_numpy(np.float32, (rows, 2)))
    _, prob_o = O.cross_entropy_fwd(x, lab)
    assert np.allclose(prob, prob_o, rtol=1e-5, atol=1e-30), "row statistics"
    gout = np.float32(0.7)
    GO = hipmem.DeviceBuffer.from_numpy(np.array([gout]))
    for acc in (False, True):
        old = rng.standard_normal((rows, C)).astype(np.float32)
        for o2 in (off, 0):
            GI = Off(old, o2)
            K.cross_entropy_bwd(rows, C, X.ptr, S.ptr, L.ptr, GO.ptr, GI.ptr, accumulate=acc)
            hipmem.synchronize()
            assert_bits(GI.read(), O.cross_entropy_bwd(prob, lab, float(gout), old if acc else None), f"bwd acc={acc}")
    lab[5] = C  # out of range: reported, and contributes nothing
    L2 = hipmem.DeviceBuffer.from_numpy(lab)
    K.cross_entropy_fwd(rows, C, X.ptr, L2.ptr, S.ptr, loss.ptr, bad.ptr, ws.ptr, nws)
    hipmem.synchronize()
    assert bad.to_numpy(np.uint64, 1)[0] == np.uint64((5 << 32) | C)


@pytest.mark.parametrize("C", [1025, 1028, 4097, 16385, 16388, 50257])
@pytest.mark.parametrize("off", [0, 1])
def test_cross_entropy_special_rows(K, C, off):
    """Rows with NaN first, NaN in a late wave, nothing but -inf, +inf in one wave, and whole waves of -inf beside finite
    values: one row a call, so that each loss stands for its row; against the oracle's loss and statistics."""
    rng = np.random.default_rng(C)
    base = (rng.standard_normal(C) * 3).astype(np.float32)
    rows = {name: base.copy() for name in ("plain", "nan first", "nan late", "all -inf", "inf early", "inf late", "waves of -inf",
                                            "last alone")}
    rows["nan first"][0] = np.nan
    rows["nan late"][C - 2] = np.nan
    rows["all -inf"][:] = -np.inf
    rows["inf early"][5] = np.inf
    rows["inf late"][C - 1] = np.inf
    rows["waves of -inf"][:C // 2] = -np.inf
    rows["last alone"][:C - 1] = -np.inf
    nws = K.loss_workspace(1, C)
    S, loss, bad, ws = (hipmem.DeviceBuffer(n) for n in (8, 4, 8, max(nws, 8)))
    for name, x in rows.items():
        for label in (0, C // 3, C - 1):
            X, Lb = Off(x[None], off), hipmem.DeviceBuffer.from_numpy(np.array([label], np.int32))
            print(f"cross entropy 1x{C} offset {off}: {name}, label {label}", flush=True)
            K.cross_entropy_fwd(1, C, X.ptr, Lb.ptr, S.ptr, loss.ptr, bad.ptr, ws.ptr, nws)
            hipmem.synchronize()
            got = loss.to_numpy(np.float32, 1)[0]
            with np.errstate(all="ignore"):
                want, prob_o = O.cross_entropy_fwd(x[None], np.array([label], np.int32))
                prob = ce_prob(x[None], S.to_numpy(np.float32, (1, 2)))
            assert bad.to_numpy(np.uint64, 1)[0] == np.uint64(0xFFFFFFFFFFFFFFFF)
            assert (np.isnan(prob) == np.isnan(prob_o)).all(), f"{name}: statistics"
            ok = ~np.isnan(prob_o)
            assert np.allclose(prob[ok], prob_o[ok], rtol=1e-5, atol=1e-30), f"{name}: statistics"
            if not np.isfinite(want):
                assert np.array_equal(got, np.float32(want), equal_nan=True), (name, got, want)
            else:  # log(sum) rounded, the label's difference, their difference
                assert abs(got - want) <= 4 * 2.0 ** -24 * (abs(want) + 12), (name, got, want)


@pytest.mark.parametrize("C", [77, 257, 513, 1023])
@pytest.mark.parametrize("over", [0, 1])
@pytest.mark.parametrize("log_form,acc", [(False, True), (True, False)])
def test_softmax_bwd_around_the_caches(K, C, over, log_form, acc):
    """The last row count of unaligned rows that is loaded through the caches, and the first that is not."""
    rows = (24 << 20) // C + over
    rng = np.random.default_rng(C + over)
    per = 64
    at = [0, rows // 2, rows - per]
    parts = [[rng.standard_normal((per, C)).astype(np.float32) for _ in range(3)] for _ in at]
    bufs = [hipmem.DeviceBuffer((rows * C + 5) * 4) for _ in range(3)]
    for b in bufs:
        b.zero()
        b.upload(np.float32([GUARD]), 0)
        b.upload(np.full(4, GUARD, np.float32), (rows * C + 1) * 4)
    for r0, part in zip(at, parts):
        for b, a in zip(bufs, part):
            b.upload(a, (r0 * C + 1) * 4)
    y, g, gi = (b.ptr + 4 for b in bufs)
    print(f"softmax bwd {rows}x{C} log={log_form}", flush=True)
    K.softmax_bwd(log_form, rows, C, y, g, gi, accumulate=acc)
    hipmem.synchronize()
    for r0, (py, pg, old) in zip(at, parts):
        got = bufs[2].to_numpy(np.float32, (per, C), (r0 * C + 1) * 4)
        Y, G = py.astype(np.float64), pg.astype(np.float64)
        if log_form:
            p = np.exp(Y)
            want, size = G - p * G.sum(1, keepdims=True), np.abs(G) + p * np.abs(G).sum(1, keepdims=True)
        else:
            want = Y * (G - (G * Y).sum(1, keepdims=True))
            size = np.abs(Y) * (np.abs(G) + np.abs(G * Y).sum(1, keepdims=True))
        o = old if acc else np.zeros_like(old)
        assert_close64(got, o + want, np.abs(o) + size, f"rows {r0}")
    assert bufs[2].to_numpy(np.float32, 1)[0] == GUARD
    assert (bufs[2].to_numpy(np.float32, 4, (rows * C + 1) * 4) == GUARD).all()


@pytest.mark.parametrize("rows,C", [(1535, 1028), (1536, 1028), (1537, 1536), (8192, 2048), (8193, 2048), (1600, 2044), (1536, 2052)])
def test_forward_rows_at_the_choice_by_rows(K, rows, C):
    """Aligned rows of 1028 to 2048 floats on both sides of where a wave takes a row: softmax, log_softmax and LayerNorm."""
    rng = np.random.default_rng(rows + C)
    x = (rng.standard_normal((rows, C)) * 3).astype(np.float32)
    x[0, C - 1] = x[0].max() + 1
    x[1, C // 2] = -np.inf
    x[2] = np.finfo(np.float32).min
    w, b = rng.standard_normal(C).astype(np.float32), rng.standard_normal(C).astype(np.float32)
    X, Y, W, B = Off(x, 0), Off(np.zeros_like(x), 0), Off(w, 0), Off(b, 0)
    x64 = x.astype(np.float64)
    d = x64 - x64.max(1, keepdims=True)
    lse = np.log(np.exp(d).sum(1, keepdims=True))
    for log_form in (False, True):
        print(f"softmax {rows}x{C} log={log_form}", flush=True)
        K.softmax_fwd(log_form, rows, C, X.ptr, Y.ptr)
        hipmem.synchronize()
        assert_close64(Y.read(), d - lse if log_form else np.exp(d - lse), 1.0 if log_form else 0.0, f"log={log_form}")
    x[1, C // 2] = 0
    x[2] = 1
    x64 = x.astype(np.float64)
    X, S = Off(x, 0), Off(np.zeros((rows, 2)), 0)
    K.layer_norm_fwd(rows, C, X.ptr, W.ptr, B.ptr, 1e-5, Y.ptr, S.ptr)
    hipmem.synchronize()
    m, r = x64.mean(1, keepdims=True), 1 / np.sqrt(x64.var(1, keepdims=True) + 1e-5)
    xh = (x64 - m) * r
    # (x - m) r w + b: the mean, rstd and four operations rounded once each
    assert (np.abs(Y.read() - (xh * w + b)) <= 8 * 2.0 ** -24 * ((np.abs(x64) + np.abs(m)) * r * np.abs(w) + np.abs(b))).all()
