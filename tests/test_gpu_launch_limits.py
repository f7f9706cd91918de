"""Row counts whose workgroups, one launch's worth of lanes each, would not fit a launch: a dispatch counts its work-items
in 32 bits, so such calls run as several launches or loop."""
import numpy as np
import pytest

from newch_amd import hip, hipmem
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu

PER_LAUNCH = 1 << 21  # rows a launch of the kernels with a workgroup a row


@pytest.fixture(scope="module")
def K():
    return hip.Kernels()


def test_narrow_rows_past_a_launch(K):
    """[2^26 + 37, 3]: a wave a row is more than 2^32 lanes; softmax loops over the rows, quantization splits."""
    rows, C, per = (1 << 26) + 37, 3, 1 << 16
    rng = np.random.default_rng(5)
    base = rng.standard_normal((per, C)).astype(np.float32)
    X = hipmem.DeviceBuffer(rows * C * 4)
    for r0 in (0, rows - per):  # the rows looked at; the others are zeros
        if r0 == 0:
            X.zero()
        X.upload(base, r0 * C * 4)
    print(f"softmax, quantize {rows}x{C}", flush=True)
    Y, Q, S = hipmem.DeviceBuffer(rows * C * 4), hipmem.DeviceBuffer(rows * C), hipmem.DeviceBuffer(rows * 4)
    K.softmax_fwd(False, rows, C, X.ptr, Y.ptr)
    K.quantize_rows(rows, C, X.ptr, Q.ptr, S.ptr)
    hipmem.synchronize()
    e = np.exp(base.astype(np.float64) - base.max(1, keepdims=True))
    want = e / e.sum(1, keepdims=True)
    wq, ws = O.quantize_rows(base)
    for r0 in (0, rows - per):
        assert np.abs(Y.to_numpy(np.float32, (per, C), r0 * C * 4) - want).max() < 1e-6
        assert (Q.to_numpy(np.int8, (per, C), r0 * C) == wq).all()
        assert (S.to_numpy(np.float32, (per,), r0 * 4) == ws).all()
    mid = PER_LAUNCH * 16  # zeros: equal shares, scale 1
    assert np.abs(Y.to_numpy(np.float32, (64, C), mid * C * 4) - 1 / 3).max() < 1e-6
    assert (S.to_numpy(np.float32, (64,), mid * 4) == 1).all()


def test_wide_rows_past_a_launch(K):
    """[2^21 + 3, 1028]: softmax, LayerNorm and quantization run as two launches; rows on both sides of the seam."""
    rows, C, per = PER_LAUNCH + 3, 1028, 8
    rng = np.random.default_rng(6)
    base = rng.standard_normal((per, C)).astype(np.float32)
    at = rows - per  # five rows of the first launch and all of the second
    X, Y = hipmem.DeviceBuffer(rows * C * 4), hipmem.DeviceBuffer(rows * C * 4)
    X.zero()
    X.upload(base, at * C * 4)
    x64 = base.astype(np.float64)
    print(f"softmax, layer_norm, quantize {rows}x{C}", flush=True)
    K.softmax_fwd(False, rows, C, X.ptr, Y.ptr)
    hipmem.synchronize()
    e = np.exp(x64 - x64.max(1, keepdims=True))
    y = Y.to_numpy(np.float32, (per, C), at * C * 4)
    assert np.abs(y - e / e.sum(1, keepdims=True)).max() < 1e-6
    G = hipmem.DeviceBuffer(rows * C * 4)
    G.zero()
    g = rng.standard_normal((per, C)).astype(np.float32)
    G.upload(g, at * C * 4)
    K.softmax_bwd(False, rows, C, Y.ptr, G.ptr, X.ptr, accumulate=True)  # x + y (g - <y, g>)
    hipmem.synchronize()
    y64 = y.astype(np.float64)
    want = x64 + y64 * (g - (y64 * g).sum(1, keepdims=True))
    assert np.abs(X.to_numpy(np.float32, (per, C), at * C * 4) - want).max() < 1e-5
    X.upload(base, at * C * 4)
    S = hipmem.DeviceBuffer(rows * 8)
    K.layer_norm_fwd(rows, C, X.ptr, None, None, 1e-5, Y.ptr, S.ptr)
    hipmem.synchronize()
    m, v = x64.mean(1, keepdims=True), x64.var(1, keepdims=True)
    assert np.abs(Y.to_numpy(np.float32, (per, C), at * C * 4) - (x64 - m) / np.sqrt(v + 1e-5)).max() < 1e-5
    assert np.abs(S.to_numpy(np.float32, (per, 2), at * 8)[:, 0] - m[:, 0]).max() < 1e-6
    K.quantize_rows(rows, C, X.ptr, Y.ptr, S.ptr)
    hipmem.synchronize()
    wq, ws = O.quantize_rows(base)
    assert (Y.to_numpy(np.int8, (per, C), at * C) == wq).all()
    assert (S.to_numpy(np.float32, (per,), at * 4) == ws).all()


def test_column_sums_past_a_launch(K):
    """[32, 2^27 - 1] summed over its rows: 2^22 groups of 32 columns, 1024 lanes each, are 2^32 lanes."""
    rows, cols, per = 32, (1 << 27) - 1, 1 << 14
    assert rows * cols < 2 ** 32 - 1
    rng = np.random.default_rng(7)
    G, X = hipmem.DeviceBuffer(rows * cols * 4), hipmem.DeviceBuffer(cols * 4)
    K.fill(G.ptr, 4, 0x3f800000, rows * cols)
    starts = (0, cols // 2, cols - per)
    parts = [rng.standard_normal((rows, per)).astype(np.float32) for _ in starts]
    for c0, part in zip(starts, parts):
        for r in range(rows):
            G.upload(part[r], (r * cols + c0) * 4)
    n = K.binary_bwd_workspace((rows, cols), (0, 1))
    ws = hipmem.DeviceBuffer(max(n, 8))
    print(f"column sums {rows}x{cols}", flush=True)
    K.binary_bwd("add", 1, (rows, cols), G.ptr, (cols, 1), G.ptr, (cols, 1), G.ptr, (0, 1), X.ptr, (0, 1), ws.ptr, n,
                 accumulate=False)
    hipmem.synchronize()
    for c0, part in zip(starts, parts):
        t = part.astype(np.float64)
        got, want = X.to_numpy(np.float32, (per,), c0 * 4), t.sum(0)
        # an fp64 sum of 32 terms, one rounding to fp32
        assert (np.abs(got - want) <= 2.0 ** -24 * np.abs(want) + 2.0 ** -46 * np.abs(t).sum(0)).all()
    assert (X.to_numpy(np.float32, (per,), per * 4) == rows).all()


@pytest.mark.parametrize("n", [2 ** 32 - 2048, 2 ** 32 - 2047, 2 ** 32 - 1023, 2 ** 32 - 2])
def test_full_sum_up_to_2_32_elements(K, n):
    """The gradient of a scalar operand, summed over just under 2^32 elements: the last part of the sum ends where 32 bits do.
    Ones, and larger values in the last part, at its start and at the very end."""
    G, X = hipmem.DeviceBuffer(n * 4), hipmem.DeviceBuffer(4)
    K.fill(G.ptr, 4, 0x3f800000, n)
    extra = {0: 3e9, n // 2: 1e9, n - (1 << 21): 5e8, n - 4: 2.5e8, n - 2: 1.25e8, n - 1: 2.0 ** 27}
    for i, v in extra.items():
        G.upload(np.float32([v]), i * 4)
    ws_bytes = K.binary_bwd_workspace((n,), (0,))
    ws = hipmem.DeviceBuffer(max(ws_bytes, 8))
    print(f"full sum of {n}", flush=True)
    K.binary_bwd("add", 1, (n,), G.ptr, (1,), G.ptr, (1,), G.ptr, (0,), X.ptr, (0,), ws.ptr, ws_bytes, accumulate=False)
    hipmem.synchronize()
    # whole numbers below 2^53: the fp64 sum is exact, and rounded once
    assert X.to_numpy(np.float32, 1)[0] == np.float32(n - len(extra) + sum(float(np.float32(v)) for v in extra.values()))
