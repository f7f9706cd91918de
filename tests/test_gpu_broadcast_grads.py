"""Gradients of broadcast operands where four elements are taken at a time: rows shorter than a group, odd rows, groups that
reach past a row or past the array, operands that repeat, lie apart or run transposed, any alignment -- gradients of the whole
shape bit for bit as the fp32 expressions give them, reduced ones against float64."""
import numpy as np
import pytest

from newch_amd import hip, hipmem

pytestmark = pytest.mark.gpu

# (shape, which dims the other operand keeps)
FORMS = [((7, 5), (0, 1)), ((3, 2, 3), (1, 0, 1)), ((3, 5, 7), (0, 1, 0)), ((5, 4, 6), (0, 1, 0)), ((2, 33, 1), (1, 1, 0)),
         ((9, 67, 31), (0, 1, 0)), ((4, 3, 1025), (0, 1, 0)), ((4, 3, 1024), (1, 0, 0)), ((50, 2, 2), (0, 1, 0)),
         ((6, 5, 64), (1, 0, 1)), ((3, 300, 18), (0, 1, 1)), ((1, 1, 4099), (0, 0, 0)), ((2, 3, 4, 5, 6), (0, 1, 0, 1, 0)),
         ((17, 3, 9, 11), (0, 1, 0, 0))]


@pytest.fixture(scope="module")
def K():
    return hip.Kernels()


def placed(a, off):
    flat = np.full(a.size + off + 4, 77, np.float32)
    flat[off:off + a.size] = a.ravel()
    return hipmem.DeviceBuffer.from_numpy(flat)


def strides(shape, keep=None):
    st, s = [], 1
    for i in reversed(range(len(shape))):
        kept = keep is None or keep[i]
        st.append(s if kept else 0)
        s *= shape[i] if kept else 1
    return tuple(reversed(st))


def parts(op, which, g, a, b):
    if op == "add":
        return g
    if op == "mul":
        return g * (b if which == 0 else a)
    return g / b if which == 0 else -((g * a) / (b * b))


@pytest.mark.parametrize("shape,keep", FORMS)
@pytest.mark.parametrize("op", ["add", "mul", "div"])
@pytest.mark.parametrize("which,small", [(0, "a"), (0, "b"), (1, "a"), (1, "b")])
@pytest.mark.parametrize("off,acc", [(0, False), (1, True)])
def test_broadcast_grads(K, shape, keep, op, which, small, off, acc):
    rng = np.random.default_rng(len(shape) * 100 + shape[-1])
    kshape = tuple(n if k else 1 for n, k in zip(shape, keep))
    sha, shb = (kshape, shape) if small == "a" else (shape, kshape)
    g, a = rng.standard_normal(shape).astype(np.float32), rng.standard_normal(sha).astype(np.float32)
    b = rng.uniform(0.5, 2, shb).astype(np.float32)
    sa, sb = (strides(shape, keep), strides(shape)) if small == "a" else (strides(shape), strides(shape, keep))
    gshape, sgx = (sha, sa) if which == 0 else (shb, sb)
    old = rng.standard_normal(gshape).astype(np.float32)
    p = 4 * off
    dg, da, db, dgx = placed(g, off), placed(a, off), placed(b, off), placed(old, off)
    n = K.binary_bwd_workspace(shape, sgx)
    ws = hipmem.DeviceBuffer.from_numpy(np.full(n + 8, 0x55, np.uint8))
    K.binary_bwd(op, which, shape, dg.ptr + p, strides(shape), da.ptr + p, sa, db.ptr + p, sb, dgx.ptr + p, sgx, ws.ptr, n,
                 accumulate=acc)
    assert (ws.to_numpy(np.uint8, n + 8)[n:] == 0x55).all(), "wrote past the workspace"
    size = int(np.prod(gshape))
    flat = dgx.to_numpy(np.float32, size + off + 4)
    assert (flat[:off] == 77).all() and (flat[off + size:] == 77).all(), "wrote outside"
    got = flat[off:off + size].reshape(gshape)
    start = old if acc else np.zeros_like(old)
    if gshape == shape:
        np.testing.assert_array_equal(got, start + parts(op, which, g, a, b))
        return
    t = parts(op, which, *(v.astype(np.float64) for v in (g, a, b)))
    axes = tuple(i for i, k in enumerate(keep) if not k and shape[i] > 1)
    want = start.astype(np.float64) + t.sum(axes, keepdims=True)
    mag = np.abs(start.astype(np.float64)) + np.abs(t).sum(axes, keepdims=True)
    # fp64 sums of up to 5000 terms of a few roundings each, then one rounding to fp32
    assert (np.abs(got - want) <= 2.0 ** -24 * np.abs(want) + 2.0 ** -38 * mag).all()


def test_strided_operands(K):
    """The other operand transposed, and taken every third element; g transposed."""
    rng = np.random.default_rng(5)
    H, W = 67, 35
    g, a = rng.standard_normal((H, W)).astype(np.float32), rng.standard_normal((H, W)).astype(np.float32)
    big = rng.standard_normal((W, H)).astype(np.float32), rng.standard_normal(H * W * 3).astype(np.float32)
    gx = hipmem.DeviceBuffer.from_numpy(np.zeros((H, W), np.float32))
    dg, da, dt = placed(g, 0), placed(a, 0), placed(np.ascontiguousarray(g.T), 0)
    d0, d1 = placed(big[0], 0), placed(big[1], 0)
    c = (W, 1)
    for arr, st, view in ((d0, (1, H), big[0].T), (d1, (3 * W, 3), big[1][::3].reshape(H, W))):
        K.binary_bwd("mul", 0, (H, W), dg.ptr, c, da.ptr, c, arr.ptr, st, gx.ptr, c, None, 0, accumulate=False)
        np.testing.assert_array_equal(gx.to_numpy(np.float32, (H, W)), g * view)
    K.binary_bwd("mul", 0, (H, W), dt.ptr, (1, H), da.ptr, c, da.ptr, c, gx.ptr, c, None, 0, accumulate=False)
    np.testing.assert_array_equal(gx.to_numpy(np.float32, (H, W)), g * a)


@pytest.mark.parametrize("C", [2, 3, 5, 63, 64, 65, 66, 255, 256, 257, 1023, 1024, 1025])
@pytest.mark.parametrize("rows", [2, 5, 4095, 4096, 4099])
@pytest.mark.parametrize("op,which,small", [("add", 1, "b"), ("mul", 1, "b"), ("div", 0, "a"), ("div", 1, "b")])
def test_row_sums(K, rows, C, op, which, small):
    """A gradient kept over the rows: by a wave an element or a group a lane, or by a workgroup; divisors of 0, infinity, NaN
    and subnormals among the rows' shared ones."""
    rng = np.random.default_rng(rows + C)
    shape, keep = (rows, C), (1, 0)
    sha, shb = ((rows, 1), shape) if small == "a" else (shape, (rows, 1))
    g, a = rng.standard_normal(shape).astype(np.float32), rng.standard_normal(sha).astype(np.float32)
    b = rng.uniform(0.5, 2, shb).astype(np.float32)
    if small == "b" and op == "div":
        special = np.float32([0, np.inf, np.nan, 1e-42, -0.0])[:rows]
        b[:len(special), 0] = special
        g[0, 1] = 0
    full, kept = (C, 1), (1, 0)
    sa, sb = (kept, full) if small == "a" else (full, kept)
    old = rng.standard_normal((rows, 1)).astype(np.float32)
    dg, da, db, dgx = placed(g, 1), placed(a, 1), placed(b, 1), placed(old, 1)
    n = K.binary_bwd_workspace(shape, kept)
    ws = hipmem.DeviceBuffer.from_numpy(np.full(n + 8, 0x55, np.uint8))
    K.binary_bwd(op, which, shape, dg.ptr + 4, full, da.ptr + 4, sa, db.ptr + 4, sb, dgx.ptr + 4, kept, ws.ptr, n,
                 accumulate=True)
    assert (ws.to_numpy(np.uint8, n + 8)[n:] == 0x55).all(), "wrote past the workspace"
    flat = dgx.to_numpy(np.float32, rows + 5)
    assert flat[0] == 77 and (flat[rows + 1:] == 77).all(), "wrote outside"
    with np.errstate(all="ignore"):
        t = parts(op, which, *(v.astype(np.float64) for v in (g, a, b)))
        want, mag = old[:, 0] + t.sum(1), np.abs(old[:, 0]) + np.abs(t).sum(1)
        got, plain = flat[1:rows + 1], np.abs(want) < 3e38
        np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
        np.testing.assert_array_equal(got[~plain & ~np.isnan(want)], want[~plain & ~np.isnan(want)].astype(np.float32))
        # fp64 sums of up to 1025 terms of a few roundings each, then one rounding to fp32
        assert (np.abs(got - want) <= 2.0 ** -24 * np.abs(want) + 2.0 ** -40 * mag)[plain].all()
