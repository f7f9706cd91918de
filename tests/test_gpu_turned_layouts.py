"""Strided copies, stores and sums between layouts whose unit-stride axes differ, at the sizes where their kernel changes
form: extents around its tiles and around the shortest it takes, outer axes on either side, and against numpy bit for bit
(each element is copied, or added once)."""
import ctypes

import numpy as np
import pytest

from newch_amd import hip, hipmem

pytestmark = pytest.mark.gpu

EXT = [1, 15, 16, 17, 63, 64, 65, 197]


@pytest.fixture(scope="module")
def K():
    return hip.Kernels()


def i64(v):
    return (ctypes.c_int64 * len(v))(*v)


def dev(a):
    return hipmem.DeviceBuffer.from_numpy(a)


def cases():
    for a in EXT:
        for b in (1, 16, 65, 130):
            yield (a, b), (1, 0)
            yield (3, a, b), (0, 2, 1)
    for perm in [(2, 1, 0), (1, 2, 0), (2, 0, 1), (1, 0, 2)]:
        yield (5, 66, 33), perm
    yield (2, 3, 40, 70), (0, 3, 1, 2)
    yield (2, 40, 3, 70), (3, 1, 0, 2)
    yield (20, 2, 3, 18), (3, 2, 1, 0)


@pytest.mark.parametrize("shape,perm", list(cases()))
@pytest.mark.parametrize("off", [0, 1])
def test_turned_layouts(K, shape, perm, off):
    """x[shape] seen through perm: gathered, and values of the view's shape stored and added at its places."""
    rng = np.random.default_rng(sum(shape) + off)
    x, v = (rng.standard_normal(int(np.prod(shape)) + 2).astype(np.float32) for _ in range(2))
    v[3 % v.size] = -0.0
    n = x.size - 2
    X = x[off:off + n].reshape(shape)
    view = X.transpose(perm)
    vs = view.shape
    st = [s // 4 for s in view.strides]
    dx, dv = dev(x), dev(v)
    out = dev(np.full(n + 2, 77, np.float32))
    args = (len(vs), i64(vs))
    assert K.lib.nc_hip_copy_strided(4, *args, dx.ptr + 4 * off, i64(st), out.ptr + 4 * off, None) == 0
    want = np.full(n + 2, 77, np.float32)
    want[off:off + n] = view.ravel()
    np.testing.assert_array_equal(out.to_numpy(np.float32, n + 2), want)
    V = v[off:off + n].reshape(vs)
    back = np.argsort(perm)
    for fn, base in ((K.lib.nc_hip_accumulate_strided, X), (K.lib.nc_hip_store_strided, np.zeros_like(X))):
        dst = dev(x)
        assert fn(*args, dv.ptr + 4 * off, dst.ptr + 4 * off, i64(st), None) == 0
        want = x.copy()
        want[off:off + n] = (base + V.transpose(back)).ravel()
        np.testing.assert_array_equal(dst.to_numpy(np.float32, n + 2).view(np.uint32), want.view(np.uint32))


def test_gaps_and_repeats(K):
    """A transposed slice whose rows lie further apart than they are long, and one repeated along a new axis."""
    rng = np.random.default_rng(4)
    x = rng.standard_normal((70, 90)).astype(np.float32)
    view = x[:, :65].T
    dx, out = dev(x), dev(np.zeros(65 * 70 * 3, np.float32))
    assert K.lib.nc_hip_copy_strided(4, 2, i64(view.shape), dx.ptr, i64((1, 90)), out.ptr, None) == 0
    np.testing.assert_array_equal(out.to_numpy(np.float32, 65 * 70).reshape(65, 70), view)
    assert K.lib.nc_hip_copy_strided(4, 3, i64((3, 65, 70)), dx.ptr, i64((0, 1, 90)), out.ptr, None) == 0
    np.testing.assert_array_equal(out.to_numpy(np.float32, 3 * 65 * 70).reshape(3, 65, 70), np.stack([view] * 3))
    v = rng.standard_normal((65, 70)).astype(np.float32)
    dv = dev(v)
    assert K.lib.nc_hip_accumulate_strided(2, i64((65, 70)), dv.ptr, dx.ptr, i64((1, 90)), None) == 0
    x[:, :65] += v.T
    np.testing.assert_array_equal(dx.to_numpy(np.float32, (70, 90)), x)
