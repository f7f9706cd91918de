"""Row quantization and its inverse at the widths where the kernels change form -- a wave or a workgroup per row, how many
registers hold it, rows of whole float4s or not -- at any alignment, with infinities, NaN and zero rows: equal to the
same fp32 steps in numpy bit for bit."""
import numpy as np
import pytest

from newch_amd import hip, hipmem

pytestmark = pytest.mark.gpu

WIDTHS = [1, 2, 3, 4, 5, 7, 255, 256, 257, 511, 513, 767, 769, 1023, 1024, 1025, 2048, 2049, 3076, 4095, 5120, 6145,
          7167, 8191, 8192, 8193, 10241, 11008, 12289, 16385, 24577, 32769, 49153, 65535, 65536, 65537]


@pytest.fixture(scope="module")
def K():
    return hip.Kernels()


def placed(a, off):
    """`a` on the device, `off` elements into a buffer of guard values (77)."""
    flat = np.full(a.size + off + 4, 77, a.dtype)
    flat[off:off + a.size] = a.ravel()
    return hipmem.DeviceBuffer.from_numpy(flat)


def read(buf, dtype, shape, off):
    n = int(np.prod(shape))
    flat = buf.to_numpy(dtype, n + off + 4)
    assert (flat[:off] == 77).all() and (flat[off + n:] == 77).all(), "wrote outside"
    return flat[off:off + n].reshape(shape)


def quantized(w):
    a = np.abs(w)
    amax = np.fmax.reduce(np.concatenate([np.zeros_like(w[:, :1]), a], 1), axis=1)
    s = np.where(amax > 0, amax / np.float32(127), np.float32(1)).astype(np.float32)
    with np.errstate(invalid="ignore"):
        v = np.rint(w * (np.float32(1) / s)[:, None])
    v = np.where(v > 127, np.float32(127), np.where(v < -127, np.float32(-127), v))
    return np.where(np.isnan(v), np.float32(0), v).astype(np.int8), s


def rows_of(rng, rows, C):
    w = (rng.standard_normal((rows, C)) * 3).astype(np.float32)
    w[1 % rows] = 0
    w[2 % rows, C - 1] = np.inf
    w[3 % rows, C // 2] = np.nan
    w[4 % rows, C - 1] = -100.0  # the row's scale comes from its last element
    return w


@pytest.mark.parametrize("C", WIDTHS)
@pytest.mark.parametrize("off", [0, 3])
def test_quantize_any_width(K, C, off):
    rows = 9 if C < 20000 else 5
    w = rows_of(np.random.default_rng(C + off), rows, C)
    dw, dq, ds = placed(w, off), placed(np.zeros((rows, C), np.int8), off), placed(np.zeros(rows, np.float32), 1)
    K.quantize_rows(rows, C, dw.ptr + 4 * off, dq.ptr + off, ds.ptr + 4)
    q, s = quantized(w)
    np.testing.assert_array_equal(read(ds, np.float32, (rows,), 1), s)
    np.testing.assert_array_equal(read(dq, np.int8, (rows, C), off), q)


@pytest.mark.parametrize("C", WIDTHS[:17] + [8193])
@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("rows", [1, 7])
def test_dequantize_any_width(K, C, off, rows):
    rng = np.random.default_rng(C + rows)
    q = rng.integers(-128, 128, (rows, C), dtype=np.int8)
    s = rng.standard_normal(rows).astype(np.float32)
    dq, ds, dw = placed(q, off), placed(s, 0), placed(np.zeros((rows, C), np.float32), off)
    K.dequantize_rows(rows, C, dq.ptr + off, ds.ptr, dw.ptr + 4 * off)
    np.testing.assert_array_equal(read(dw, np.float32, (rows, C), off), q.astype(np.float32) * s[:, None])
