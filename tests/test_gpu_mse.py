"""The mean squared error in one pass: lengths around its unrolled loads and its partition, operands at any alignment,
gradients stored, added to or not asked for; the differences and the gradients bit for bit, the mean against float64."""
import numpy as np
import pytest

from newch_amd import hip, hipmem

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    return hip.Kernels()


def placed(a, off):
    flat = np.full(a.size + off + 4, 77, np.float32)
    flat[off:off + a.size] = a
    return hipmem.DeviceBuffer.from_numpy(flat)


def read(buf, n, off):
    flat = buf.to_numpy(np.float32, n + off + 4)
    assert (flat[:off] == 77).all() and (flat[off + n:] == 77).all(), "wrote outside"
    return flat[off:off + n]


@pytest.mark.parametrize("n", [1, 3, 4, 5, 1023, 1024, 4095, 4096, 4097, 4100, 8192, 1000003, 1 << 22, (1 << 22) + 4099])
@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("acc_a,acc_b", [(0, 0), (1, 1), (0, None), (None, 1)])
def test_mse_kernels(K, n, off, acc_a, acc_b):
    rng = np.random.default_rng(n + off)
    a, b, ga, gb = (rng.standard_normal(n).astype(np.float32) for _ in range(4))
    g = np.float32(1.7)
    da, db, dd = placed(a, off), placed(b, off), placed(np.zeros(n), 0)
    dga, dgb = placed(ga, off), placed(gb, off)
    dg, loss = placed(np.array([g]), 0), placed(np.zeros(1), 0)
    nws = K.lib.nc_hip_mse_loss_workspace(n)
    ws = hipmem.DeviceBuffer.from_numpy(np.full(nws + 8, 0x55, np.uint8))
    p = 4 * off
    assert K.lib.nc_hip_mse_loss_fwd(n, da.ptr + p, db.ptr + p, dd.ptr, loss.ptr, ws.ptr, nws, None) == 0
    d = a - b
    np.testing.assert_array_equal(read(dd, n, 0), d)
    want = (d * d).astype(np.float64).mean()
    assert abs(read(loss, 1, 0)[0] - want) <= 2.0 ** -23 * want  # one rounding of an fp64 sum
    assert (ws.to_numpy(np.uint8, nws + 8)[nws:] == 0x55).all(), "wrote past the workspace"
    assert K.lib.nc_hip_mse_loss_bwd(n, dd.ptr, dg.ptr, dga.ptr + p if acc_a is not None else None,
                                     dgb.ptr + p if acc_b is not None else None, acc_a or 0, acc_b or 0, None) == 0
    u = (np.float32(1) / np.float32(n) * g) * d
    for buf, old, acc, sign in ((dga, ga, acc_a, 1), (dgb, gb, acc_b, -1)):
        want = old if acc is None else (old if acc else np.float32(0)) + np.float32(sign) * (u + u)
        np.testing.assert_array_equal(read(buf, n, off), want)
