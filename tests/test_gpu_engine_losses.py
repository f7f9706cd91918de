"""The losses through nc.h: the label check that the host watches for, behind a long queue and without one."""
import numpy as np
import pytest

from newch_amd import abi
from tests.ncdrive import Engine
from tests.test_gpu_parity import assert_bits, assert_close64

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    L = abi.load(abi.LIB_PATH)
    assert L.nc_device_count() > 0, "no HIP device visible: the GPU tests need an MI355X"
    return L


@pytest.fixture()
def eng(lib):
    e = Engine(lib=lib)
    yield e
    e.close()


@pytest.mark.parametrize("form", ["ce", "nll"])
def test_label_check_behind_long_work(eng, form):
    """Work of several milliseconds queued before the loss: the host stops watching for the check's result after two, waits for
    the stream, and finds a bad label or none as it would at once; calls right after each other use the same word."""
    L = eng.lib
    rng = np.random.default_rng(1)
    n, rows, C = 8192, 33, 7
    x = rng.standard_normal((rows, C)).astype(np.float32)
    lab = rng.integers(0, C, rows).astype(np.int32)
    bad = lab.copy()
    bad[17] = C
    d = x - x.max(1, keepdims=True)
    logp = (d - np.log(np.exp(d).sum(1, keepdims=True))).astype(np.float32)
    want = -logp.astype(np.float64)[np.arange(rows), lab].mean()
    big = eng.tensor(np.full((n, n), 1e-3, np.float32))
    X = eng.tensor(x if form == "ce" else logp)
    good_t, bad_t = eng.tensor(lab), eng.tensor(bad)

    def loss(t):
        return L.nc_cross_entropy(X, t) if form == "ce" else L.nc_nll_loss(X, t, 0)

    for queued in (True, False, True):
        print(f"{form} label check, queued={queued}", flush=True)
        if queued:
            assert L.nc_matmul(big, big)  # 8192^3, about 8 ms
        out = loss(bad_t)
        assert not out and L.nc_status_code(eng.ctx) != 0
        msg = L.nc_error(eng.ctx).decode()
        assert f"label {C} at row 17" in msg, msg
        L.nc_clear_error(eng.ctx)
        if queued:
            assert L.nc_matmul(big, big)
        out = loss(good_t)
        assert out, L.nc_error(eng.ctx)
        assert_close64(eng.read(out), want, abs(want), form)
