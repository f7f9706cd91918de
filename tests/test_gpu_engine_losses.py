"""Through nc.h: the label check that the host watches for, behind a long queue and without one; mse_loss as one op against the
sub, mul and mean it stands for; transposes' gradients, stored where they come first and added where they do not."""
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


def composite_mse(L, a, b):
    d = L.nc_sub(a, b)
    return L.nc_mean(L.nc_mul(d, d), abi.ALL_AXES, 0)


def both_ways(eng, build, passes=1, flags=abi.BACKWARD_RETAIN):
    """(loss, gradients of the leaves) by nc_mse_loss and by the composite; build(mse) -> (loss, leaves)."""
    L, out = eng.lib, []
    for mse in (L.nc_mse_loss, lambda a, b: composite_mse(L, a, b)):
        loss, leaves = build(mse)
        eng.check()
        value = eng.read(loss)
        for _ in range(passes):
            assert L.nc_backward_ex(loss, flags, None, 0) == 0, L.nc_error(eng.ctx)
        out.append((value, [eng.grad(t) for t in leaves]))
        eng.step_end()
    return out


def same(out, what):
    (v1, g1), (v2, g2) = out
    # the mean: an fp64 sum either way, rounded to fp32 once, or twice in the composite (the sum, then times 1 / n)
    assert abs(float(v1) - float(v2)) <= 3 * 2.0 ** -24 * abs(float(v2)), what
    for a, b in zip(g1, g2):
        assert_bits(a, b, what)


SHAPES = [(1,), (3, 5), (64, 257), (2, 3, 4, 5), (4099,)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("want", ["pred", "target", "both"])
@pytest.mark.parametrize("passes", [1, 2])
def test_mse_gradients_are_the_composites(eng, shape, want, passes):
    """One, the other or both operands with gradients, run back once and twice (leaves add, the rest starts anew)."""
    rng = np.random.default_rng(len(shape))
    a, b = (rng.standard_normal(shape).astype(np.float32) for _ in range(2))

    def build(mse):
        A = eng.param(a) if want != "target" else eng.tensor(a)
        B = eng.param(b) if want != "pred" else eng.tensor(b)
        return mse(A, B), [t for t, w in ((A, "pred"), (B, "target")) if want in (w, "both")]

    same(both_ways(eng, build, passes), f"mse {shape} {want} x{passes}")


@pytest.mark.parametrize("flags", [0, abi.BACKWARD_RETAIN, abi.BACKWARD_FREE_GRAPH])
def test_mse_of_views_and_shared_leaves(eng, flags):
    """Transposed and sliced operands, operands of one leaf, a prediction that feeds another term too, and leaves that hold a
    gradient from before."""
    L = eng.lib
    rng = np.random.default_rng(9)
    a, b = rng.standard_normal((6, 10)).astype(np.float32), rng.standard_normal((10, 6)).astype(np.float32)

    def transposed(mse):
        A, B = eng.param(a), eng.param(b)
        return mse(L.nc_transpose(A, 0, 1), B), [A, B]

    def sliced(mse):
        A, B = eng.param(a), eng.param(b)
        return mse(L.nc_slice(A, 0, 1, 3, 2), L.nc_slice(L.nc_transpose(B, 0, 1), 0, 2, 3, 1)), [A, B]

    def one_leaf(mse):
        A = eng.param(a)
        return mse(L.nc_slice(A, 0, 0, 3, 1), L.nc_slice(A, 0, 3, 3, 1)), [A]

    def two_terms(mse):
        A, B = eng.param(a), eng.param(b)
        p = L.nc_matmul(A, B)
        return L.nc_add(mse(p, eng.tensor(np.eye(6, dtype=np.float32))), L.nc_sum(L.nc_mul(p, p), abi.ALL_AXES, 0)), [A, B]

    def held(mse):
        A, B = eng.param(a), eng.param(b)
        first = L.nc_sum(L.nc_mul(A, A), abi.ALL_AXES, 0)
        assert L.nc_backward(first) == 0
        return mse(A, L.nc_transpose(B, 0, 1)), [A, B]

    for build in (transposed, sliced, one_leaf, two_terms, held):
        same(both_ways(eng, build, flags=flags), f"mse {build.__name__} flags={flags}")


def test_mse_of_other_operands_is_the_composite(eng):
    """Broadcast operands, a tensor against itself, and empty ones: as the ops give them."""
    L = eng.lib
    rng = np.random.default_rng(3)
    a, r = rng.standard_normal((5, 7)).astype(np.float32), rng.standard_normal(7).astype(np.float32)

    def broadcast(mse):
        A, R = eng.param(a), eng.param(r)
        return mse(A, R), [A, R]

    def itself(mse):
        A = eng.param(a)
        return mse(A, A), [A]

    for build in (broadcast, itself):
        same(both_ways(eng, build), f"mse {build.__name__}")
    e = eng.tensor(np.zeros((0, 3), np.float32))
    one, two = eng.read(L.nc_mse_loss(e, e)), eng.read(composite_mse(L, e, e))
    assert np.isnan(one) == np.isnan(two)


@pytest.mark.parametrize("shape,axes", [((70, 33), (0, 1)), ((3, 40, 50), (1, 2)), ((40, 3, 50), (0, 2)), ((5, 6), (0, 1)),
                                        ((7, 7), (0, 0))])
@pytest.mark.parametrize("first", ["transpose", "plain"])
def test_transpose_gradients_stored_and_added(eng, shape, axes, first):
    """A leaf read through a transpose and directly: whichever consumer's gradient comes first is stored into the fresh buffer,
    the other added; and once more into gradients that are held."""
    L = eng.lib
    rng = np.random.default_rng(sum(shape))
    x = rng.standard_normal(shape).astype(np.float32)
    tshape = list(shape)
    tshape[axes[0]], tshape[axes[1]] = tshape[axes[1]], tshape[axes[0]]
    gt, gp = rng.standard_normal(tshape).astype(np.float32), rng.standard_normal(shape).astype(np.float32)
    X = eng.param(x)
    want = None
    for step in range(2):
        def t_term():
            return L.nc_sum(L.nc_mul(L.nc_transpose(X, *axes), eng.tensor(gt)), abi.ALL_AXES, 0)

        def p_term():
            return L.nc_sum(L.nc_mul(X, eng.tensor(gp)), abi.ALL_AXES, 0)

        # the backward pass runs the newest node first
        late, early = (t_term, p_term) if first == "transpose" else (p_term, t_term)
        e = early()
        loss = L.nc_add(e, late())
        assert L.nc_backward(loss) == 0, L.nc_error(eng.ctx)
        back = np.swapaxes(gt, *axes)
        order = (back, gp) if first == "transpose" else (gp, back)
        want = order[0] + np.float32(0) if want is None else want + order[0]
        want = want + order[1]
        assert_bits(eng.grad(X), np.ascontiguousarray(want), f"step {step}")
        eng.step_end()
