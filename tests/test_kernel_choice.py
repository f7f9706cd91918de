"""Which kernel the products run on, asked of the library without a device: every choice is one that a launch can hold (a
dispatch counts its work-items in 32 bits), whatever the sizes."""
import pytest

from newch_amd import hip

MOST = 2 ** 32 - 1  # work-items of a launch


@pytest.fixture(scope="module")
def K():
    return hip.Kernels()


# long and thin int8 products: 16 x 16 or 16 x 32 tiles of 1024 lanes are the cheapest by what they load, and 2^22 of them are
# more lanes than a launch has
@pytest.mark.parametrize("M,N,Kd", [(16, 1 << 27, 64), (1 << 26, 16, 64), ((1 << 26) + 16, 8, 64), (1 << 15, 1 << 15, 0),
                                    (1 << 26, 16, 1), (1, 1 << 28, 128), (1 << 28, 1, 4096), (16, (1 << 26) + 1, 64),
                                    (33, 1 << 27, 100), (65, 1 << 26, 7)])
@pytest.mark.parametrize("align", [1, 4, 16])
@pytest.mark.parametrize("f32", [False, True])
def test_int8_product_fits_a_launch(K, M, N, Kd, align, f32):
    kernel, lanes = K.gemm_s8_plan(M, N, Kd, align, f32)
    assert kernel >= 0 and 0 < lanes <= MOST


def test_int8_product_of_refused_sizes(K):
    assert K.gemm_s8_plan(-1, 1, 1, 16)[0] == -1
    assert K.gemm_s8_plan(1, 1 << 31, 1, 16)[0] == -1


# batches of small matrices whose 256 x 256 tiles (512 lanes each) no launch holds: another tile runs them, or the call says so
@pytest.mark.parametrize("M,N,Kd,count,runs", [(256, 256, 32, 1 << 23, False), (4, 4, 32, (1 << 23) + 1, True),
                                               (32, 32, 32, 16777215, True), (32, 32, 32, 1 << 24, False),
                                               (16, 16, 4096, 1 << 24, False), (1 << 27, 16, 32, 1, True),
                                               (2 ** 31 - 1, 1, 1, 1, False), (64, 1 << 28, 64, 1, True)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("aligned", [False, True])
def test_fp32_product_fits_a_launch(K, ta, tb, M, N, Kd, count, runs, aligned):
    kernel, lanes = K.gemm_f32_plan(ta, tb, M, N, Kd, count, aligned)
    assert lanes <= MOST
    assert (kernel >= 0) == runs


def test_int8_products_of_short_rows_take_wide_tiles(K):
    """A tile's start and exchange count where K is short: many small tiles of a few bytes each are not the cheapest."""
    for M, N, Kd in ((4099, 4096, 8), (3072, 1024, 16), (8192, 300, 32), (768, 3072, 16), (256, 8192, 16), (2048, 1000, 1)):
        for align in (1, 4, 16):
            assert K.gemm_s8_plan(M, N, Kd, align)[0] >= 5, (M, N, Kd, align)
    assert K.gemm_s8_plan(16, 4096, 4096, 16)[0] == 0 and K.gemm_s8_plan(16, 4096, 4096, 16, True)[0] == 0
