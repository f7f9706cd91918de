"""The int8 product at the edges of its tiles, K splits and alignments: whole numbers, so equal to the 64-bit product
bit for bit; the fused linear equal to its own steps in fp32."""
import numpy as np
import pytest

from newch_amd import hip, hipmem

pytestmark = pytest.mark.gpu

# (M, N, K): one past and one short of the tiles' edges; K within a step, a whole number of steps, short of and past a wave's
# turn, unaligned rows.  (Which tile a shape runs on: the tests by kernel below.)
SHAPES = [(1, 1, 1), (1, 17, 15), (15, 16, 16), (16, 16, 127), (17, 15, 128), (3, 100, 129), (16, 4096, 2048),
          (1, 4100, 2049), (16, 8200, 1031), (33, 4090, 260), (64, 4096, 1000), (127, 4096, 520), (129, 4099, 333),
          (257, 4097, 640), (512, 4096, 250), (1000, 4000, 384), (1030, 4100, 77), (4100, 4090, 65),
          (4097, 4096, 128), (5, 70000, 129), (31, 33, 6243), (16, 64, 0)]


GUARD = -7


@pytest.fixture(scope="module")
def K():
    return hip.Kernels()


def ints(rng, rows, cols):
    return rng.integers(-127, 128, (rows, cols), dtype=np.int8)


def placed(a, ld, off):
    """`a` on the device, rows `ld` bytes apart from byte `off` of its buffer."""
    flat = np.full(off + a.shape[0] * ld + 1, 99, np.int8)
    flat[off:off + a.shape[0] * ld].reshape(a.shape[0], ld)[:, :a.shape[1]] = a
    return hipmem.DeviceBuffer.from_numpy(flat)


def product(a, b):
    return (a.astype(np.float64) @ b.astype(np.float64).T).astype(np.int32)


@pytest.mark.parametrize("M,N,Kd", SHAPES)
@pytest.mark.parametrize("pad,off", [(0, 0), (5, 3)])
def test_gemm_s8_exact(K, M, N, Kd, pad, off):
    rng = np.random.default_rng(M + N + Kd)
    a, b = ints(rng, M, Kd), ints(rng, N, Kd)
    lda, ldb, ldc = Kd + pad, Kd + 2 * pad, N + pad
    da, db = placed(a, lda, off), placed(b, ldb, off)
    dc = hipmem.DeviceBuffer.from_numpy(np.full(M * ldc + 4, GUARD, np.int32))
    K.gemm_s8_nt(M, N, Kd, da.ptr + off, lda, db.ptr + off, ldb, dc.ptr, ldc)
    flat = dc.to_numpy(np.int32, M * ldc + 4)
    c = flat[:M * ldc].reshape(M, ldc)
    np.testing.assert_array_equal(c[:, :N], product(a, b))
    assert (c[:, N:] == GUARD).all() and (flat[M * ldc:] == GUARD).all(), "wrote outside"


@pytest.mark.parametrize("M,N,Kd", [(1, 1, 1), (7, 515, 130), (16, 4096, 512), (40, 4097, 257), (130, 4098, 129),
                                    (300, 4095, 384)])
@pytest.mark.parametrize("bias", [True, False])
def test_linear_int8_equals_its_steps(K, M, N, Kd, bias):
    rng = np.random.default_rng(M + N + Kd)
    x = rng.standard_normal((M, Kd)).astype(np.float32)
    w, ws = ints(rng, N, Kd), (rng.random(N) + 0.5).astype(np.float32)
    b = rng.standard_normal(N).astype(np.float32) if bias else np.zeros(N, np.float32)
    dx, dw, dws, db = (hipmem.DeviceBuffer.from_numpy(v) for v in (x, w, ws, b))
    dy = hipmem.DeviceBuffer.from_numpy(np.zeros((M, N), np.float32))
    n = K.linear_int8_workspace(M, Kd)
    scratch = hipmem.DeviceBuffer.from_numpy(np.zeros(n, np.int8))
    K.linear_int8(M, Kd, N, dx.ptr, dw.ptr, dws.ptr, db.ptr if bias else None, dy.ptr, scratch.ptr, n)
    dq, ds = (hipmem.DeviceBuffer.from_numpy(v) for v in (np.zeros((M, Kd), np.int8), np.zeros(M, np.float32)))
    K.quantize_rows(M, Kd, dx.ptr, dq.ptr, ds.ptr)
    q, s = dq.to_numpy(np.int8, M * Kd).reshape(M, Kd), ds.to_numpy(np.float32, M)
    want = product(q, w).astype(np.float32) * s[:, None] * ws + b
    np.testing.assert_array_equal(dy.to_numpy(np.float32, M * N).reshape(M, N), want)


@pytest.mark.parametrize("Kd", [2 ** 31 - 1, 2 ** 31 - 129, 2 ** 31 - 2048])
def test_gemm_s8_longest_rows(K, Kd):
    """Rows that end at or just short of 2^31 bytes: a step index of 32 bits with a sign would pass its end and go negative.
    Ones against zeros but for a few places around the steps' edges and the row's end."""
    a, b = hipmem.DeviceBuffer(Kd), hipmem.DeviceBuffer(Kd)
    K.fill(a.ptr, 1, 1, Kd)
    b.zero()
    at = [0, 127, 128, Kd // 2, Kd - 2049, Kd - 130, Kd - 17, Kd - 16, Kd - 1]
    for i in at:
        b.upload(np.array([7], np.int8), i)
    c = hipmem.DeviceBuffer.from_numpy(np.full(2, GUARD, np.int32))
    print(f"gemm_s8 1x1x{Kd}", flush=True)
    K.gemm_s8_nt(1, 1, Kd, a.ptr, Kd, b.ptr, Kd, c.ptr, 1)
    assert c.to_numpy(np.int32, 2).tolist() == [7 * len(at), GUARD]


# by kernel (gemm_s8_plan: 16x16, 16x32, 32x32, 64x32, 64x64 with K over the waves, 128, 256, direct to LDS) and alignment
# of the rows: M, N and K that end inside a tile and a step
BY_KERNEL = {
    (0, 1): (1, 1, 43), (0, 4): (17, 15, 252), (0, 16): (15, 33, 272), (1, 1): (1, 4260, 64), (1, 4): (3, 4225, 140),
    (1, 16): (1, 4321, 288), (2, 1): (4281, 1, 207), (2, 4): (4151, 1, 40), (2, 16): (4113, 1, 160), (3, 1): (2767, 69, 144),
    (3, 4): (4177, 37, 480), (3, 16): (4099, 40, 1088), (4, 1): (3130, 161, 496), (4, 4): (3538, 202, 96),
    (4, 16): (2802, 281, 368), (5, 1): (3554, 136, 40), (5, 4): (3554, 136, 40), (5, 16): (136, 3372, 48),
    (6, 1): (4023, 4024, 535), (6, 4): (4011, 3910, 1192), (7, 16): (3900, 3847, 128), (7, 17): (3900, 3847, 256),
}
LINEAR_BY_KERNEL = {
    (0, 1): (1, 1, 151), (0, 4): (17, 15, 140), (0, 16): (15, 33, 160), (1, 1): (1, 4211, 202), (1, 4): (1, 4225, 140),
    (1, 16): (1, 4231, 416), (2, 1): (4281, 1, 207), (2, 4): (4367, 2, 204), (2, 16): (4113, 1, 160), (3, 1): (4148, 43, 387),
    (3, 4): (2772, 65, 1652), (3, 16): (4376, 34, 1120), (4, 1): (3533, 207, 133), (4, 4): (226, 3075, 140),
    (4, 16): (609, 1219, 144), (5, 1): (581, 1690, 131), (5, 4): (1553, 658, 132), (5, 16): (884, 1462, 144),
    (6, 1): (4068, 3885, 1373), (7, 16): (3967, 3972, 128), (7, 17): (3967, 3972, 256),
}


@pytest.mark.parametrize("kernel,align", BY_KERNEL)
def test_gemm_s8_by_kernel(K, kernel, align):
    M, N, Kd = BY_KERNEL[kernel, align]
    align = min(align, 16)  # 17: whole pairs of steps, the pipelined loop
    ld = -(-Kd // align) * align + (5 if align == 1 else 0)
    off = 3 if align == 1 else align
    K.set_grid_cus(256)
    try:
        assert K.gemm_s8_plan(M, N, Kd, align)[0] == kernel, "the choice has moved: another shape has to cover this kernel"
        rng = np.random.default_rng(kernel * 20 + align)
        a, b = ints(rng, M, Kd), ints(rng, N, Kd)
        da, db = placed(a, ld, off), placed(b, ld, off)
        dc = hipmem.DeviceBuffer.from_numpy(np.full(M * N + 4, GUARD, np.int32))
        print(f"gemm_s8 kernel {kernel} align {align} {M}x{N}x{Kd}", flush=True)
        K.gemm_s8_nt(M, N, Kd, da.ptr + off, ld, db.ptr + off, ld, dc.ptr, N)
        hipmem.synchronize()
    finally:
        K.set_grid_cus(0)
    flat = dc.to_numpy(np.int32, M * N + 4)
    np.testing.assert_array_equal(flat[:M * N].reshape(M, N), product(a, b))
    assert (flat[M * N:] == GUARD).all(), "wrote outside"


@pytest.mark.parametrize("kernel,align", LINEAR_BY_KERNEL)
def test_linear_int8_by_kernel(K, kernel, align):
    M, N, Kd = LINEAR_BY_KERNEL[kernel, align]
    assert min(align, 16) == (16 if Kd % 16 == 0 else 4 if Kd % 4 == 0 else 1)
    K.set_grid_cus(256)
    try:
        assert K.gemm_s8_plan(M, N, Kd, min(align, 16), True)[0] == kernel, "the choice has moved"
        print(f"linear_int8 kernel {kernel} {M}x{N}x{Kd}", flush=True)
        test_linear_int8_equals_its_steps(K, M, N, Kd, True)
    finally:
        K.set_grid_cus(0)
