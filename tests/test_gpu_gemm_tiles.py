"""The fp32 GEMM's kernels at their edges, against fp64: every kernel in every operand layout (each asserted), with rows,
columns and k that end inside a tile or a panel, operands that start off 16 bytes with odd leading dims, and
matrices of 1 to 3 rows.  What lies between the rows of the operands is NaN (nothing outside them may reach a
sum) and of C a guard value.  The bound is the K-term one of the other GEMM tests (pyoracle.gemm_excess)."""
import ctypes

import numpy as np
import pytest

from newch_amd import hip, hipmem
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu

GUARD = np.float32(12345.0)

# by layout (ta, tb): small and thin sizes, short K, K within a panel (which kernel each runs on: BY_KERNEL below)
SIZES = {
    (0, 1): [(1, 1, 476), (8, 520, 700), (1, 1, 220), (4760, 2, 269), (1, 1, 75), (199, 615, 559), (156, 2863, 36),
             (1, 1, 36), (33, 65, 31), (1, 1, 1), (2763, 170, 172), (204, 5476, 5), (137, 5793, 2), (1482, 689, 107),
             (515, 3830, 2), (5, 7, 0)],
    (0, 0): [(1, 1, 325), (1, 4158, 291), (17, 15, 317), (2, 3, 36), (130, 974, 578), (65, 4142, 2), (1, 1, 1),
             (5731, 65, 2), (1806, 287, 129), (296, 4138, 3), (3392, 257, 1), (2347, 400, 68), (538, 3639, 1),
             (1110, 2693, 1), (64, 2, 90)],
    (1, 0): [(1, 1, 259), (3, 2, 246), (4133, 5, 244), (2, 31, 35), (460, 292, 323), (83, 4193, 1), (1, 3, 1),
             (71, 5889, 2), (80, 5895, 66), (154, 5531, 2), (4998, 770, 99), (5471, 208, 3), (1026, 1979, 34),
             (866, 3458, 2)],
    (1, 1): [(1, 1, 325), (3, 129, 291), (130, 974, 578), (65, 4142, 2), (1806, 287, 129), (296, 4138, 3),
             (2347, 401, 68), (1110, 2693, 1), (2, 5, 33)],
}
CASES = [(ta, tb, *s) for (ta, tb), sizes in SIZES.items() for s in sizes]


@pytest.fixture(scope="module")
def K():
    return hip.Kernels()


def padded(a, ld, offset):
    """a's rows ld apart, `offset` floats into the buffer, NaN everywhere else."""
    flat = np.full(offset + a.shape[0] * ld + 4, np.nan, np.float32)
    flat[offset:offset + a.shape[0] * ld].reshape(a.shape[0], ld)[:, :a.shape[1]] = a
    return hipmem.DeviceBuffer.from_numpy(flat)


@pytest.mark.parametrize("ta,tb,M,N,Kd", CASES)
def test_gemm_f32_tiles(K, ta, tb, M, N, Kd):
    rng = np.random.default_rng(M + 3 * N + 7 * Kd + ta + 2 * tb)
    A = rng.standard_normal((Kd, M) if ta else (M, Kd)).astype(np.float32)
    B = rng.standard_normal((N, Kd) if tb else (Kd, N)).astype(np.float32)
    C0 = rng.standard_normal((M, N)).astype(np.float32)
    lda, ldb, ldc = A.shape[1] + 3, B.shape[1] + 1, N + 2
    print(f"gemm tile ta={ta} tb={tb} {M}x{N}x{Kd}", flush=True)
    Ad, Bd = padded(A, lda, 1), padded(B, ldb, 2)
    Cw = np.full((M, ldc), GUARD, np.float32)
    Cw[:, :N] = C0
    Cd = hipmem.DeviceBuffer.from_numpy(Cw)
    K.gemm_f32(ta, tb, M, N, Kd, 0.75, Ad.ptr + 4, lda, Bd.ptr + 8, ldb, 1.0, Cd.ptr, ldc)
    hipmem.synchronize()
    got = Cd.to_numpy(np.float32, (M, ldc))
    assert (got[:, N:] == GUARD).all(), "wrote past N"
    opA, opB = (A.T if ta else A).astype(np.float64), (B.T if tb else B).astype(np.float64)
    want = 0.75 * (opA @ opB) + C0
    terms = 0.75 * (np.abs(opA) @ np.abs(opB)) + np.abs(C0)
    assert O.gemm_excess(got[:, :N], want, terms, Kd + 1) <= 1.0


@pytest.mark.parametrize("ta,tb,M,N,Kd,count", [(0, 1, 197, 197, 64, 5), (1, 0, 3, 65, 70, 4), (0, 0, 40, 33, 45, 3)])
def test_gemm_f32_tiles_pointer_batch(K, ta, tb, M, N, Kd, count):
    """Matrices anywhere: each of the batch at its own 4-byte aligned address."""
    rng = np.random.default_rng(M + N + Kd)
    A = rng.standard_normal((count, Kd, M) if ta else (count, M, Kd)).astype(np.float32)
    B = rng.standard_normal((count, N, Kd) if tb else (count, Kd, N)).astype(np.float32)
    print(f"gemm pointer batch {count} of {M}x{N}x{Kd}", flush=True)
    Ad = [padded(A[i], A.shape[2], i % 4) for i in range(count)]
    Bd = [padded(B[i], B.shape[2], (i + 1) % 4) for i in range(count)]
    Cd = [hipmem.DeviceBuffer.from_numpy(np.full(M * N + 4, GUARD, np.float32)) for _ in range(count)]

    def table(ptrs):
        return hipmem.DeviceBuffer.from_numpy(np.array(ptrs, np.uint64))

    pa = table([d.ptr + 4 * (i % 4) for i, d in enumerate(Ad)])
    pb = table([d.ptr + 4 * ((i + 1) % 4) for i, d in enumerate(Bd)])
    pc = table([d.ptr + 4 * (i % 3) for i, d in enumerate(Cd)])
    K.gemm_f32_batched(ta, tb, M, N, Kd, 1.0, ctypes.c_void_p(pa.ptr), A.shape[2], ctypes.c_void_p(pb.ptr), B.shape[2],
                       0.0, ctypes.c_void_p(pc.ptr), N, count)
    hipmem.synchronize()
    for i in range(count):
        flat = Cd[i].to_numpy(np.float32, M * N + 4)
        got = flat[i % 3:i % 3 + M * N].reshape(M, N)
        assert (flat[:i % 3] == GUARD).all() and (flat[i % 3 + M * N:] == GUARD).all(), "wrote outside C"
        opA, opB = (A[i].T if ta else A[i]).astype(np.float64), (B[i].T if tb else B[i]).astype(np.float64)
        assert O.gemm_excess(got, opA @ opB, np.abs(opA) @ np.abs(opB), Kd) <= 1.0, f"matrix {i}"


# by layout, one size for each kernel in gemm_f32_plan's order: the 14 register-staged tiles (operands not 16-byte aligned, K
# ending inside a panel), then the 256 x 256 and 128 x 128 direct-to-LDS ones (aligned operands)
BY_KERNEL = {
    (0, 0): [(4674, 644, 34), (3447, 604, 33), (129, 5702, 34), (1355, 739, 65), (5001, 266, 33), (68, 6068, 33),
             (6097, 67, 139), (33, 4411, 73), (37, 4183, 33), (1, 1, 33), (4892, 17, 490), (1, 1, 225), (1, 4186, 262),
             (1, 1, 323), (2308, 5152, 96), (584, 4900, 96)],
    (0, 1): [(3375, 2244, 33), (3447, 604, 33), (129, 5702, 34), (353, 2761, 98), (5001, 266, 33), (68, 6068, 33),
             (65, 5896, 178), (1, 1, 33), (79, 4110, 34), (1, 1, 65), (18, 4171, 570), (4397, 1, 283), (1, 1, 193),
             (1, 1, 385), (2116, 5732, 96), (584, 4900, 96)],
    (1, 0): [(938, 5749, 33), (3447, 604, 33), (461, 6186, 41), (4603, 309, 35), (129, 5702, 34), (68, 6068, 33),
             (5914, 71, 65), (37, 4183, 33), (79, 4110, 34), (1, 1, 33), (17, 4297, 334), (1, 1, 225), (1, 4186, 262),
             (1, 1, 257), (2308, 4572, 96), (584, 4900, 96)],
    (1, 1): [(4674, 644, 34), (3447, 604, 33), (129, 5702, 34), (1355, 739, 65), (5001, 266, 33), (68, 6068, 33),
             (6097, 67, 139), (33, 4411, 73), (37, 4183, 33), (1, 1, 33), (4892, 17, 490), (1, 1, 225), (1, 4186, 262),
             (1, 1, 323), (2308, 5152, 96), (584, 4900, 96)],
}


@pytest.mark.parametrize("ta,tb,kernel", [(ta, tb, k) for ta, tb in BY_KERNEL for k in range(16)])
def test_gemm_f32_by_kernel(K, ta, tb, kernel):
    M, N, Kd = BY_KERNEL[ta, tb][kernel]
    aligned = kernel >= 14
    assert K.gemm_f32_plan(ta, tb, M, N, Kd, 1, aligned)[0] == kernel, "the choice has moved: another size has to cover it"
    if not aligned:
        test_gemm_f32_tiles(K, ta, tb, M, N, Kd)
        return
    rng = np.random.default_rng(M + 3 * N + 7 * Kd + ta + 2 * tb)
    A = rng.standard_normal((Kd, M) if ta else (M, Kd)).astype(np.float32)
    B = rng.standard_normal((N, Kd) if tb else (Kd, N)).astype(np.float32)
    lda, ldb, ldc = A.shape[1] + 4, B.shape[1] + 8, N + 1
    print(f"gemm kernel {kernel} ta={ta} tb={tb} {M}x{N}x{Kd}", flush=True)
    Ad, Bd = padded(A, lda, 4), padded(B, ldb, 8)
    Cd = hipmem.DeviceBuffer.from_numpy(np.full((M, ldc), GUARD, np.float32))
    K.gemm_f32(ta, tb, M, N, Kd, 1.0, Ad.ptr + 16, lda, Bd.ptr + 32, ldb, 0.0, Cd.ptr, ldc)
    hipmem.synchronize()
    got = Cd.to_numpy(np.float32, (M, ldc))
    assert (got[:, N:] == GUARD).all(), "wrote past N"
    opA, opB = (A.T if ta else A).astype(np.float64), (B.T if tb else B).astype(np.float64)
    assert O.gemm_excess(got[:, :N], opA @ opB, np.abs(opA) @ np.abs(opB), Kd) <= 1.0
    # the same sums from operands that are not aligned, which go to a staged tile: the same bits where it does not split K
    other = K.gemm_f32_plan(ta, tb, M, N, Kd, 1, False)[0]
    if other in (0, 2, 5):
        Au, Bu = padded(A, A.shape[1] + 3, 1), padded(B, B.shape[1] + 1, 2)
        K.gemm_f32(ta, tb, M, N, Kd, 1.0, Au.ptr + 4, A.shape[1] + 3, Bu.ptr + 8, B.shape[1] + 1, 0.0, Cd.ptr, ldc)
        hipmem.synchronize()
        np.testing.assert_array_equal(Cd.to_numpy(np.float32, (M, ldc)), got)
