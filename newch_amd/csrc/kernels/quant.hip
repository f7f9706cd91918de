// int8 absmax quantization and dequantization (quantize_row / nc_quantize_rows, ops_quant.c:11-39;
// dequantize = to_dtype i8 -> f32 then a row-broadcast multiply, ops_shape.c:491-504 and
// ops_elementwise.c:22).
//
// quantize: a row of up to 65536 floats stays in registers -- in one wave up to 1024, else spread over a
// workgroup of 256, 512 or 1024 lanes -- so w is read once (4 B/el) and q written once (1 B/el, four int8
// packed per 32-bit store), whatever the row's length and alignment.  Rows are independent, so 48
// stacked 4096x4096 matrices are a single launch.
// dequantize: a streaming map, each lane reading 4 int8 (one 32-bit load) and writing one 128-bit
// float vector, lane-contiguous so loads and stores coalesce.
//
// Both are bound by memory.  us, element by element (rows past 8192 floats, or not of whole aligned float4s)
// and now: 4096 x 11008 quantized 71 and 38 (6.0 TB/s), 4096 x 9001 60 and 32, 8192 x 5001 65 and 35, 1000 x 60000 200
// and 67; 8192 x 5001 expanded 42 and 29, 2000 x 30001 105 and 41.
//
// Arithmetic is the reference's exactly: amax = max |x| (fmaxf, NaN ignored, order-free),
// s = amax / 127 (1 for a zero row), inv = 1 / s, q = clamp(rne(x * inv), -127, 127); the
// float -> int8 conversion maps NaN to 0 as the reference's truncating conversion does.
#include "common.hpp"
#include "intdiv.hpp"

namespace nchip {

constexpr int kQB = 256;

__device__ __forceinline__ int quant1(float x, float inv) {
    const float v = __builtin_rintf(x * inv);
    const float c = v > 127.0f ? 127.0f : v < -127.0f ? -127.0f : v;
    return c != c ? 0 : (int)c;
}

__device__ __forceinline__ uint32_t pack4(int a, int b, int c, int d) {
    return (uint32_t)(a & 0xff) | ((uint32_t)(b & 0xff) << 8) | ((uint32_t)(c & 0xff) << 16) |
           ((uint32_t)(d & 0xff) << 24);
}

__device__ __forceinline__ float amax4(float m, f4 v) {
    return __builtin_fmaxf(m, __builtin_fmaxf(__builtin_fmaxf(__builtin_fabsf(v.x), __builtin_fabsf(v.y)),
                                              __builtin_fmaxf(__builtin_fabsf(v.z), __builtin_fabsf(v.w))));
}

typedef uint32_t u32u __attribute__((aligned(1)));

// piece j (columns 4 j .. 4 j + 3) of a row quantized; FULL: the row is made of whole pieces and q 4-byte aligned
template <bool FULL>
__device__ __forceinline__ void quant_store(f4 v, float inv, int8_t *qr, int C, int j) {
    const uint32_t p = pack4(quant1(v.x, inv), quant1(v.y, inv), quant1(v.z, inv), quant1(v.w, inv));
    if (FULL) {
        __builtin_nontemporal_store(p, (uint32_t *)qr + j);
    } else if (4 * j + 4 <= C) {
        *(u32u *)(qr + 4 * j) = p;
    } else {
#pragma unroll
        for (int e = 0; e < 3; e++)
            if (4 * j + e < C) qr[4 * j + e] = (int8_t)(p >> (8 * e));
    }
}

// Rows of up to 256 VPL floats: a wave per row.  AL: 16-byte aligned rows of whole pieces.
template <int VPL, bool AL>
__global__ __launch_bounds__(kQB) void k_quant_reg(const float *__restrict__ w, int8_t *__restrict__ q,
                                                   float *__restrict__ scale, int64_t rows, int cols) {
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t r = ((int64_t)blockIdx.x * kQB + threadIdx.x) / kWave;
    if (r >= rows) return;
    const float *wr = w + r * cols;
    f4 v[VPL];
    float amax = 0.0f;
#pragma unroll
    for (int k = 0; k < VPL; k++) {
        const int j = lane + k * kWave;
        v[k] = 4 * j < cols ? row_load<AL>(wr, cols, j, 0.0f) : f4{0.0f, 0.0f, 0.0f, 0.0f};
        amax = amax4(amax, v[k]);
    }
    amax = wave_max_nan_skip(amax);
    const float s = amax > 0.0f ? amax / 127.0f : 1.0f;
    const float inv = 1.0f / s;
    int8_t *qr = q + r * cols;
#pragma unroll
    for (int k = 0; k < VPL; k++) {
        const int j = lane + k * kWave;
        if (4 * j < cols) quant_store<AL>(v[k], inv, qr, cols, j);
    }
    if (lane == 0) scale[r] = s;
}

// Longer rows: a workgroup of NT lanes per row, each lane holding VPT float4 of it, the waves' maxima meeting in LDS,
// and a grid with a workgroup for every row.  A wave then has a part of a row in flight and many rows are resident at
// once: the 48 x 4096 x 4096 quantization runs at 665-673 us where one wave per 16 KiB row took 712-723, and the same
// workgroups looping over rows took 790-804.  FULL: aligned rows of VPT NT whole float4s, without bounds.
template <int VPT, int NT, bool FULL>
__global__ __launch_bounds__(NT) void k_quant_wg(const float *__restrict__ w, int8_t *__restrict__ q,
                                                 float *__restrict__ scale, int cols) {
    __shared__ float sh[NT / kWave];
    const int tid = threadIdx.x;
    const int64_t r = blockIdx.x;
    const float *wr = w + r * cols;
    f4 v[VPT];
    float amax = 0.0f;
#pragma unroll
    for (int k = 0; k < VPT; k++)
        v[k] = FULL ? row_load<true>(wr, cols, tid + k * NT, 0.0f) : row_load_or(wr, cols, tid + k * NT, 0.0f);
#pragma unroll
    for (int k = 0; k < VPT; k++) amax = amax4(amax, v[k]);
    amax = wave_max_nan_skip(amax);
    if ((tid & (kWave - 1)) == 0) sh[tid / kWave] = amax;
    __syncthreads();
    amax = sh[0];
#pragma unroll
    for (int i = 1; i < NT / kWave; i++) amax = __builtin_fmaxf(amax, sh[i]);
    const float s = amax > 0.0f ? amax / 127.0f : 1.0f;
    const float inv = 1.0f / s;
    int8_t *qr = q + r * cols;
#pragma unroll
    for (int k = 0; k < VPT; k++) {
        const int j = tid + k * NT;
        if (FULL || 4 * j < cols) quant_store<FULL>(v[k], inv, qr, cols, j);
    }
    if (tid == 0) scale[r] = s;
}

// rows past 65536 floats: one workgroup per row, two passes over the (L2-resident) row
__global__ __launch_bounds__(kQB) void k_quant_blk(const float *__restrict__ w, int8_t *__restrict__ q,
                                                   float *__restrict__ scale, int64_t rows, int64_t cols) {
    __shared__ float sh[kQB / kWave];
    for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
        const float *wr = w + r * cols;
        float amax = 0.0f;
        for (int64_t i = threadIdx.x; i < cols; i += kQB) amax = __builtin_fmaxf(amax, __builtin_fabsf(wr[i]));
        amax = wave_max_nan_skip(amax);
        __syncthreads();
        if ((threadIdx.x & (kWave - 1)) == 0) sh[threadIdx.x / kWave] = amax;
        __syncthreads();
        amax = sh[0];
#pragma unroll
        for (int i = 1; i < kQB / kWave; i++) amax = __builtin_fmaxf(amax, sh[i]);
        const float s = amax > 0.0f ? amax / 127.0f : 1.0f;
        const float inv = 1.0f / s;
        for (int64_t i = threadIdx.x; i < cols; i += kQB) q[r * cols + i] = (int8_t)quant1(wr[i], inv);
        if (threadIdx.x == 0) scale[r] = s;
    }
}

// Lane-contiguous dequantization: lane j reads 4 int8 as one 32-bit word and writes one 128-bit
// float vector, so a wave reads 256 contiguous bytes and writes 1 KiB contiguous; U words in
// flight per lane.  Requires cols % 4 == 0, q 4-byte and w 16-byte aligned, rows * cols / 4 < 2^32.
#ifndef NC_DQ_UNROLL
#define NC_DQ_UNROLL 2
#endif
#ifndef NC_DQ_BLOCK
#define NC_DQ_BLOCK 128
#endif
#ifndef NC_DQ_GRID_PER_CU
#define NC_DQ_GRID_PER_CU 65536
#endif
constexpr int kDqU = NC_DQ_UNROLL;
constexpr int kDqB = NC_DQ_BLOCK;
__global__ __launch_bounds__(kDqB) void k_dequant4(const uint32_t *__restrict__ q, const float *__restrict__ scale,
                                                  f4 *__restrict__ w, uint32_t n4, IntDiv per_row4) {
    const uint64_t step = (uint64_t)gridDim.x * kDqB * kDqU;
    for (uint64_t base = (uint64_t)blockIdx.x * kDqB * kDqU + threadIdx.x; base < n4; base += step) {
        uint32_t v[kDqU];
#pragma unroll
        for (int u = 0; u < kDqU; u++) {
            const uint64_t j = base + (uint64_t)u * kDqB;
            if (j < n4) v[u] = __builtin_nontemporal_load(q + j);
        }
#pragma unroll
        for (int u = 0; u < kDqU; u++) {
            const uint64_t j = base + (uint64_t)u * kDqB;
            if (j < n4) {
                const float s = scale[per_row4.div((uint32_t)j)];
                const uint32_t x = v[u];
                f4 r;
                r.x = (float)(int8_t)(x & 0xffu) * s;
                r.y = (float)(int8_t)((x >> 8) & 0xffu) * s;
                r.z = (float)(int8_t)((x >> 16) & 0xffu) * s;
                r.w = (float)(int8_t)(x >> 24) * s;
                __builtin_nontemporal_store(r, w + j);
            }
        }
    }
}

// The same over element groups e .. e + 3 of the whole array where rows are not a multiple of 4 long (cols >= 4: a
// group meets at most two rows) or the arrays not aligned; the last rows * cols % 4 elements go one by one.
__global__ __launch_bounds__(kQB) void k_dequant4_any(const int8_t *__restrict__ q, const float *__restrict__ scale,
                                                      float *__restrict__ w, uint32_t n, IntDiv row) {
    const uint32_t e = (blockIdx.x * kQB + threadIdx.x) * 4, C = row.d;
    if (e >= n) return;
    const uint32_t r = row.div(e), c = e - r * C;
    const bool two = c + 4 > C && e + (C - c) < n;  // the group crosses into row r + 1
    const float s0 = scale[r], s1 = two ? scale[r + 1] : s0;
    if (e + 4 <= n) {
        const uint32_t x = *(const u32u *)(q + e);
        f4 o;
#pragma unroll
        for (int j = 0; j < 4; j++) o[j] = (float)(int8_t)(x >> (8 * j) & 0xffu) * (c + j >= C ? s1 : s0);
        __builtin_nontemporal_store(o, (f4u *)(w + e));
    } else {
#pragma unroll
        for (int j = 0; j < 3; j++)
            if (e + j < n) w[e + j] = (float)q[e + j] * (c + j >= C ? s1 : s0);
    }
}

__global__ __launch_bounds__(kQB) void k_dequant1(const int8_t *__restrict__ q, const float *__restrict__ scale,
                                                  float *__restrict__ w, int64_t n, int64_t cols) {
    const int64_t step = (int64_t)gridDim.x * kQB;
    for (int64_t i = (int64_t)blockIdx.x * kQB + threadIdx.x; i < n; i += step) w[i] = (float)q[i] * scale[i / cols];
}

template <int VPL>
static void quant_wave(bool al, const float *w, int8_t *q, float *scale, int64_t rows, int C, hipStream_t st) {
    const unsigned g = (unsigned)((rows + kQB / kWave - 1) / (kQB / kWave));
    if (al) hipLaunchKernelGGL((k_quant_reg<VPL, true>), g, kQB, 0, st, w, q, scale, rows, C);
    else hipLaunchKernelGGL((k_quant_reg<VPL, false>), g, kQB, 0, st, w, q, scale, rows, C);
}

template <int VPT, int NT>
static void quant_wg(bool al, const float *w, int8_t *q, float *scale, int64_t rows, int C, hipStream_t st) {
    if (al && C == 4 * VPT * NT)
        hipLaunchKernelGGL((k_quant_wg<VPT, NT, true>), (unsigned)rows, NT, 0, st, w, q, scale, C);
    else
        hipLaunchKernelGGL((k_quant_wg<VPT, NT, false>), (unsigned)rows, NT, 0, st, w, q, scale, C);
}

}  // namespace nchip

using namespace nchip;

extern "C" NC_HIP_API int nc_hip_quantize_rows(int64_t rows, int64_t cols, const float *w, int8_t *q, float *scale,
                                               void *stream) {
    if (rows < 0 || cols < 0) return set_error(NC_HIP_ERR_ARG, "nc_hip_quantize_rows: negative size");
    if (rows == 0) return NC_HIP_OK;
    hipStream_t st = as_stream(stream);
    if (cols == 0) {  // empty rows: scale 1
        nc_hip_fill(scale, 4, 0x3f800000u, rows, stream);
        return check_launch("nc_hip_quantize_rows");
    }
    const bool al = cols % 4 == 0 && aligned16(w) && ((uintptr_t)q & 3u) == 0;
    // a launch's rows: four a workgroup of 256 lanes in the wave kernels, one a workgroup in the others
    const int64_t most = cols < 1024 ? kMaxLanes / kWave / 4 * 4 : kWgRowsPerLaunch;
    if (cols <= 65536 && rows > most) {
        const int rc = nc_hip_quantize_rows(most, cols, w, q, scale, stream);
        return rc ? rc : nc_hip_quantize_rows(rows - most, cols, w + most * cols, q + most * cols, scale + most, stream);
    }
    if (cols > 65536) {
        const unsigned g = (unsigned)(rows < num_cus() * 8 ? rows : num_cus() * 8);
        hipLaunchKernelGGL(k_quant_blk, g, kQB, 0, st, w, q, scale, rows, cols);
        return check_launch("nc_hip_quantize_rows");
    }
    const int C = (int)cols;
    // A wave a row while four pieces a lane hold it, else the smallest workgroup whose lanes hold it in 8 (12, 16 past
    // 16384: rows there are rare and every wave of the CU is taken).  us, workgroups of 256 / 512 / 1024 lanes: 4096
    // rows of 11008 39.7 / 37.9 / 41.4, of 9001 33.6 / 31.6 / 37.8, 2048 of 16384 29.7 / 27.9 / 28.0.
    if (C <= 256) quant_wave<1>(al, w, q, scale, rows, C, st);
    else if (C <= 512) quant_wave<2>(al, w, q, scale, rows, C, st);
    else if (C <= 768) quant_wave<3>(al, w, q, scale, rows, C, st);
    else if (C < 1024 || (C == 1024 && !al)) quant_wave<4>(al, w, q, scale, rows, C, st);
    else if (C <= 1024) quant_wg<1, 256>(al, w, q, scale, rows, C, st);
    else if (C <= 2048) quant_wg<2, 256>(al, w, q, scale, rows, C, st);
    else if (C <= 3072) quant_wg<3, 256>(al, w, q, scale, rows, C, st);
    else if (C <= 4096) quant_wg<4, 256>(al, w, q, scale, rows, C, st);
    else if (C <= 5120) quant_wg<5, 256>(al, w, q, scale, rows, C, st);
    else if (C <= 6144) quant_wg<6, 256>(al, w, q, scale, rows, C, st);
    else if (C <= 7168) quant_wg<7, 256>(al, w, q, scale, rows, C, st);
    else if (C <= 8192) quant_wg<8, 256>(al, w, q, scale, rows, C, st);
    else if (C <= 10240) quant_wg<5, 512>(al, w, q, scale, rows, C, st);
    else if (C <= 12288) quant_wg<6, 512>(al, w, q, scale, rows, C, st);
    else if (C <= 16384) quant_wg<8, 512>(al, w, q, scale, rows, C, st);
    else if (C <= 24576) quant_wg<12, 512>(al, w, q, scale, rows, C, st);
    else if (C <= 32768) quant_wg<8, 1024>(al, w, q, scale, rows, C, st);
    else if (C <= 49152) quant_wg<12, 1024>(al, w, q, scale, rows, C, st);
    else quant_wg<16, 1024>(al, w, q, scale, rows, C, st);
    return check_launch("nc_hip_quantize_rows");
}

extern "C" NC_HIP_API int nc_hip_dequantize_rows(int64_t rows, int64_t cols, const int8_t *q, const float *scale,
                                                 float *w, void *stream) {
    if (rows < 0 || cols < 0) return set_error(NC_HIP_ERR_ARG, "nc_hip_dequantize_rows: negative size");
    const int64_t n = rows * cols;
    if (n == 0) return NC_HIP_OK;
    hipStream_t st = as_stream(stream);
    if (cols % 4 == 0 && ((uintptr_t)q & 3u) == 0 && aligned16(w) && n / 4 < (int64_t)UINT32_MAX) {
        const int64_t n4 = n / 4;
        hipLaunchKernelGGL(k_dequant4, stream_grid((n4 + kDqU - 1) / kDqU, kDqB, NC_DQ_GRID_PER_CU), kDqB, 0, st, (const uint32_t *)q,
                           scale, (f4 *)w, (uint32_t)n4, IntDiv((uint32_t)(cols / 4)));
    } else if (cols >= 4 && cols <= INT32_MAX && n < (int64_t)UINT32_MAX - 4 * kQB) {
        const unsigned grid = (unsigned)((n + 4 * kQB - 1) / (4 * kQB));
        hipLaunchKernelGGL(k_dequant4_any, grid, kQB, 0, st, q, scale, w, (uint32_t)n, IntDiv((uint32_t)cols));
    } else {
        hipLaunchKernelGGL(k_dequant1, stream_grid(n, kQB, 16), kQB, 0, st, q, scale, w, n, cols);
    }
    return check_launch("nc_hip_dequantize_rows");
}
