// Shared pieces of the fp32 GEMM kernels (gemm.hip: entry points and the 256 x 256 direct-to-LDS kernel;
// gemm_tile.hpp: the register-staged tiles).
#pragma once

#include "common.hpp"

namespace nchip {

constexpr int kSgGroupM = 8;  // tile-rows per group in the block order

struct SgBatch {
    int nb;  // 0: one matrix per operand
    int64_t shape[NC_HIP_MAX_DIMS];
    int64_t st[3][NC_HIP_MAX_DIMS];  // element strides of A, B, C per batch axis
};

struct SgArgs {
    const float *A, *B;
    float *C;
    const float *const *pa;  // pointer-array batches (instead of strides) when set
    const float *const *pb;
    float *const *pc;
    int64_t lda, ldb, ldc;
    int M, N, K;
    float alpha, beta;
    const float *bias;  // N floats added to every row after alpha A B + beta C, or none
    int tiles_m, tiles_n;
    SgBatch bat;
};

// global-memory views, so loads are global_load (counted by vmcnt alone) rather than flat
typedef const __attribute__((address_space(1))) float gfloat;
typedef const __attribute__((address_space(1))) f4 gf4;
typedef const __attribute__((address_space(1))) f4u gf4u;

// a / b for wave-uniform operands, the quotient kept in a scalar register
__device__ __forceinline__ uint32_t udiv(uint32_t a, uint32_t b) { return __builtin_amdgcn_readfirstlane(a / b); }

// element offset of batch matrix `idx` for operand o (0 A, 1 B, 2 C); batch counts and extents fit 32 bits
__device__ __forceinline__ int64_t batch_off(const SgBatch &bt, int o, uint32_t idx) {
    int64_t off = 0;
    for (int d = bt.nb - 1; d >= 0; d--) {
        const uint32_t e = (uint32_t)bt.shape[d], q = udiv(idx, e);
        off += (int64_t)(idx - q * e) * bt.st[o][d];
        idx = q;
    }
    return off;
}

// The workgroup's tile: block -> (batch matrix, tile) with XCD-contiguous runs and groups of
// kSgGroupM tile-rows; the batch matrix's operands.
struct TileAt {
    int m0, n0;
    const float *A, *B;
    float *C;
};

template <int BM, int BN>
__device__ __forceinline__ TileAt locate(const SgArgs &p) {
    // XCD x runs blocks b with b % 8 == x: it gets the x-th of 8 contiguous runs of tiles
    const uint32_t nblk = gridDim.x, x = blockIdx.x & 7, per = nblk >> 3, rem = nblk & 7;
    const uint32_t id = x * per + min(x, rem) + (blockIdx.x >> 3);
    const uint32_t per_batch = (uint32_t)p.tiles_m * (uint32_t)p.tiles_n;
    const uint32_t batch = udiv(id, per_batch);
    const int tile = (int)(id - batch * per_batch);
    const int per_group = kSgGroupM * p.tiles_n;
    const int group = (int)udiv(tile, per_group), in_group = tile - group * per_group;
    const int first_m = group * kSgGroupM;
    const int gsize = min(p.tiles_m - first_m, kSgGroupM);
    const int n = (int)udiv(in_group, gsize);
    TileAt at;
    at.m0 = (first_m + in_group - n * gsize) * BM;
    at.n0 = n * BN;
    if (p.pa) {
        at.A = p.pa[batch], at.B = p.pb[batch], at.C = p.pc[batch];
    } else {
        at.A = p.A + batch_off(p.bat, 0, batch), at.B = p.B + batch_off(p.bat, 1, batch);
        at.C = p.C + batch_off(p.bat, 2, batch);
    }
    return at;
}

// One 4-column piece of a C row: C = alpha acc + beta C (+ bias[n]), columns n .. n + 3 of which the
// first `cols` exist.  The bias is added to the rounded alpha acc + beta C, as a separate broadcast add
// of it would.
__device__ __forceinline__ void write4(const SgArgs &p, float *crow, int n, f4 acc) {
    f4 r = p.alpha * acc;
    if (n + 4 <= p.N) {
        f4u *c = (f4u *)(crow + n);
        if (p.beta != 0.0f) r = r + p.beta * (f4)*c;
        if (p.bias) r = r + (f4) * (const f4u *)(p.bias + n);
        *c = r;
    } else {
#pragma unroll
        for (int v = 0; v < 4; v++) {
            if (n + v >= p.N) break;
            float *c = crow + n + v;
            const float t = p.beta != 0.0f ? r[v] + p.beta * *c : r[v];
            *c = p.bias ? t + p.bias[n + v] : t;
        }
    }
}

// Runs a problem on tile `id` of kSgTiles (gemm_tile.hpp) for one operand layout: `ak` / `bk` = the
// operand is K-contiguous.  One translation unit each.
int sg_tile_nt(SgArgs &p, int id, int64_t count, hipStream_t st, const char *what);  // A and B K-contiguous
int sg_tile_nn(SgArgs &p, int id, int64_t count, hipStream_t st, const char *what);  // A K-, B N-contiguous
int sg_tile_tt(SgArgs &p, int id, int64_t count, hipStream_t st, const char *what);  // A M-, B K-contiguous
int sg_tile_tn(SgArgs &p, int id, int64_t count, hipStream_t st, const char *what);  // A M-, B N-contiguous

}  // namespace nchip
