// fp32 GEMM on the matrix cores (the reference's gemm_f32 kernel-table entry, kernels.h:36-41, as
// ops_linalg.c:58-330 calls it): hand-written for gfx950 around v_mfma_f32_16x16x4_f32.
//
// C (M x N, row-major, leading dim ldc) = alpha op(A) op(B) + beta C with op(A) M x K and op(B) K x N.
// An operand is stored K-contiguous (A untransposed, B transposed) or M/N-contiguous (A transposed, B
// untransposed), each with its own leading dim; batched forms take per-axis batch strides or pointer
// arrays.  beta = 0 never reads C.
//
// Tiling.  A workgroup owns a BM x BN tile of C and each of its waves a (16 TM) x (16 TN) block of it (or of its
// share of K, gemm_tile.hpp), held as TM x TN 16 x 16 accumulator tiles (4 floats per lane each).  Each operand
// keeps its global layout in LDS, so every operand layout runs without a transposing pass.  The MFMAs take
// the B fragment first and so produce C^T tiles: each lane holds consecutive columns of a row of C, and the
// epilogue writes (and, for beta != 0, reads) C 16 bytes at a time.
//
// k mapping.  One MFMA multiplies a 16 x 4 slice of A by a 4 x 16 slice of B, quarter-wave q (lanes
// 16 q .. 16 q + 15) holding one k.  In each half panel of 16 k, quarter q gives the s-th MFMA (s = 0..3)
// the value at k = 4 q + s, for A and B alike, so a K-contiguous operand feeds four MFMAs from one
// 16-byte LDS read.
//
// Summation order (blocked, like the reference's register blocks summed from zero and added into C,
// kernels_avx2.c:234-247): K is cut into panels of 32 k.  A panel's 32 products of an output element are summed
// from zero, four per MFMA (eight MFMAs), and the panel sum is added into a running total (one fp32 add per 32 k);
// where a tile's waves split K, wave group g of S sums panels g, g + S, ... so and the S totals are added in
// order.  A small panel sum is not rounded against the whole running total, so the error of a K-term dot product
// grows like that of a blocked sum rather than like K sequential additions.  A panel that K ends inside comes
// first.  The kernel, and with it S, is chosen (sg_pick) from M, N, K, the layout, the number of matrices in the call and
// whether the operands' rows are 16-byte aligned: the same call gives the same bits run to run and on any device, but a
// row of a batch, or a matrix of a batched product, may be summed in another order alone than in company, and aligned
// operands in another than unaligned ones.  The order differs from the reference's serial one too, so
// the parity bar is the fp32 error bound of a K-term dot product.
//
// Kernels: k_sgemm_dma (256 x 256 or 128 x 128 tiles, panels loaded straight into LDS) for aligned problems that give every CU
// such tiles, the register-staged tiles of gemm_tile.hpp for the rest.  Blocks are remapped so each XCD
// (blocks b with b % 8 equal) works a contiguous run of tiles, and tiles run in groups of 8 tile-rows so
// neighbouring blocks share panels in L2.
#include "gemm.hpp"

namespace nchip {

constexpr int kSgBK = 16;      // k per stage
constexpr int kSgPanel = 2;    // stages per summation panel (32 k)

// The direct-to-LDS tile: TM x TN 16 x 16 accumulator tiles per wave, WGM x WGN waves
template <int TM_, int TN_, int WGM_, int WGN_>
struct SgCfg {
    static constexpr int TM = TM_, TN = TN_, WGM = WGM_, WGN = WGN_;
    static constexpr int NT = 64 * WGM * WGN;
    static constexpr int BM = 16 * TM * WGM, BN = 16 * TN * WGN;
    // bytes of one stage of an operand panel in LDS (R rows by 16 k, either layout)
    static constexpr int SLAB_A = 64 * BM, SLAB_B = 64 * BN;
    static constexpr int STAGE = SLAB_A + SLAB_B;
};
using SgBig = SgCfg<8, 4, 2, 4>;   // 256 x 256
using SgHalf = SgCfg<2, 4, 4, 2>;  // 128 x 128, 8 waves

// ---- operand panels of the direct-to-LDS kernel ---------------------------------------------------
// One stage of an operand: R rows (M or N) by 16 k in 16-byte chunks.
//   * K-contiguous operand: rows of 64 bytes, logical chunk c of row r at chunk c ^ kc_swz(r), so the 16-byte
//     fragment reads spread over all banks;
//   * M/N-contiguous operand: 16 k-rows of R floats (R >= 64), the chunk of rows 4 c .. 4 c + 3 of k-row k at
//     chunk c ^ mn_swz(k), so the four quarter-waves' fragment reads (k-rows k, k + 4, k + 8, k + 12 of 16
//     consecutive rows) land in different banks.  Either layout is 64 R bytes per stage, with no padding, so
//     a load straight into LDS fills it 1 KiB at a time.
// The chunk permutation of K-contiguous panel row r (an XOR mask on its four 16-byte chunks).
// (r >> 1) & 3 leaves the 16-byte fragment reads of the 16 rows and 4 quarter-waves free of bank
// conflicts (SQ_LDS_BANK_CONFLICT reads 0; (r >> 2) & 3 read a third to a half of the LDS cycles).
__device__ __forceinline__ int kc_swz(int r) { return (r >> 1) & 3; }

// The chunk permutation of M/N-contiguous panel k-row k: quarter-wave q reads k-rows 4 q .. 4 q + 3,
// so XOR-ing bits 2-3 of the chunk index with q puts the four quarters' 16 rows in four disjoint
// groups of 16 banks (the 64 banks of 4 bytes, since a k-row's 4 R bytes are a multiple of 256).
__device__ __forceinline__ int mn_swz(int k) { return ((k >> 2) & 3) << 2; }

// The four values (s = 0..3) of panel row r that quarter-wave q gives the stage's MFMAs.
template <int R, bool KC>
__device__ __forceinline__ f4 fragment(const char *slab, int r, int q) {
    if constexpr (KC) {
        return *(const f4 *)(slab + r * 64 + ((q ^ kc_swz(r)) << 4));
    } else {
        static_assert(R >= 64, "the k-row permutation needs 16 chunks");
        const float *b = (const float *)slab + 4 * q * R + 4 * ((r >> 2) ^ (q << 2)) + (r & 3);
        return f4{b[0], b[R], b[2 * R], b[3 * R]};
    }
}

// A wave's stores of one row block's final totals during the last panel: C row (tile row + fr) of row
// block 0 at byte offset `off` from the tile's C (lane's four columns), row block i `rb` bytes further.
struct RbStore {
    const float *base;  // the batch matrix's C (wave-uniform)
    uint32_t off;       // this lane's first element, row block 0, tile column 0, in bytes
    uint32_t rb;        // 16 rows of C, in bytes
    float alpha;
};

// One 16-byte store at a wave-uniform base plus a 32-bit offset.  The store reads its data registers
// after it issues, and a VALU instruction may overwrite them only two wait states later on this
// family; the compiler inserts those after its own stores, not after inline assembly, so the s_nop
// (three wait states) is part of the statement (without it the next value's fourth component reached
// memory now and then).
__device__ __forceinline__ void store16(const float *base, uint32_t off, f4 v) {
    asm volatile("global_store_dwordx4 %0, %1, %2\n\ts_nop 2" ::"v"(off), "v"(v), "s"(base) : "memory");
}

// The direct-to-LDS kernel has a whole panel in LDS and works it row block by row block, so only one
// row block's TN panel sums are live beside the totals: the B fragments of the panel's stages are read
// once; per row block the A fragments are read, each tile sums its panel's products from zero (stage
// 0's four MFMAs, then stage 1's), and the sums are added into the totals.  st (the tile's last panel,
// stored as it completes, through rs): once the next row block's adds have made a row block's totals
// final, its TN tiles are stored between that row block's MFMAs, so a tile's 256 x 256 output leaves
// spread over its last panel instead of all CUs storing at the same moment after it.
template <class Cfg, bool AK, bool BK>
__device__ __forceinline__ void panel_mfma(const char *c0, const char *c1, f4 (&tot)[Cfg::TM][Cfg::TN], int wm, int wn,
                                           int fr, int fq, const RbStore *rs = nullptr, bool st = false) {
    auto store_rb = [&](int i) {
#pragma unroll
        for (int j = 0; j < Cfg::TN; j++) store16(rs->base, rs->off + (uint32_t)i * rs->rb + (uint32_t)(j * 64), rs->alpha * tot[i][j]);
    };
    static_assert(Cfg::TN == 4, "one previous-row-block add per k step");
    f4 b0[Cfg::TN], b1[Cfg::TN];
#pragma unroll
    for (int j = 0; j < Cfg::TN; j++) {
        b0[j] = fragment<Cfg::BN, BK>(c0 + Cfg::SLAB_A, (wn * Cfg::TN + j) * 16 + fr, fq);
        b1[j] = fragment<Cfg::BN, BK>(c1 + Cfg::SLAB_A, (wn * Cfg::TN + j) * 16 + fr, fq);
    }
    f4 a0 = fragment<Cfg::BM, AK>(c0, wm * Cfg::TM * 16 + fr, fq);
    f4 a1 = fragment<Cfg::BM, AK>(c1, wm * Cfg::TM * 16 + fr, fq);
    // Issue order, pinned by scheduling barriers: per row block, 8 k steps of the TN tiles' independent
    // MFMAs; in each of the first TN steps one tile of the previous row block adds its finished sum
    // into its total (the sum's last MFMA was issued at least TN MFMAs earlier, so the add needs no
    // wait states and issues between MFMAs); the next row block's A fragments are read meanwhile.
    f4 tp[Cfg::TN];
#pragma unroll
    for (int i = 0; i < Cfg::TM; i++) {
        f4 na0 = a0, na1 = a1;
        if (i + 1 < Cfg::TM) {
            const int row = (wm * Cfg::TM + i + 1) * 16 + fr;
            na0 = fragment<Cfg::BM, AK>(c0, row, fq);
            na1 = fragment<Cfg::BM, AK>(c1, row, fq);
        }
        f4 t[Cfg::TN];
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const f4 &a = s < 4 ? a0 : a1;
#pragma unroll
            for (int j = 0; j < Cfg::TN; j++) {
                const f4 &b = s < 4 ? b0[j] : b1[j];
                t[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[s & 3], a[s & 3], s == 0 ? f4{0.f, 0.f, 0.f, 0.f} : t[j],
                                                            0, 0, 0);
            }
            if (i > 0 && s < Cfg::TN) tot[i - 1][s] = tot[i - 1][s] + tp[s];
            if (st && i > 0 && s == Cfg::TN) store_rb(i - 1);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int j = 0; j < Cfg::TN; j++) tp[j] = t[j];
        a0 = na0, a1 = na1;
    }
#pragma unroll
    for (int j = 0; j < Cfg::TN; j++) tot[Cfg::TM - 1][j] = tot[Cfg::TM - 1][j] + tp[j];
    if (st) store_rb(Cfg::TM - 1);
}

// C = alpha acc + beta C (+ bias[n]) over the wave's tiles.  acc[i][j] is the 16 x 16 tile C^T: lane l,
// element v holds row (tile row + l % 16), column (tile column + 4 (l / 16) + v).
template <class Cfg>
__device__ __forceinline__ void write_tiles(const SgArgs &p, const TileAt &at, const f4 (&acc)[Cfg::TM][Cfg::TN],
                                            int wm, int wn, int fr, int fq) {
#pragma unroll
    for (int i = 0; i < Cfg::TM; i++) {
        const int m = at.m0 + (wm * Cfg::TM + i) * 16 + fr;
        if (m >= p.M) continue;
#pragma unroll
        for (int j = 0; j < Cfg::TN; j++) {
            const int n = at.n0 + (wn * Cfg::TN + j) * 16 + 4 * fq;
            if (n < p.N) write4(p, at.C + (int64_t)m * p.ldc, n, acc[i][j]);
        }
    }
}

// ------------------------------------------------------------------------------------------------
// Large aligned problems with K a multiple of 32: the 256 x 256 tile (or 128 x 128), its operand panels loaded straight
// from global memory into LDS (global_load_lds_dwordx4) a summation panel (two stages) ahead through
// four LDS stages, with no staging registers and no LDS write instructions; one barrier per summation
// panel.  A stage of an R-row panel is R / 16 load
// instructions of 1 KiB each: 16 rows of a K-contiguous panel (lane l: row l / 4, the chunk that
// belongs at position l % 4 under the row's permutation) or 256 / R k-rows of a M/N-contiguous one
// (lane l: k-row l / (R / 4), position l % (R / 4), loading the rows the k-row's permutation puts
// there).  The 32 (16) instructions of a stage, half of them for A, are dealt four (two) to a wave.  Rows past
// the matrix are clamped onto its last row (last 4-row chunk), so every load is in bounds.
constexpr int kSgDmaStages = 4;

template <class Cfg>
struct SgDma {
    static constexpr int NW = Cfg::NT / kWave;
    static constexpr int IA = Cfg::BM / 16, IB = Cfg::BN / 16;  // load instructions per stage
    static constexpr int PER = (IA + IB) / NW;                    // per wave
    static_assert((IA + IB) % NW == 0, "the stage's loads deal evenly over the waves");
    static constexpr size_t LDS = kSgDmaStages * (size_t)Cfg::STAGE;
};

// s_waitcnt vmcnt(N) for a compile-time N
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N <= 15, "vmcnt immediate");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

template <class Cfg, bool AK, bool BK>
__global__ __launch_bounds__(Cfg::NT, 1) void k_sgemm_dma(SgArgs p) {
    using D = SgDma<Cfg>;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const TileAt at = locate<Cfg::BM, Cfg::BN>(p);
    const int t = threadIdx.x, lane = t & (kWave - 1), wid = t / kWave;
    const int wm = wid / Cfg::WGN, wn = wid % Cfg::WGN, fr = lane & 15, fq = lane >> 4;

    // this wave's load instructions per stage (each one wave-uniform in its panel)
    const float *src[D::PER];
    int64_t kstep[D::PER];  // elements from one stage to the next
    uint32_t loff[D::PER];
#pragma unroll
    for (int i = 0; i < D::PER; i++) {
        const int j = wid * D::PER + i;
        const bool pb = j >= D::IA;
        const int idx = pb ? j - D::IA : j;
        const bool kc = pb ? BK : AK;
        const float *base = pb ? at.B : at.A;
        const int64_t ld = pb ? p.ldb : p.lda;
        const int rows = pb ? p.N : p.M, r0 = pb ? at.n0 : at.m0;
        const int R = pb ? Cfg::BN : Cfg::BM;
        if (kc) {
            const int prow = 16 * idx + (lane >> 2), c = (lane & 3) ^ kc_swz(prow);
            src[i] = base + (int64_t)min(r0 + prow, rows - 1) * ld + 4 * c;
        } else {
            const int per_row = R / 4;  // chunks per k-row
            const int k = idx * (kWave / per_row) + lane / per_row, c = (lane % per_row) ^ mn_swz(k);
            src[i] = base + (int64_t)k * ld + min(r0 + 4 * c, rows - 4);
        }
        kstep[i] = kc ? kSgBK : kSgBK * ld;
        loff[i] = (uint32_t)(idx * 1024) + (pb ? Cfg::SLAB_A : 0);
    }
    const uint32_t sbase = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)smem;
    auto issue = [&](int kt) {
        const uint32_t st = sbase + (uint32_t)(kt % kSgDmaStages) * Cfg::STAGE;
#pragma unroll
        for (int i = 0; i < D::PER; i++) dma16(src[i] + kt * kstep[i], __builtin_amdgcn_readfirstlane(st + loff[i]));
    };

    f4 tot[Cfg::TM][Cfg::TN];  // running totals
#pragma unroll
    for (int i = 0; i < Cfg::TM; i++)
#pragma unroll
        for (int j = 0; j < Cfg::TN; j++) tot[i][j] = f4{0.f, 0.f, 0.f, 0.f};

    // LDS stage slots 0-1 and 2-3 alternate between panels: panel q + 1 loads while panel q is worked
    // (K is a multiple of 32: whole panels)
    const int npanel = p.K / (kSgBK * kSgPanel);
    // both operands K-contiguous (the layouts with registers to spare for it), a whole tile, C = alpha A B
    // with 16-byte rows and the tile within 4 GiB of the matrix's start: the last panel stores its row
    // blocks as they complete (uniform over the workgroup).  The 64 x [1024,128] x [128,1024] batched
    // product spent a quarter of its time (185 us against 141 without stores) on its output leaving in one
    // burst per tile round: 185 -> 162-166 us.
    const bool stream_st = AK && BK && p.beta == 0.0f && !p.bias && ((uintptr_t)at.C & 15) == 0 && p.ldc % 4 == 0 &&
                           at.m0 + Cfg::BM <= p.M && at.n0 + Cfg::BN <= p.N &&
                           ((int64_t)at.m0 + Cfg::BM) * p.ldc * 4 < ((int64_t)1 << 32);
    RbStore rs;
    rs.base = at.C;
    rs.off = (uint32_t)(((int64_t)(at.m0 + wm * Cfg::TM * 16 + fr) * p.ldc + at.n0 + wn * Cfg::TN * 16 + 4 * fq) * 4);
    rs.rb = (uint32_t)(16 * p.ldc * 4);
    rs.alpha = p.alpha;
    auto issue_panel = [&](int q) {
        issue(kSgPanel * q);
        issue(kSgPanel * q + 1);
    };
    if (npanel > 0) issue_panel(0);
    for (int q = 0; q < npanel; q++) {
        wait_vmcnt<0>();               // this wave's loads of panel q (the only ones in flight)
        __builtin_amdgcn_s_barrier();  // every wave's loads of panel q have landed; panel q - 1 is read
        asm volatile("" ::: "memory");
        if (q + 1 < npanel) issue_panel(q + 1);  // into the slots panel q - 1 used
        const int k0 = kSgPanel * q;
        panel_mfma<Cfg, AK, BK>(smem + (k0 % kSgDmaStages) * Cfg::STAGE,
                                smem + ((k0 + 1) % kSgDmaStages) * Cfg::STAGE, tot, wm, wn, fr, fq, &rs,
                                stream_st && q + 1 == npanel);
    }
    if (!stream_st) write_tiles<Cfg>(p, at, tot, wm, wn, fr, fq);
}

template <class Cfg, bool AK, bool BK>
static int sg_launch_dma(SgArgs &p, int64_t count, hipStream_t st, const char *what) {
    p.tiles_m = (p.M + Cfg::BM - 1) / Cfg::BM;
    p.tiles_n = (p.N + Cfg::BN - 1) / Cfg::BN;
    const int64_t blocks = (int64_t)p.tiles_m * p.tiles_n * count;
    static bool done[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < 64 && !done[dev]) {
        (void)hipFuncSetAttribute((const void *)k_sgemm_dma<Cfg, AK, BK>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)SgDma<Cfg>::LDS);
        done[dev] = true;
    }
    hipLaunchKernelGGL((k_sgemm_dma<Cfg, AK, BK>), dim3((unsigned)blocks), dim3(Cfg::NT), SgDma<Cfg>::LDS, st, p);
    return check_launch(what);
}

// ------------------------------------------------------------------------------------------------
// Which tile.  A problem's time on a tile shape is close to a0 + a1 P + L (s0 + s1 P) microseconds, with P its 32-k
// panels and L the most tiles a CU of a 256-CU part gets: a the latency of a tile that has a CU to itself beyond its
// share of the matrix cores, s what each tile adds.  The coefficients are least-squares fits (4% off on average, 17% at
// most) of this kernel's times at L = 1, 2, 3, 4, 6 and K = 256, 2048, for 0, 1 and 2 operands that are M/N-contiguous;
// the tiles are the ones that a choice by them over sizes from 1 to 8192 takes, and together cost 0.2% over the whole
// family of shapes tried.  Small tiles split K over the waves of a workgroup: a product with few tiles still fills
// the chip (x[8,4096] W[4096,4096]^T: 109 us on the 64 x 64 tile that was the smallest, 14 us on 16 x 16 with 16
// waves).  The choice fixes how K is split, so it depends on the call alone -- sizes, layout, count and alignment -- and is
// planned for kPlanCUs, never for the device.
struct SgTile {
    int bm, bn, lanes;
    float c[3][4];  // a0, a1, s0, s1 by M/N-contiguous operands
};
static const SgTile kSgTiles[] = {  // in the order of sg_tile_run
    {128, 64, 256, {{2.95f, 0.410f, 2.01f, 0.975f}, {3.65f, 0.459f, 1.36f, 1.032f}, {4.24f, 0.316f, 1.11f, 1.267f}}},
    {96, 96, 512, {{3.45f, 0.049f, 2.35f, 1.346f}, {2.94f, 0.089f, 3.19f, 1.353f}, {3.16f, 0.079f, 3.33f, 1.369f}}},
    {96, 64, 256, {{2.85f, 0.367f, 1.28f, 0.710f}, {3.25f, 0.330f, 1.25f, 0.810f}, {4.04f, 0.346f, 1.00f, 0.899f}}},
    {96, 64, 512, {{2.98f, 0.131f, 1.94f, 0.746f}, {2.29f, 0.039f, 2.53f, 0.949f}, {2.43f, 0.048f, 2.73f, 1.015f}}},
    {64, 96, 512, {{3.10f, 0.118f, 1.94f, 0.753f}, {2.11f, 0.026f, 2.88f, 0.981f}, {2.15f, 0.065f, 2.62f, 1.061f}}},
    {64, 64, 256, {{2.42f, 0.242f, 1.26f, 0.486f}, {2.90f, 0.227f, 0.95f, 0.561f}, {2.89f, 0.305f, 1.02f, 0.565f}}},
    {64, 64, 512, {{2.98f, 0.075f, 1.39f, 0.520f}, {2.86f, 0.113f, 1.41f, 0.582f}, {2.83f, 0.142f, 1.35f, 0.601f}}},
    {64, 32, 512, {{1.73f, 0.004f, 1.99f, 0.332f}, {2.00f, -0.002f, 1.82f, 0.386f}, {1.71f, 0.020f, 2.07f, 0.412f}}},
    {32, 64, 512, {{1.71f, 0.010f, 2.12f, 0.313f}, {1.82f, 0.012f, 1.96f, 0.390f}, {1.75f, 0.013f, 2.07f, 0.409f}}},
    {32, 32, 256, {{2.74f, 0.063f, 0.65f, 0.162f}, {2.67f, 0.064f, 0.65f, 0.192f}, {2.75f, 0.062f, 0.71f, 0.195f}}},
    {32, 32, 512, {{2.82f, -0.014f, 1.40f, 0.188f}, {2.19f, -0.004f, 1.73f, 0.218f}, {1.93f, 0.003f, 1.98f, 0.206f}}},
    {32, 16, 512, {{3.55f, -0.028f, 1.08f, 0.114f}, {3.12f, -0.024f, 1.30f, 0.137f}, {3.24f, -0.026f, 1.18f, 0.155f}}},
    {16, 32, 512, {{3.10f, -0.022f, 1.15f, 0.114f}, {3.37f, -0.023f, 1.21f, 0.135f}, {3.06f, -0.025f, 1.35f, 0.156f}}},
    {16, 16, 1024, {{3.61f, -0.031f, 1.37f, 0.063f}, {3.65f, -0.034f, 1.43f, 0.086f}, {3.61f, -0.033f, 1.39f, 0.094f}}},
};
constexpr int kSgTileCount = (int)(sizeof(kSgTiles) / sizeof(kSgTiles[0]));
// The 256 x 256 direct-to-LDS kernel, one tile per CU at a time
static const float kSgDma[4] = {3.0f, 0.0f, 8.3f, 8.05f};
// The 128 x 128 one, two tiles per CU at a time
static const float kSgHalf[3][4] = {{5.0f, 0.0f, 1.7f, 2.13f}, {5.0f, 0.0f, 1.9f, 2.18f}, {5.0f, 0.0f, 2.0f, 2.24f}};

static int64_t tiles_of(int64_t M, int64_t N, int bm, int bn) { return ((M + bm - 1) / bm) * ((N + bn - 1) / bn); }

static float sg_cost(const float *c, int64_t tiles, float panels) {
    const float per_cu = (float)((tiles + kPlanCUs - 1) / kPlanCUs);
    const float t = c[0] + c[1] * panels + per_cu * (c[2] + c[3] * panels);
    return t > 4.5f ? t : 4.5f;  // a launch
}

// The cheapest kernel for M x N x K: a tile's id, kSgDmaId or kSgHalfId for the direct-to-LDS kernels (vec: 16-byte aligned
// rows), or -1 where no launch holds the problem.  *lanes: its work-items.
constexpr int kSgDmaId = kSgTileCount, kSgHalfId = kSgTileCount + 1;

static int sg_pick(int64_t M, int64_t N, int64_t K, bool ak, bool bk, bool vec, int64_t count, int64_t *lanes) {
    // the direct-to-LDS kernel clamps M/N-contiguous chunks onto the last 4 rows: at least 4 rows there, and whole chunks
    const bool dma = vec && K > 0 && K % (kSgBK * kSgPanel) == 0 && (ak || (M >= 4 && M % 4 == 0)) &&
                     (bk || (N >= 4 && N % 4 == 0));
    const float panels = (float)((K + 31) / 32);
    const int mc = !ak + !bk;
    int best = -1;
    float least = 3e38f;
    const auto offer = [&](int id, int bm, int bn, int nt, float margin, const float *c) {
        const int64_t each = tiles_of(M, N, bm, bn);
        if (each > kMaxLanes / nt / count) return;  // more lanes than a launch has
        const float cost = margin * sg_cost(c, each * count, panels);
        if (cost >= least) return;
        best = id;
        least = cost;
        *lanes = each * count * nt;
    };
    // Another tile has to beat the direct-to-LDS kernel by more than the fits are off: predicted 0.8% ahead of it at
    // x[8192,4096] W[4096,4096]^T, the 64 x 64 tile ran 2176 us against its 2085.
    if (dma) offer(kSgDmaId, SgBig::BM, SgBig::BN, SgBig::NT, 0.94f, kSgDma);
    for (int i = 0; i < kSgTileCount; i++) offer(i, kSgTiles[i].bm, kSgTiles[i].bn, kSgTiles[i].lanes, 1.0f, kSgTiles[i].c[mc]);
    // The 128 x 128 direct-to-LDS kernel takes over from the tiles that do not split K: the same sums in the same order.  An
    // operand that is M/N-contiguous costs it next to nothing, the staged tiles 10-15%: A^T B of 8192 x 1024 x 1024 took
    // 168 us on 64 x 64 tiles, 150 on the staged 128 x 128 ones before them, and 152 here (A^T B^T 170, 156 and 149).
    if (dma && (best == 0 || best == 2 || best == 5)) offer(kSgHalfId, SgHalf::BM, SgHalf::BN, SgHalf::NT, 1.0f, kSgHalf[mc]);
    return best;
}

// Runs the problem on the cheapest kernel for it; the direct-to-LDS one takes aligned problems (16-byte rows, K a
// multiple of 32: whole summation panels).
static int sg_run(SgArgs &p, int ta, int tb, int64_t count, hipStream_t st, const char *what) {
    // 16-byte loads need every matrix's rows 16-byte aligned: the matrices behind a pointer array may
    // start anywhere
    bool vec = !p.pa && aligned16(p.A) && aligned16(p.B) && p.lda % 4 == 0 && p.ldb % 4 == 0;
    for (int d = 0; d < p.bat.nb; d++) vec = vec && p.bat.st[0][d] % 4 == 0 && p.bat.st[1][d] % 4 == 0;
    const bool ak = !ta, bk = tb != 0;
    int64_t lanes = 0;
    const int id = sg_pick(p.M, p.N, p.K, ak, bk, vec, count, &lanes);
    if (id < 0)
        return set_error(NC_HIP_ERR_ARG, "%s: %lld products of %d x %d exceed one launch", what, (long long)count, p.M, p.N);
    if (id >= kSgDmaId) {
#define NC_SG_DMA(AK_, BK_)                                                                  \
    if (ak == AK_ && bk == BK_)                                                              \
        return id == kSgDmaId ? sg_launch_dma<SgBig, AK_, BK_>(p, count, st, what) : sg_launch_dma<SgHalf, AK_, BK_>(p, count, st, what);
        NC_SG_DMA(true, true)
        NC_SG_DMA(true, false)
        NC_SG_DMA(false, true)
        NC_SG_DMA(false, false)
#undef NC_SG_DMA
    }
    if (ak) return bk ? sg_tile_nt(p, id, count, st, what) : sg_tile_nn(p, id, count, st, what);
    return bk ? sg_tile_tt(p, id, count, st, what) : sg_tile_tn(p, id, count, st, what);
}

static bool fits_int(int64_t v) { return v >= 0 && v <= INT32_MAX; }

static SgArgs sg_args(int64_t M, int64_t N, int64_t K, float alpha, const float *A, int64_t lda, const float *B,
                      int64_t ldb, float beta, float *C, int64_t ldc) {
    SgArgs p{};
    p.A = A, p.B = B, p.C = C;
    p.lda = lda, p.ldb = ldb, p.ldc = ldc;
    p.M = (int)M, p.N = (int)N, p.K = (int)K;
    p.alpha = alpha, p.beta = beta;
    return p;
}

// ------------------------------------------------------------------------------------------------
// batch axes (ops_linalg.c:89-252): per-operand strides over the output's batch shape (0 = broadcast)
// ------------------------------------------------------------------------------------------------
// drops size-1 batch axes and merges neighbours that step uniformly for all three operands
static void coalesce_batch(SgBatch &bd) {
    int w = 0;
    for (int d = 0; d < bd.nb; d++) {
        if (bd.shape[d] == 1) continue;
        if (w > 0) {
            bool merge = true;
            for (int o = 0; o < 3; o++) merge = merge && bd.st[o][w - 1] == bd.st[o][d] * bd.shape[d];
            if (merge) {
                bd.shape[w - 1] *= bd.shape[d];
                for (int o = 0; o < 3; o++) bd.st[o][w - 1] = bd.st[o][d];
                continue;
            }
        }
        bd.shape[w] = bd.shape[d];
        for (int o = 0; o < 3; o++) bd.st[o][w] = bd.st[o][d];
        w++;
    }
    bd.nb = w;
}

// true when batch index idx is the first (in index order) to write its C block: zero on every axis
// along which C is shared
static bool first_writer(const SgBatch &bd, int64_t idx) {
    for (int d = bd.nb - 1; d >= 0; d--) {
        if (bd.st[2][d] == 0 && idx % bd.shape[d] != 0) return false;
        idx /= bd.shape[d];
    }
    return true;
}

static int64_t host_batch_off(const SgBatch &bd, int o, int64_t idx) {
    int64_t off = 0;
    for (int d = bd.nb - 1; d >= 0; d--) {
        off += (idx % bd.shape[d]) * bd.st[o][d];
        idx /= bd.shape[d];
    }
    return off;
}

}  // namespace nchip

using namespace nchip;

extern "C" NC_HIP_API int nc_hip_gemm_f32_plan(int ta, int tb, int64_t M, int64_t N, int64_t K, int64_t count, int aligned,
                                               int64_t *lanes) {
    int64_t l = 0;
    const bool ok = fits_int(M) && fits_int(N) && fits_int(K) && M > 0 && N > 0 && count > 0;
    const int id = ok ? sg_pick(M, N, K, !ta, tb != 0, aligned != 0, count, &l) : -1;
    if (lanes) *lanes = l;
    return id;
}

extern "C" NC_HIP_API int nc_hip_gemm_f32(int ta, int tb, int64_t M, int64_t N, int64_t K, float alpha, const float *A,
                                          int64_t lda, const float *B, int64_t ldb, float beta, float *C, int64_t ldc,
                                          void *stream) {
    if (!fits_int(M) || !fits_int(N) || !fits_int(K)) return set_error(NC_HIP_ERR_ARG, "nc_hip_gemm_f32: bad size");
    if (M == 0 || N == 0) return NC_HIP_OK;
    if (ldc < N) return set_error(NC_HIP_ERR_ARG, "nc_hip_gemm_f32: ldc %lld < N %lld", (long long)ldc, (long long)N);
    if (K > 0 && (lda < (ta ? M : K) || ldb < (tb ? K : N)))
        return set_error(NC_HIP_ERR_ARG, "nc_hip_gemm_f32: leading dim too small");
    SgArgs p = sg_args(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc);
    return sg_run(p, ta, tb, 1, as_stream(stream), "nc_hip_gemm_f32");
}

extern "C" NC_HIP_API int nc_hip_gemm_f32_bias(int ta, int tb, int64_t M, int64_t N, int64_t K, float alpha,
                                               const float *A, int64_t lda, const float *B, int64_t ldb,
                                               const float *bias, float *C, int64_t ldc, void *stream) {
    if (!fits_int(M) || !fits_int(N) || !fits_int(K)) return set_error(NC_HIP_ERR_ARG, "nc_hip_gemm_f32_bias: bad size");
    if (M == 0 || N == 0) return NC_HIP_OK;
    if (ldc < N) return set_error(NC_HIP_ERR_ARG, "nc_hip_gemm_f32_bias: ldc %lld < N %lld", (long long)ldc, (long long)N);
    if (K > 0 && (lda < (ta ? M : K) || ldb < (tb ? K : N)))
        return set_error(NC_HIP_ERR_ARG, "nc_hip_gemm_f32_bias: leading dim too small");
    SgArgs p = sg_args(M, N, K, alpha, A, lda, B, ldb, 0.0f, C, ldc);
    p.bias = bias;
    return sg_run(p, ta, tb, 1, as_stream(stream), "nc_hip_gemm_f32_bias");
}

extern "C" NC_HIP_API int nc_hip_gemm_f32_batched(int ta, int tb, int64_t M, int64_t N, int64_t K, float alpha,
                                                  const float *const *A, int64_t lda, const float *const *B,
                                                  int64_t ldb, float beta, float *const *C, int64_t ldc, int64_t count,
                                                  void *stream) {
    if (!fits_int(M) || !fits_int(N) || !fits_int(K) || count < 0)
        return set_error(NC_HIP_ERR_ARG, "nc_hip_gemm_f32_batched: bad size");
    if (M == 0 || N == 0 || count == 0) return NC_HIP_OK;
    if (!A || !B || !C) return set_error(NC_HIP_ERR_ARG, "nc_hip_gemm_f32_batched: NULL pointer array");
    if (ldc < N || (K > 0 && (lda < (ta ? M : K) || ldb < (tb ? K : N))))
        return set_error(NC_HIP_ERR_ARG, "nc_hip_gemm_f32_batched: leading dim too small");
    SgArgs p = sg_args(M, N, K, alpha, nullptr, lda, nullptr, ldb, beta, nullptr, ldc);
    p.pa = A, p.pb = B, p.pc = C;
    return sg_run(p, ta, tb, count, as_stream(stream), "nc_hip_gemm_f32_batched");
}

extern "C" NC_HIP_API size_t nc_hip_gemm_f32_bmm_workspace(int64_t count) {
    (void)count;
    return 0;
}

extern "C" NC_HIP_API int nc_hip_gemm_f32_bmm(int ta, int tb, int64_t M, int64_t N, int64_t K, const float *A,
                                              int64_t lda, const float *B, int64_t ldb, float beta, float *C,
                                              int64_t ldc, int nb, const int64_t *bshape, const int64_t *sa,
                                              const int64_t *sb, const int64_t *sc, void *ws, size_t ws_bytes,
                                              void *stream) {
    (void)ws, (void)ws_bytes;
    if (!fits_int(M) || !fits_int(N) || !fits_int(K) || nb < 0 || nb > NC_HIP_MAX_DIMS)
        return set_error(NC_HIP_ERR_ARG, "nc_hip_gemm_f32_bmm: bad sizes");
    SgBatch bd{};
    bd.nb = nb;
    int64_t count = 1;
    for (int d = 0; d < nb; d++) {
        if (bshape[d] < 0) return set_error(NC_HIP_ERR_ARG, "nc_hip_gemm_f32_bmm: negative batch dim");
        bd.shape[d] = bshape[d];
        bd.st[0][d] = sa[d];
        bd.st[1][d] = sb[d];
        bd.st[2][d] = sc[d];
        count *= bshape[d];
    }
    if (M == 0 || N == 0 || count == 0) return NC_HIP_OK;
    if (ldc < N || (K > 0 && (lda < (ta ? M : K) || ldb < (tb ? K : N))))
        return set_error(NC_HIP_ERR_ARG, "nc_hip_gemm_f32_bmm: leading dim too small");
    coalesce_batch(bd);
    bool c_shared = false;  // several batch matrices add into one C block
    for (int d = 0; d < bd.nb; d++) c_shared = c_shared || bd.st[2][d] == 0;
    if (c_shared) {
        // in batch index order, every GEMM after a block's first adding into what the earlier ones wrote
        for (int64_t i = 0; i < count; i++) {
            const int rc = nc_hip_gemm_f32(ta, tb, M, N, K, 1.0f, A + host_batch_off(bd, 0, i), lda,
                                           B + host_batch_off(bd, 1, i), ldb, first_writer(bd, i) ? beta : 1.0f,
                                           C + host_batch_off(bd, 2, i), ldc, stream);
            if (rc != NC_HIP_OK) return rc;
        }
        return NC_HIP_OK;
    }
    SgArgs p = sg_args(M, N, K, 1.0f, A, lda, B, ldb, beta, C, ldc);
    p.bat = bd;
    return sg_run(p, ta, tb, count, as_stream(stream), "nc_hip_gemm_f32_bmm");
}
