// Register-staged fp32 GEMM tiles on v_mfma_f32_16x16x4_f32: every problem the 256 x 256 direct-to-LDS
// kernel does not take -- any size, leading dim and 4-byte alignment -- on the tile shape that fills the
// chip best.  (Layouts, the k mapping and the summation order: gemm.hip.)
#pragma once

#include "gemm.hpp"

namespace nchip {

constexpr int kTilePanel = 32;  // k per LDS buffer: one summation panel

// TM x TN 16 x 16 accumulator tiles per wave, WGM x WGN waves per K group, KS K groups per workgroup
template <int TM_, int TN_, int WGM_, int WGN_, int KS_>
struct TileCfg {
    static constexpr int TM = TM_, TN = TN_, WGM = WGM_, WGN = WGN_, KS = KS_;
    static constexpr int NTG = 64 * WGM * WGN, NT = NTG * KS;
    static constexpr int BM = 16 * TM * WGM, BN = 16 * TN * WGN;
};

// Which row of an operand's T tiles (16 T rows of a wave) lane position x of tile j stands for.  K-contiguous: 16 j + x.
// M/N-contiguous: tiles work in groups of 4, 2 or 1 whose rows interleave (group of G: row G x + c is position x of
// its tile c), so that one LDS read of G floats of a k-row serves G tiles.
template <int T, bool KC>
struct TileRows {
    static constexpr int groups = KC ? T : (T + 1) / 2 - (T == 4);
    static constexpr int first(int g) { return KC ? g : 2 * g; }
    static constexpr int size(int g) { return KC ? 1 : T == 4 ? 4 : T - 2 * g >= 2 ? 2 : 1; }
    __device__ __forceinline__ static int row(int j, int x) {
        const int g = KC ? j : T == 4 ? 0 : j / 2, G = size(g);
        return 16 * first(g) + G * x + (j - first(g));
    }
};

// One operand's 32-k panel: R rows (M or N), T tiles of 16 a wave, loaded 16 bytes a lane into registers and then
// stored to LDS.
//   * K-contiguous: unit u is row u / 8, k 4 (u % 8) .. + 3; in LDS two halves of 16 k, rows of 64 bytes, logical
//     chunk c of row r at c ^ ((r >> 1) & 3): a tile's fragment is one 16-byte read, free of bank conflicts;
//   * M/N-contiguous: unit u is k-row u / (R / 4), rows 4 (u % (R / 4)) .. + 3; in LDS k-rows of R floats and a pad
//     that puts the four quarter-waves' reads of G floats (k-rows 4 q + s) in different banks.
template <int R, int T, bool KC, int NT>
struct TilePanel {
    static constexpr int UNITS = 8 * R, UPT = (UNITS + NT - 1) / NT;
    static constexpr bool GUARD = UNITS % NT != 0;
    static constexpr int PITCH = R + (T == 2 || T == 3 ? 8 : 4);
    static constexpr int BYTES = KC ? 128 * R : kTilePanel * PITCH * 4;

    f4 reg[UPT];
    gfloat *src[UPT];
    const float *p;
    int64_t ld;
    int rows, K, r0, t;
    bool edge;  // M/N-contiguous: the tile's last 4-row unit crosses the matrix's end (uniform)

    __device__ __forceinline__ static void pos(int u, int &row, int &k) {
        if constexpr (KC) {
            row = u >> 3, k = (u & 7) * 4;
        } else {
            k = u / (R / 4), row = (u % (R / 4)) * 4;
        }
    }
    __device__ __forceinline__ bool owns(int i) const { return !GUARD || t + i * NT < UNITS; }

    // Rows past the matrix are clamped onto it (what they produce is never stored); a 4-row unit that crosses
    // its end is loaded from rows - 4 and shifted into place before it is stored.
    __device__ __forceinline__ void init(const float *p_, int64_t ld_, int rows_, int K_, int r0_, int t_) {
        p = p_, ld = ld_, rows = rows_, K = K_, r0 = r0_, t = t_;
        edge = !KC && r0 + R > rows && (rows & 3) != 0;
#pragma unroll
        for (int i = 0; i < UPT; i++) {
            int row, k;
            pos(t + i * NT, row, k);
            if constexpr (KC) src[i] = (gfloat *)(p + (int64_t)min(r0 + row, rows - 1) * ld + k);
            else src[i] = (gfloat *)(p + (int64_t)k * ld + max(min(r0 + row, rows - 4), 0));
        }
    }
    // the whole panel at k0
    __device__ __forceinline__ void load(int k0) {
        const int64_t step = KC ? k0 : (int64_t)k0 * ld;
        if (!KC && rows < 4) {  // 1-3 rows: an element at a time
#pragma unroll
            for (int i = 0; i < UPT; i++) {
                if (!owns(i)) continue;
                gfloat *s = src[i] + step;
                reg[i] = f4{s[0], s[rows > 1 ? 1 : 0], s[rows > 2 ? 2 : 0], 0.f};
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < UPT; i++)
            if (owns(i)) reg[i] = *(gf4u *)(src[i] + step);
    }
    // the panel that K ends inside, zeros past it
    __device__ __forceinline__ void load_tail(int k0) {
#pragma unroll
        for (int i = 0; i < UPT; i++) {
            if (!owns(i)) continue;
            int row, k;
            pos(t + i * NT, row, k);
            row += r0, k += k0;
            f4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int kk = KC ? k + j : k, rr = KC ? min(row, rows - 1) : unit_row(row) + j;
                if (kk < K && rr < rows) v[j] = *(gfloat *)(p + (KC ? (int64_t)rr * ld + kk : (int64_t)kk * ld + rr));
            }
            reg[i] = v;
        }
    }
    // the first row an M/N-contiguous unit at `row` is loaded from
    __device__ __forceinline__ int unit_row(int row) const { return max(min(row, rows - 4), 0); }

    __device__ __forceinline__ void store(char *lds) const {
#pragma unroll
        for (int i = 0; i < UPT; i++) {
            if (!owns(i)) continue;
            int row, k;
            pos(t + i * NT, row, k);
            if constexpr (KC) {
                const int c = (k >> 2) & 3;
                *(f4 *)(lds + (k >> 4) * 64 * R + row * 64 + ((c ^ ((row >> 1) & 3)) << 4)) = reg[i];
            } else {
                f4 v = reg[i];
                if (edge) {
                    const int s = r0 + row - unit_row(r0 + row);  // 1 .. 3 where the unit crosses the end
                    if (s == 1) v = f4{v[1], v[2], v[3], 0.f};
                    if (s == 2) v = f4{v[2], v[3], 0.f, 0.f};
                    if (s == 3) v = f4{v[3], 0.f, 0.f, 0.f};
                }
                *(f4 *)(lds + (k * PITCH + row) * 4) = v;
            }
        }
    }
    // the four values (s = 0..3) that quarter-wave q gives half h's MFMAs of the tiles of group g, rows from w0 on
    __device__ __forceinline__ static void read(const char *lds, int h, int g, int w0, int x, int q, f4 (&f)[T]) {
        using Rows = TileRows<T, KC>;
        if constexpr (KC) {
            const int r = w0 + 16 * g + x;
            f[g] = *(const f4 *)(lds + h * 64 * R + r * 64 + ((q ^ ((r >> 1) & 3)) << 4));
        } else {
            const int j = Rows::first(g);
            const float *b = (const float *)lds + (16 * h + 4 * q) * PITCH + w0 + 16 * j + Rows::size(g) * x;
#pragma unroll
            for (int s = 0; s < 4; s++) {
                if (Rows::size(g) == 4) {
                    const f4 v = *(const f4 *)(b + s * PITCH);
#pragma unroll
                    for (int c = 0; c < 4; c++) f[(j + c) % T][s] = v[c];
                } else if (Rows::size(g) == 2) {
                    const f2 v = *(const f2 *)(b + s * PITCH);
                    f[j][s] = v.x, f[(j + 1) % T][s] = v.y;
                } else {
                    f[j][s] = b[s * PITCH];
                }
            }
        }
    }
};

// A workgroup owns a BM x BN tile; its KS groups of waves take the 32-k panels in turn (group g panels g, g + KS,
// ...), each through its own pair of LDS buffers, and meet at one barrier per panel.  A panel's fragments are read
// first; once its first MFMAs are issued the next panel goes from registers to the other buffer and the one after
// it is requested: a load has a whole panel's matrix work to arrive in.  The MFMAs take the B fragment first: the
// tiles are C^T, a lane holding consecutive columns of a row.  With KS > 1 the groups' totals meet in LDS and are
// added in group order.
//
// Bound by the matrix cores and, at one workgroup per CU, by what its waves wait for together (LDS reads after
// the barrier, the barrier itself): x[2048,3072] W[768,3072]^T, 256 tiles of 64 x 96 with 2 K groups, 135 us on the
// 64 x 64 tile of 16-k stages before (384 tiles over 256 CUs, one stage of loads in flight), 105 us with the panel
// loaded and stored between two panels and the reads left to the compiler, 86 us (112 TFLOP/s) in this order timed
// alone and 94 among a training step's launches.  A third LDS buffer with the next panel's fragments read ahead
// timed no better (105 us).  M/N-contiguous operands cost 10-15% more (their reads into LDS are as many, their
// fragments 2 to 4 reads).
template <class Cfg, bool AK, bool BK>
__global__ __launch_bounds__(Cfg::NT) void k_sgemm_tile(SgArgs p) {
    constexpr int TM = Cfg::TM, TN = Cfg::TN, KS = Cfg::KS;
    using PA = TilePanel<Cfg::BM, TM, AK, Cfg::NTG>;
    using PB = TilePanel<Cfg::BN, TN, BK, Cfg::NTG>;
    using RA = TileRows<TM, AK>;
    using RB = TileRows<TN, BK>;
    constexpr int BUF = PA::BYTES + PB::BYTES;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const TileAt at = locate<Cfg::BM, Cfg::BN>(p);
    const int grp = KS == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / Cfg::NTG);
    const int t = KS == 1 ? threadIdx.x : threadIdx.x % Cfg::NTG;
    const int lane = t & (kWave - 1), wid = t / kWave;
    const int wm = wid / Cfg::WGN, wn = wid % Cfg::WGN, fr = lane & 15, fq = lane >> 4;

    PA la;
    PB lb;
    la.init(at.A, p.lda, p.M, p.K, at.m0, t);
    lb.init(at.B, p.ldb, p.N, p.K, at.n0, t);
    f4 tot[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) tot[i][j] = f4{0.f, 0.f, 0.f, 0.f};

    // the panels in working order: the one that K ends inside first, then the whole ones
    const int tail = p.K % kTilePanel != 0, npan = p.K / kTilePanel + tail, iters = (npan + KS - 1) / KS;
    char *const base = smem + grp * 2 * BUF;
    auto load = [&](int q) {
        if (q < npan) {
            la.load((q - tail) * kTilePanel);
            lb.load((q - tail) * kTilePanel);
        }
    };
    auto store = [&](int q, char *buf) {
        if (q < npan) {
            la.store(buf);
            lb.store(buf + PA::BYTES);
        }
    };
    if (tail && grp == 0) {
        la.load_tail(p.K - p.K % kTilePanel);
        lb.load_tail(p.K - p.K % kTilePanel);
    } else {
        load(grp);
    }
    store(grp, base);
    load(grp + KS);
    lds_barrier();
    for (int it = 0; it < iters; it++) {
        const int q = it * KS + grp;
        if (q < npan) {
            const char *ba = base + (it & 1) * BUF, *bb = ba + PA::BYTES;
            const int wa = wm * TM * 16, wb = wn * TN * 16;
            f4 a0[TM], a1[TM], b0[TN], b1[TN];
#pragma unroll
            for (int g = 0; g < RB::groups; g++) {
                PB::read(bb, 0, g, wb, fr, fq, b0);
                if (g == 0) PA::read(ba, 0, 0, wa, fr, fq, a0);
            }
#pragma unroll
            for (int g = 0; g < RB::groups; g++) PB::read(bb, 1, g, wb, fr, fq, b1);
            PA::read(ba, 1, 0, wa, fr, fq, a1);
            // Issue order, pinned by scheduling barriers: per row block, 8 k steps of the TN tiles' independent MFMAs;
            // the next row block's A fragments are read and the previous one's finished sums added to the totals
            // meanwhile.  After the first steps the next panel goes from registers to LDS and the one after it is
            // requested.
            f4 sp[TN];
#pragma unroll
            for (int i = 0; i < TM; i++) {
                f4 s[TN];
#pragma unroll
                for (int g = 1; g < RA::groups; g++)  // the group that starts with the next row block
                    if (RA::first(g) == i + 1) {
                        PA::read(ba, 0, g, wa, fr, fq, a0);
                        PA::read(ba, 1, g, wa, fr, fq, a1);
                    }
#pragma unroll
                for (int k = 0; k < 8; k++) {
#pragma unroll
                    for (int j = 0; j < TN; j++)
                        s[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(k < 4 ? b0[j][k & 3] : b1[j][k & 3], k < 4 ? a0[i][k & 3] : a1[i][k & 3],
                                                                    k == 0 ? f4{0.f, 0.f, 0.f, 0.f} : s[j], 0, 0, 0);
                    if (i > 0 && k < TN) tot[i - 1][k] = tot[i - 1][k] + sp[k];
                    __builtin_amdgcn_sched_barrier(0);
                    if (i == 0 && k == 1) {
                        // the other buffer was last read before the barrier that ended the previous panel
                        store(q + KS, base + ((it + 1) & 1) * BUF);
                        load(q + 2 * KS);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
#pragma unroll
                for (int j = 0; j < TN; j++) sp[j] = s[j];
            }
#pragma unroll
            for (int j = 0; j < TN; j++) tot[TM - 1][j] = tot[TM - 1][j] + sp[j];
        }
        lds_barrier();
    }

    // lane l, element v of tile (i, j): row position l % 16 of A's tile i, row position 4 (l / 16) + v of B's tile j.
    // A group of B's tiles is 4 G consecutive columns of a lane.
    auto put = [&](int i, int g, const f4 *c) {  // c: the group's tiles
        const int m = at.m0 + wm * TM * 16 + RA::row(i, fr), G = RB::size(g);
        const int n = at.n0 + wn * TN * 16 + 16 * RB::first(g) + 4 * G * fq;
        if (m >= p.M) return;
        float *crow = at.C + (int64_t)m * p.ldc;
#pragma unroll
        for (int u = 0; u < G; u++) {
            f4 v;
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = c[(4 * u + e) % G][(4 * u + e) / G];
            if (n + 4 * u < p.N) write4(p, crow, n + 4 * u, v);
        }
    };
    if constexpr (KS > 1) {
        f4 *red = (f4 *)smem;  // [group][tile][thread of the group]
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) red[(grp * TM * TN + i * TN + j) * Cfg::NTG + t] = tot[i][j];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int g = 0; g < RB::groups; g++) {
                if ((i * RB::groups + g) % KS != grp) continue;  // the K groups share out the pieces
                f4 c[4];
#pragma unroll
                for (int w = 0; w < RB::size(g); w++) {
                    const int tile = i * TN + RB::first(g) + w;
                    c[w] = red[tile * Cfg::NTG + t];
#pragma unroll
                    for (int k = 1; k < KS; k++) c[w] = c[w] + red[(k * TM * TN + tile) * Cfg::NTG + t];
                }
                put(i, g, c);
            }
    } else {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int g = 0; g < RB::groups; g++) put(i, g, &tot[i][RB::first(g)]);
    }
}

template <class Cfg, bool AK, bool BK>
static int sg_tile_launch(SgArgs &p, int64_t count, hipStream_t st, const char *what) {
    constexpr int buf = TilePanel<Cfg::BM, Cfg::TM, AK, Cfg::NTG>::BYTES + TilePanel<Cfg::BN, Cfg::TN, BK, Cfg::NTG>::BYTES;
    constexpr int red = Cfg::KS > 1 ? Cfg::KS * Cfg::BM * Cfg::BN * 4 : 0;
    constexpr int lds = 2 * Cfg::KS * buf > red ? 2 * Cfg::KS * buf : red;
    static_assert(lds <= 160 * 1024, "the tile's buffers fit the CU's LDS");
    p.tiles_m = (p.M + Cfg::BM - 1) / Cfg::BM;
    p.tiles_n = (p.N + Cfg::BN - 1) / Cfg::BN;
    const int64_t blocks = (int64_t)p.tiles_m * p.tiles_n * count;
    if constexpr (lds > 64 * 1024) {
        // dynamic LDS above 64 KiB has to be allowed per kernel, once per device
        static bool done[64] = {};
        int dev = 0;
        if (hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < 64 && !done[dev]) {
            (void)hipFuncSetAttribute((const void *)k_sgemm_tile<Cfg, AK, BK>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
            done[dev] = true;
        }
    }
    hipLaunchKernelGGL((k_sgemm_tile<Cfg, AK, BK>), dim3((unsigned)blocks), dim3(Cfg::NT), lds, st, p);
    return check_launch(what);
}

// the tile shapes, in the order of kSgTiles (gemm.hip)
template <bool AK, bool BK>
static int sg_tile_run(SgArgs &p, int id, int64_t count, hipStream_t st, const char *what) {
    switch (id) {
#define NC_SG_TILE(I, ...) \
    case I: return sg_tile_launch<TileCfg<__VA_ARGS__>, AK, BK>(p, count, st, what);
        NC_SG_TILE(0, 4, 2, 2, 2, 1)
        NC_SG_TILE(1, 3, 3, 2, 2, 2)
        NC_SG_TILE(2, 3, 2, 2, 2, 1)
        NC_SG_TILE(3, 3, 2, 2, 2, 2)
        NC_SG_TILE(4, 2, 3, 2, 2, 2)
        NC_SG_TILE(5, 2, 2, 2, 2, 1)
        NC_SG_TILE(6, 2, 2, 2, 2, 2)
        NC_SG_TILE(7, 2, 2, 2, 1, 4)
        NC_SG_TILE(8, 2, 2, 1, 2, 4)
        NC_SG_TILE(9, 2, 2, 1, 1, 4)
        NC_SG_TILE(10, 2, 2, 1, 1, 8)
        NC_SG_TILE(11, 2, 1, 1, 1, 8)
        NC_SG_TILE(12, 1, 2, 1, 1, 8)
        NC_SG_TILE(13, 1, 1, 1, 1, 16)
#undef NC_SG_TILE
    default: return set_error(NC_HIP_ERR_ARG, "%s: unknown tile", what);
    }
}

}  // namespace nchip
