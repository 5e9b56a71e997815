// Projection GEMM of the f32 weight format on the matrix cores:
//   C[M,N] = A[M,K] . W[N,K]^T, every product and sum in f32
// (v_mfma_f32_32x32x2_f32: f32 operands, fused f32 accumulation, 64 cycles
// per 32 x 32 x 2 block, 157 TFLOP/s over the chip).
//
// Tiles go global -> LDS directly (16 bytes per lane) through a ring of
// 16-key stages; a tile row is 64 bytes and chunk c of row r sits at slot
// c ^ ((r >> 2) & 3), so a quarter-wave's 16 rows fall on 16 distinct
// 16-byte slots mod 256 bytes. A lane's 16-byte read holds four keys of its
// row: lane half h takes chunk 2 kk + h, and product j of the four pairs key
// j of both halves, so the order of keys within a stage differs from
// memory's but is the same for A and W.
//
// Above 32 rows the matrix-core time of the last round of tiles bounds it, so
// tile and split are chosen for even rounds (fg_splits); up to 32 rows the
// weight stream does. Against the vector-ALU kernel it replaced (64 x 64
// tiles, element loads, no split), 1B-shape projections, us per launch: 301
// rows gate/up 434 -> 208 (97 TFLOP/s), o and down 904 -> 77 on average,
// q/k/v 379 -> 54; 8 rows gate/up ~1700 -> 32 (134 MB of weights, partly
// from the memory-side cache).
#include "common.hpp"
#include "dev.hpp"
#include "kernels_extra.hpp"

namespace esp {

typedef float f32x16f_t __attribute__((ext_vector_type(16)));
typedef float f32x4f_t __attribute__((ext_vector_type(4)));
typedef const void __attribute__((address_space(1))) *gfptr_t;
typedef void __attribute__((address_space(3))) *lfptr_t;

constexpr int FG_BK = 16, FG_ROWB = FG_BK * 4, FG_XCDS = 8;
constexpr int FG_PARTIAL = 16;  // epilogue: raw sums of one k split to ws

// Wave grid WM x (4 / WM); each wave owns RB x CB blocks of 32 x 32 per
// weight matrix. A block's A tile has 32 * WM * RB rows (at least 64 in LDS,
// so every wave issues the same number of loads; the extra ones repeat the
// last row), its weight tile 32 * CB * (4 / WM) rows per matrix.
template <int NB, int WM, int RB, int CB, int STG> struct FgForm {
    static constexpr int WN = 4 / WM;
    static constexpr int BM = 32 * WM * RB, BN = 32 * WN * CB;
    static constexpr int AROWS = BM < 64 ? 64 : BM, BROWS = NB * BN;
    static constexpr int STAGE = (AROWS + BROWS) * FG_ROWB;
    static constexpr size_t LDS = (size_t)STG * STAGE;
    static constexpr int QA = AROWS / 64, QB = BROWS / 64;  // direct loads per wave and stage
    static constexpr int LPS = QA + QB;
    static_assert(QA * 64 == AROWS && QB * 64 == BROWS, "tile rows split over the waves");
    static_assert((STG - 2) * LPS < 64, "waits count up to STG - 2 later stages");
};

constexpr int fg_vm(int n) { return (n & 15) | (7 << 4) | (15 << 8) | ((n >> 4) << 14); }
__device__ __forceinline__ int fg_swz(int r) { return (r >> 2) & 3; }

template <int EPI, int NB, int WM, int RB, int CB, int STG>
__global__ void __launch_bounds__(256) gemm_f32_k(GemmArgs g, float *ws, int k_per_split, int mt, int nt) {
    using F = FgForm<NB, WM, RB, CB, STG>;
    extern __shared__ __attribute__((aligned(16))) char lds_f[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int wm = wave / F::WN, wn = wave % F::WN;
    // XCD-major tile order, row tiles fastest: a weight tile is fetched into
    // one XCD's L2 and serves all its row tiles there
    const int total = mt * nt, per = (total + FG_XCDS - 1) / FG_XCDS;
    const int tile = (blockIdx.x % FG_XCDS) * per + blockIdx.x / FG_XCDS;
    if (tile >= total) return;
    int m0, M, grp;  // M: end of this tile's group
    if (!group_tile(g.grp_offs, g.grp_n, g.M, tile % mt, F::BM, m0, M, grp)) return;
    const int n0 = tile / mt * F::BN, N = g.N, K = g.K;
    const size_t woff = (size_t)grp * g.grp_w_stride;
    const int kbeg = blockIdx.z * k_per_split;
    const int KT = (min(K, kbeg + k_per_split) - kbeg) / FG_BK;

    // this lane's sources: wave-instruction q covers slots q * 64 + lane (16
    // rows of four chunks); rows past M or N repeat the last valid row
    const float *asrc[F::QA], *bsrc[F::QB];
#pragma unroll
    for (int q = 0; q < F::QA; ++q) {
        const int sl = (wave * F::QA + q) * 64 + lane, r = sl >> 2, c = (sl & 3) ^ fg_swz(r);
        asrc[q] = (const float *)g.a + (size_t)min(m0 + r, M - 1) * K + kbeg + c * 4;
    }
#pragma unroll
    for (int q = 0; q < F::QB; ++q) {
        const int sl = (wave * F::QB + q) * 64 + lane, r = sl >> 2, c = (sl & 3) ^ fg_swz(r);
        const int b = r / F::BN, n = min(n0 + r % F::BN, N - 1);
        bsrc[q] = (const float *)(b ? g.w2 : g.w) + woff + (size_t)n * K + kbeg + c * 4;
    }
    auto issue = [&](int kt) {
        char *base = lds_f + (kt % STG) * F::STAGE;
#pragma unroll
        for (int q = 0; q < F::QA; ++q)
            __builtin_amdgcn_global_load_lds((gfptr_t)(asrc[q] + kt * FG_BK),
                                             (lfptr_t)(base + (wave * F::QA + q) * 1024), 16, 0, 0);
#pragma unroll
        for (int q = 0; q < F::QB; ++q)
            __builtin_amdgcn_global_load_lds(
                (gfptr_t)(bsrc[q] + kt * FG_BK),
                (lfptr_t)(base + F::AROWS * FG_ROWB + (wave * F::QB + q) * 1024), 16, 0, 0);
    };

    f32x16f_t acc[NB][RB][CB];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
            for (int j = 0; j < CB; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[b][i][j][e] = 0.f;
#pragma unroll
    for (int st = 0; st < STG - 1; ++st)
        if (st < KT) issue(st);
    for (int kt = 0; kt < KT; ++kt) {
        // stage kt has landed once at most the later stages' loads remain
        if (KT - 1 - kt >= STG - 2) __builtin_amdgcn_s_waitcnt(fg_vm((STG - 2) * F::LPS));
        else __builtin_amdgcn_s_waitcnt(fg_vm(0));
        __builtin_amdgcn_s_barrier();  // every wave's loads landed; stage kt - 1 is free
        if (kt + STG - 1 < KT) issue(kt + STG - 1);
        const char *ab = lds_f + (kt % STG) * F::STAGE, *bb = ab + F::AROWS * FG_ROWB;
        f32x4f_t fa[2][RB], fb[2][NB][CB];
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const int c = 2 * kk + (lane >> 5);
#pragma unroll
            for (int i = 0; i < RB; ++i) {
                const int r = (wm * RB + i) * 32 + (lane & 31);
                fa[kk][i] = *(const f32x4f_t *)(ab + r * FG_ROWB + ((c ^ fg_swz(r)) << 4));
            }
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int j = 0; j < CB; ++j) {
                    const int r = b * F::BN + (wn * CB + j) * 32 + (lane & 31);
                    fb[kk][b][j] = *(const f32x4f_t *)(bb + r * FG_ROWB + ((c ^ fg_swz(r)) << 4));
                }
        }
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int b = 0; b < NB; ++b)
#pragma unroll
                    for (int i = 0; i < RB; ++i)
#pragma unroll
                        for (int j = 0; j < CB; ++j)
                            acc[b][i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[kk][i][e], fb[kk][b][j][e],
                                                                                acc[b][i][j], 0, 0, 0);
    }

    // lane holds column (lane & 31) of each 32 x 32 block, rows
    // (e / 4) * 8 + (lane >> 5) * 4 + e % 4
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j) {
            const int col = n0 + (wn * CB + j) * 32 + (lane & 31);
            if (col >= N) continue;
            const float bias = EPI != FG_PARTIAL && EPI != GEMM_SWIGLU && g.bias ? g.bias[col] : 0.f;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int row = m0 + (wm * RB + i) * 32 + (e >> 2) * 8 + (lane >> 5) * 4 + (e & 3);
                if (row >= M) continue;
                if (EPI == FG_PARTIAL) {
#pragma unroll
                    for (int b = 0; b < NB; ++b)
                        ws[(((size_t)blockIdx.z * NB + b) * g.M + row) * N + col] = acc[b][i][j][e];
                    continue;
                }
                float *c = (float *)g.c + (size_t)row * g.ldc + col;
                if (EPI == GEMM_SWIGLU) {
                    *c = silu(acc[0][i][j][e]) * acc[NB - 1][i][j][e];
                } else {
                    const float v = g.bias ? acc[0][i][j][e] + bias : acc[0][i][j][e];
                    *c = EPI == GEMM_RESIDUAL ? *c + v : v;
                }
            }
        }
}

// K in 16-key stages and 16-byte aligned rows; f32 activations and output
bool gemm_f32_ok(Dt wt, const GemmArgs &a) {
    auto al16 = [](const void *p) { return ((uintptr_t)p & 15) == 0; };
    return wt == DT_F32 && !a.a_lo && !a.c_lo && a.K >= FG_BK && a.K % FG_BK == 0 &&
           a.grp_w_stride % 4 == 0 && al16(a.a) && al16(a.w) && (!a.w2 || al16(a.w2));
}

// Whether `s` k splits, of at least 256 keys each, have room for their sums.
static bool fg_split_fits(const GemmArgs &a, int NB, int s) {
    return s <= 32 && a.K / s >= 256 && a.ws && (size_t)s * NB * a.M * a.N * 4 <= a.ws_bytes;
}

// Split count of a launch above 32 rows and its estimated time (us). `key_us`
// is the time a CU spends on 16 keys of one tile divided by 16 (the
// matrix-core time of the tile's blocks; measured, one tile per CU): `tiles *
// s` tiles of K / s keys run in ceil(tiles s / cus) rounds, so splits pay
// where they even the last round out, against the reduction launch (~4 us)
// and the partial sums written and read once (~4 TB/s).
static int fg_splits(const GemmArgs &a, int NB, long long tiles, double key_us, int cus, double *us) {
    int best = 1;
    double cost = 0;
    for (int s = 1; s == 1 || fg_split_fits(a, NB, s); s *= 2) {
        const double bytes = (double)s * NB * a.M * a.N * 8;
        const double c = (double)((tiles * s + cus - 1) / cus) * a.K / s * key_us +
                         (s > 1 ? 4.0 + bytes * 2.5e-7 : 0.0);
        if (s == 1 || c < cost) best = s, cost = c;
    }
    *us = cost;
    return best;
}

template <int NB, int WM, int RB, int CB, int STG> static long long fg_tiles(const GemmArgs &a) {
    using F = FgForm<NB, WM, RB, CB, STG>;
    return (long long)((a.N + F::BN - 1) / F::BN) * ((a.M + F::BM - 1) / F::BM + (a.grp_offs ? a.grp_n : 0));
}

template <int EPI, int NB, int WM, int RB, int CB, int STG>
static void fg_launch(const GemmArgs &a, int splits, hipStream_t s) {
    using F = FgForm<NB, WM, RB, CB, STG>;
    static bool attr = false;
    if (!attr) {
        ESP_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(gemm_f32_k<EPI, NB, WM, RB, CB, STG>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)F::LDS));
        ESP_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(gemm_f32_k<FG_PARTIAL, NB, WM, RB, CB, STG>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)F::LDS));
        attr = true;
    }
    const int nt = (a.N + F::BN - 1) / F::BN, mt = (a.M + F::BM - 1) / F::BM + (a.grp_offs ? a.grp_n : 0);
    const int blocks = FG_XCDS * ((nt * mt + FG_XCDS - 1) / FG_XCDS);
    if (splits == 1) {
        gemm_f32_k<EPI, NB, WM, RB, CB, STG><<<dim3(blocks), 256, F::LDS, s>>>(a, nullptr, a.K, mt, nt);
        return;
    }
    int kps = (a.K + splits - 1) / splits;
    kps = (kps + FG_BK - 1) / FG_BK * FG_BK;
    gemm_f32_k<FG_PARTIAL, NB, WM, RB, CB, STG><<<dim3(blocks, 1, splits), 256, F::LDS, s>>>(a, a.ws, kps, mt, nt);
    if (a.defer_splits) *a.defer_splits = splits;
    else launch_gemm_reduce((GemmEpi)EPI, a, a.ws, splits, s);
}

template <int EPI> static void fg_dispatch(const GemmArgs &a, hipStream_t s) {
    constexpr int NB = EPI == GEMM_SWIGLU ? 2 : 1;
    static int cus = 0;
    if (!cus) {
        int dev = 0;
        ESP_HIP(hipGetDevice(&dev));
        ESP_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    }
    // 32-row tiles up to 32 rows; above, 64-row tiles of 64 or 128 weight
    // rows, or 128 x 128, whichever the estimate favours (key times measured
    // on MI355X at K 2048: 43, 74 and 138 us per round of one tile per CU)
    constexpr double T64 = 0.0210, T128 = 0.0361, T256 = 0.0674;
    double u0, u1, u2;
    if (a.M <= 32) {
        // the weight stream bounds these: splits until two blocks per CU
        constexpr int ST = NB == 1 ? 6 : 4;
        const long long tiles = fg_tiles<NB, 1, 1, 1, ST>(a);
        int sp = 1;
        while (tiles * sp < 2 * cus && fg_split_fits(a, NB, sp * 2)) sp *= 2;
        fg_launch<EPI, NB, 1, 1, 1, ST>(a, sp, s);
        return;
    }
    const int s1 = fg_splits(a, NB, fg_tiles<NB, 2, 1, 2 / NB, 4>(a), T128, cus, &u1);
    const int s2 = fg_splits(a, NB, fg_tiles<NB, 2, 2, 2 / NB, 4>(a), T256, cus, &u2);
    if constexpr (NB == 1) {
        const int s0 = fg_splits(a, NB, fg_tiles<1, 2, 1, 1, 4>(a), T64, cus, &u0);
        if (u0 < u1 && u0 < u2) {
            fg_launch<EPI, 1, 2, 1, 1, 4>(a, s0, s);
            return;
        }
    }
    if (u1 <= u2) fg_launch<EPI, NB, 2, 1, 2 / NB, 4>(a, s1, s);
    else fg_launch<EPI, NB, 2, 2, 2 / NB, 4>(a, s2, s);
}

void launch_gemm_f32(GemmEpi epi, const GemmArgs &a, hipStream_t s) {
    if (epi == GEMM_STORE) fg_dispatch<GEMM_STORE>(a, s);
    else if (epi == GEMM_RESIDUAL) fg_dispatch<GEMM_RESIDUAL>(a, s);
    else fg_dispatch<GEMM_SWIGLU>(a, s);
}

}  // namespace esp
