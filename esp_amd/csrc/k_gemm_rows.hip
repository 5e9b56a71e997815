// Projection GEMM of few rows over bf16 weights: a few sequences decoding
// together, a short forced span, the rows that a router gives each expert.
//   C[M,N] (f32) = A[M,K] (bf16 hi / lo planes) . W[N,K]^T
// The weights are the stream. A block of four waves owns 128 (gate/up: 64)
// weight columns, one tile of up to 16 * R rows and one k range; the
// activation planes of 512 or 256 keys at a time sit in LDS, so the waves meet
// only when the next chunk is brought in, and each streams the weight rows of
// its own two 16-column units (two column groups, or one of each matrix)
// global -> registers a group of 128 keys ahead: 256 contiguous bytes of each
// row, used at once, in the B-operand layout of v_mfma_f32_16x16x32_bf16.
// Fewer rows leave room for longer chunks (4 rows: 2048 keys), so the waves
// meet less often. Bound by HBM (kernel traces): 8B-shape gate/up (235 MB) at 4
// rows 55 -> 47.1 us (5.0 TB/s; before: 64-row tiles that met at every 32-key
// stage), down 24.8, q/k/v 13.7; experts of 2048 x 7168 that six tokens reach,
// two each: gate/up 77 - 102 us, down 41 - 45 by the number of experts hit
// (before: 128-row tiles, down unsplit; one layer's products 239 -> 163).
#include "common.hpp"
#include "dev.hpp"
#include "kernels_extra.hpp"

namespace esp {

int gemm_skinny_rounds(const GemmArgs &a);  // k_gemm_mfma.hip

typedef __bf16 bf16x8r_t __attribute__((ext_vector_type(8)));
typedef float f32x4r_t __attribute__((ext_vector_type(4)));
typedef const void __attribute__((address_space(1))) *grptr_t;
typedef void __attribute__((address_space(3))) *lrptr_t;

constexpr int GR_ROWB = 64;            // bytes of a 32-key tile row
constexpr int GR_G = 4, GR_GK = 128;   // 32-key blocks and keys of a group
constexpr int GR_PARTIAL = 16;         // epilogue: raw sums of one k split to ws
// keys of a resident chunk: 32 KB of planes (64 KB for 64 rows)
template <int ROWS> constexpr int gr_keys() { return ROWS <= 32 ? 8192 / ROWS : 256; }

// 16-byte chunk c of row r sits at slot c ^ ((r >> 2) & 3): a quarter-wave's
// 16 rows fall on 16 distinct 16-byte slots mod 256 bytes
__device__ __forceinline__ int gr_swz(int r) { return (r >> 2) & 3; }

// ROWS: rows held in LDS, 4, 8, 16, 32 or 64; a product block of 16 rows reads
// four (two) rows again and again where fewer are held.
template <int EPI, int NB, int ROWS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(ROWS <= 16 ? 3 : 2)))
    gemm_rows_k(GemmArgs g, float *ws, int k_per_split) {
    constexpr int R = ROWS <= 16 ? 1 : ROWS / 16;
    constexpr int CK = gr_keys<ROWS>(), NST = CK / 32, GPC = CK / GR_GK;
    constexpr int NC = 2 / NB;        // 16-column groups per wave and matrix
    constexpr int BN = 64 * NC;
    constexpr int AST = ROWS * GR_ROWB, APL = NST * AST;  // a stage of one plane; a plane
    extern __shared__ __attribute__((aligned(16))) char lds_r[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    int m0, mend, grp;
    if (!group_tile(g.grp_offs, g.grp_n, g.M, blockIdx.y, ROWS, m0, mend, grp)) return;
    const int N = g.N, K = g.K, n0 = blockIdx.x * BN, kbeg = blockIdx.z * k_per_split;
    const int kn = min(K, kbeg + k_per_split) - kbeg, NG = kn / GR_GK;
    const size_t woff = (size_t)grp * g.grp_w_stride;

    // unit u: matrix u / NC, columns n0 + 16 (wave NC + u % NC) ..; columns
    // past N repeat the last one
    const uint16_t *wsrc[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int n = min(n0 + 16 * (wave * NC + u % NC) + (lane & 15), N - 1);
        wsrc[u] = (const uint16_t *)(u / NC ? g.w2 : g.w) + woff + (size_t)n * K + kbeg + (lane >> 4) * 8;
    }
    struct Wt {
        bf16x8r_t v[2][GR_G];
    };
    auto issue_w = [&](int gi, Wt &w) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int st = 0; st < GR_G; ++st)
                w.v[u][st] = *(const bf16x8r_t *)(wsrc[u] + (size_t)gi * GR_GK + st * 32);
        __builtin_amdgcn_sched_barrier(0);
    };
    // activation chunk: an instruction brings 16 row pieces of one plane (a
    // piece: 64 bytes, one stage of a row; pieces in order of stage, then
    // row); rows past the tile's end repeat the last, stages past the range
    // are skipped (the range is a multiple of four stages)
    const int prow = lane >> 2;  // piece of the instruction
    constexpr int IPS = ROWS <= 16 ? 1 : ROWS / 16;  // instructions per stage (or one per 16 / ROWS stages)
    static_assert(4 % IPS == 0, "a wave's instructions share their rows");
    const int srow = (wave % IPS * 16 + prow) % ROWS, arow = min(m0 + srow, mend - 1);
    const size_t aoff = (size_t)(g.a_rows ? g.a_rows[arow] : arow) * K + kbeg + (((lane & 3) ^ gr_swz(srow)) * 8);
    auto bring_a = [&](int k0) {
        const int n_st = min(CK, kn - k0) / 32;
        const int per_plane = n_st * ROWS / 16;  // instructions
        for (int q = wave; q < 2 * per_plane; q += 4) {
            const int p = q >= per_plane, qq = q - p * per_plane;
            const int st = ROWS >= 16 ? qq / IPS : qq * (16 / ROWS) + prow / ROWS;
            const uint16_t *src = (const uint16_t *)(p ? g.a_lo : g.a) + aoff + k0 + st * 32;
            __builtin_amdgcn_global_load_lds((grptr_t)src, (lrptr_t)(lds_r + p * APL + qq * 1024), 16, 0, 0);
        }
        __builtin_amdgcn_s_waitcnt(7 << 4 | 15 << 8);  // vmcnt(0)
        __syncthreads();
    };
    f32x4r_t acc[2][R];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < R; ++i) acc[u][i] = f32x4r_t{0.f, 0.f, 0.f, 0.f};

    auto group = [&](Wt &w, Wt &nw, int gi) {
        if (gi % GPC == 0) {
            if (gi) __syncthreads();  // every wave is done with the previous chunk
            bring_a(gi * GR_GK);
        }
        issue_w(min(gi + 1, NG - 1), nw);  // always, so that the wait for w is exact
        const char *base = lds_r + gi % GPC * GR_G * AST;
        bf16x8r_t fa[2][2][R];  // [stage parity][hi / lo]
        auto read_a = [&](int st, bf16x8r_t (&o)[2][R]) {
#pragma unroll
            for (int i = 0; i < R; ++i) {
                const int r = (i * 16 + (lane & 15)) % ROWS, off = r * GR_ROWB + (((lane >> 4) ^ gr_swz(r)) << 4);
                o[0][i] = *(const bf16x8r_t *)(base + st * AST + off);
                o[1][i] = *(const bf16x8r_t *)(base + st * AST + APL + off);
            }
        };
        read_a(0, fa[0]);
#pragma unroll
        for (int st = 0; st < GR_G; ++st) {
            __builtin_amdgcn_sched_barrier(0);
            if (st + 1 < GR_G) read_a(st + 1, fa[(st + 1) & 1]);
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int i = 0; i < R; ++i)
                        acc[u][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[st & 1][p][i], w.v[u][st], acc[u][i], 0, 0, 0);
        }
    };
    Wt w0, w1;
    issue_w(0, w0);
    for (int gi = 0; gi < NG; gi += 2) {
        group(w0, w1, gi);
        if (gi + 1 < NG) group(w1, w0, gi + 1);
    }

    // a 16 x 16 block: column lane & 15, rows 4 (lane >> 4) + e
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int col = n0 + 16 * (wave * NC + c) + (lane & 15);
        if (col >= N) continue;
        const float bias = EPI != GR_PARTIAL && EPI != GEMM_SWIGLU && g.bias ? g.bias[col] : 0.f;
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = m0 + i * 16 + (lane >> 4) * 4 + e;
                if (row >= mend) continue;
                const float v = acc[c][i][e], v2 = acc[NB == 2 ? 1 : c][i][e];
                if (EPI == GR_PARTIAL) {
                    float *o = ws + ((size_t)blockIdx.z * NB * g.M + row) * N + col;
                    *o = v;
                    if (NB == 2) o[(size_t)g.M * N] = v2;
                    continue;
                }
                const size_t ci = (size_t)row * g.ldc + col;
                if (EPI == GEMM_SWIGLU) {
                    const float y = silu(v) * v2;
                    if (g.c_lo) {
                        const uint16_t h = f2bf(y);
                        ((uint16_t *)g.c)[ci] = h;
                        ((uint16_t *)g.c_lo)[ci] = f2bf(y - bf2f(h));
                    } else {
                        ((float *)g.c)[ci] = y;
                    }
                    continue;
                }
                float *o = (float *)g.c + ci;
                const float y = g.bias ? v + bias : v;
                *o = EPI == GEMM_RESIDUAL ? *o + y : y;
            }
    }
}

// Dense launches (2 - 15 rows) that the skinny streamed form, 128 columns and
// one k range a block, does not do better. Where its blocks fill one round of
// the CUs or less it keeps up: a block's whole range is then in flight from the
// start. Past one round the last round is ragged; gate/up below a round gets
// twice the blocks here; and from 96 MB on the resident activations pay. us per
// launch (events around it), skinny -> here, at 2 and 14 rows: o of the 1B
// shape (128 blocks) 7.9 -> 7.9, 8.1 -> 8.9, its gate/up (256, 67 MB) 20.2 ->
// 20.0, 21.4 -> 22.9, down (256, 34 MB) 12.9 -> 13.6, 13.0 -> 15.2; 8B-shape
// q/k/v (384 blocks) 19.0 -> 15.4, 19.4 -> 17.5, gate/up (448) 61.7 -> 53.6,
// 62.8 -> 58.4, down (256, 117 MB) 32.4 -> 29.7, 34.9 -> 33.0; gate/up of 1024
// x 2816 (88) 13.6 -> 11.4, 14.0 -> 12.5; gate/up of 3072 x 8192 (256, 101 MB)
// 33 -> 28, 33.3 -> 31.6.
static bool dense_rows(const GemmArgs &a) {
    const int nb = a.w2 ? 2 : 1, rounds = gemm_skinny_rounds(a);
    return rounds > 0 || (nb == 2 && rounds < 0) || (long long)nb * a.N * a.K * 2 >= 96000000;
}

// Rows per tile; 0: not this form. Dense launches of at most 15 rows (from 16
// on gemm_skinny_k and gemm_lds_k serve; 16 rows would gain here as well, 8B
// shape, two layers, 332 -> 314 us, and are not taken). Grouped launches of up
// to 48 rows per group on average, whose groups' weights are read once per
// tile: past 64 rows a second tile reads them again. Products of a layer of
// eight experts, us, wide tiles -> here, rows spread over the experts / all on
// two of them: 24 per expert 270 -> 248 / 166 -> 133, 48 295 -> 273 / 213 ->
// 209, 56 299 -> 328 / 220 -> 227, 100 344 -> 445 / 314 -> 382.
static int rows_tile(const GemmArgs &a) {
    if (a.K % GR_GK) return 0;
    if (!a.grp_offs) return a.M >= 16 || !dense_rows(a) ? 0 : a.M <= 4 ? 4 : a.M <= 8 ? 8 : 16;
    const int avg = (a.M + a.grp_n - 1) / a.grp_n;
    return a.M <= 4 ? 4 : avg <= 3 ? 8 : avg <= 8 ? 16 : avg <= 20 ? 32 : avg <= 48 ? 64 : 0;
}
bool gemm_rows_ok(const GemmArgs &a) { return rows_tile(a) != 0; }

template <int EPI, int NB, int ROWS> static void rows_launch(const GemmArgs &a, hipStream_t s) {
    constexpr size_t LDSB = (size_t)gr_keys<ROWS>() * ROWS * 4;
    static int cus = 0;
    if (!cus) {
        int dev = 0;
        ESP_HIP(hipGetDevice(&dev));
        for (const void *k : {reinterpret_cast<const void *>(gemm_rows_k<EPI, NB, ROWS>),
                              reinterpret_cast<const void *>(gemm_rows_k<GR_PARTIAL, NB, ROWS>)})
            ESP_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDSB));
        ESP_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    }
    constexpr int BN = 128 / NB;
    const int gx = (a.N + BN - 1) / BN, gy = (a.M + ROWS - 1) / ROWS + (a.grp_offs ? a.grp_n : 0);
    // K splits of at least 256 keys until two blocks per CU; grouped launches
    // until three, the groups' tiles counted as one per group that can have a
    // row. (Three for dense ones cost more in chunk refills and partial sums:
    // 8B-shape down at 4 rows 33.1 -> 30.1 us, 1B-shape 8-row pass -1.5%.)
    const int want = (a.grp_offs ? 3 : 2) * cus;
    const long long tiles = (long long)gx * (a.grp_offs ? std::min(a.grp_n, a.M) : 1);
    int splits = 1;
    while (tiles * splits < want && a.K / (splits * 2) >= 256 && a.ws &&
           (size_t)(splits * 2) * NB * a.M * a.N * 4 <= a.ws_bytes)
        splits *= 2;
    const int kps = ((a.K + splits - 1) / splits + GR_GK - 1) / GR_GK * GR_GK;
    splits = (a.K + kps - 1) / kps;
    if (splits == 1) {
        gemm_rows_k<EPI, NB, ROWS><<<dim3(gx, gy), 256, LDSB, s>>>(a, nullptr, a.K);
        return;
    }
    gemm_rows_k<GR_PARTIAL, NB, ROWS><<<dim3(gx, gy, splits), 256, LDSB, s>>>(a, a.ws, kps);
    if (a.defer_splits) *a.defer_splits = splits;
    else launch_gemm_reduce((GemmEpi)EPI, a, a.ws, splits, s);
}

template <int EPI> static void rows_dispatch(const GemmArgs &a, hipStream_t s) {
    constexpr int NB = EPI == GEMM_SWIGLU ? 2 : 1;
    switch (rows_tile(a)) {
    case 4: rows_launch<EPI, NB, 4>(a, s); break;
    case 8: rows_launch<EPI, NB, 8>(a, s); break;
    case 16: rows_launch<EPI, NB, 16>(a, s); break;
    case 32: rows_launch<EPI, NB, 32>(a, s); break;
    default: rows_launch<EPI, NB, 64>(a, s); break;
    }
}

void launch_gemm_rows(GemmEpi epi, const GemmArgs &a, hipStream_t s) {
    if (epi == GEMM_STORE) rows_dispatch<GEMM_STORE>(a, s);
    else if (epi == GEMM_RESIDUAL) rows_dispatch<GEMM_RESIDUAL>(a, s);
    else rows_dispatch<GEMM_SWIGLU>(a, s);
}

}  // namespace esp
