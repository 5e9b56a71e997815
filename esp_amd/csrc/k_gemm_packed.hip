// Projection GEMM of the packed formats (q8 / q4 block-32) on the matrix
// cores, straight from the packed bytes:
//   C[M,N] (f32) = A[M,K] . (q[N,K] * scale[N,K/32])^T
// The integers are exact in bf16, so a 32-key block is multiplied as
//   t = (a_hi + a_lo [+ a_lo2]) . q   (v_mfma_f32_32x32x16_bf16)
// and joins the sum as acc += t * scale: two products per weight instead of
// the three that a weight split into two bf16 halves needs, no dequantized
// copy, and no rounding of q * scale. t overflows from |a| = 8e34 on, where
// a . (q * scale) need not: a block whose sums are not all finite computes its
// outputs again with the scale inside (pk_plain).
// Activations arrive as P bf16 planes: hi / lo, as for bf16 weights, or three
// (the output head, whose activations stay whole).
//
// q4 nibbles are widened in the high half of a byte, as 16 q (exact in bf16
// too), and the block's scale is divided by 16.
#include "common.hpp"
#include "dev.hpp"
#include "kernels_extra.hpp"

namespace esp {

typedef __bf16 bf16x8p_t __attribute__((ext_vector_type(8)));
typedef float f32x16p_t __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4p_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2p_t __attribute__((ext_vector_type(2)));
typedef float f32x4p_t __attribute__((ext_vector_type(4)));
typedef const void __attribute__((address_space(1))) *gpptr_t;
typedef void __attribute__((address_space(3))) *lpptr_t;

constexpr int PK_ROWB = 64;  // bytes of a 32-key tile row of bf16
constexpr int PK_XCDS = 8;
constexpr int PK_PARTIAL = 16;  // epilogue: raw sums of one k split to ws

// slot of 16-byte chunk c of tile row r: c ^ ((r >> 2) & 3), so a quarter-
// wave's 16 rows fall on 16 distinct 16-byte slots mod 256 bytes
__device__ __forceinline__ int pk_swz(int r) { return (r >> 2) & 3; }
constexpr int pk_vm(int n) { return (n & 15) | (7 << 4) | (15 << 8) | ((n >> 4) << 14); }

// sixteen keys of one weight row as loaded: 16 bytes (q8) or 8 bytes (q4)
__device__ __forceinline__ const uint16_t *pk_plane(const GemmArgs &g, int p) {
    return (const uint16_t *)(p == 0 ? g.a : p == 1 ? g.a_lo : g.a_lo2);
}

template <bool Q4> struct PkLoad { typedef u32x4p_t T; };
template <> struct PkLoad<true> { typedef u32x2p_t T; };

// eight keys to bf16: q8 from two dwords, q4 (as 16 q) from one
__device__ __forceinline__ bf16x8p_t pk_bytes(uint32_t even, uint32_t odd, bool interleave) {
    bf16x8p_t r;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float e = (float)(int8_t)(even >> (8 * j)), o = (float)(int8_t)(odd >> (8 * j));
        r[interleave ? 2 * j : j] = (__bf16)e;
        r[interleave ? 2 * j + 1 : 4 + j] = (__bf16)o;
    }
    return r;
}
__device__ __forceinline__ void pk_widen(const u32x4p_t &w, bf16x8p_t (&o)[2]) {
    o[0] = pk_bytes(w.x, w.y, false);
    o[1] = pk_bytes(w.z, w.w, false);
}
__device__ __forceinline__ void pk_widen(const u32x2p_t &w, bf16x8p_t (&o)[2]) {
    o[0] = pk_bytes((w.x << 4) & 0xF0F0F0F0u, w.x & 0xF0F0F0F0u, true);
    o[1] = pk_bytes((w.y << 4) & 0xF0F0F0F0u, w.y & 0xF0F0F0F0u, true);
}

template <int EPI, int NB>
__device__ __forceinline__ void pk_store(const GemmArgs &g, float *ws, int z, int row, int col,
                                         const float (&v)[NB], float bias) {
    if (EPI == PK_PARTIAL) {
#pragma unroll
        for (int b = 0; b < NB; ++b) ws[(((size_t)z * NB + b) * g.M + row) * g.N + col] = v[b];
        return;
    }
    const size_t ci = (size_t)row * g.ldc + col;
    if (EPI == GEMM_SWIGLU) {
        const float y = silu(v[0]) * v[NB - 1];
        if (g.c_lo) {
            const uint16_t h = f2bf(y);
            ((uint16_t *)g.c)[ci] = h;
            ((uint16_t *)g.c_lo)[ci] = f2bf(y - bf2f(h));
        } else {
            ((float *)g.c)[ci] = y;
        }
        return;
    }
    float *c = (float *)g.c + ci;
    const float y = g.bias ? v[0] + bias : v[0];
    *c = EPI == GEMM_RESIDUAL ? *c + y : y;
}

// Whether a launch can meet activations above 8e34: o_proj and down_proj (one
// matrix, two planes) can; what reads a norm's output stays below sqrt(H) times
// an f16 weight.
template <int EPI, int NB, int P> constexpr bool pk_may_overflow() {
    return NB == 1 && P == 2 && (EPI == GEMM_RESIDUAL || EPI == PK_PARTIAL);
}
__device__ __forceinline__ bool pk_finite(float x) { return fabsf(x) < INFINITY; }

// The block's outputs (rows [m0, m0 + rows), columns [n0, n0 + cols), keys [k0,
// k0 + kn)) as plain sums of a * (q * scale), for a block of 256 threads. An
// output that is not finite here either ends its own sum.
template <int EPI, bool Q4>
__device__ void pk_plain(const GemmArgs &g, float *ws, int z, int m0, int rows, int n0, int cols, int k0, int kn) {
    rows = min(rows, g.M - m0);
    cols = min(cols, g.N - n0);
    for (int i = threadIdx.x; i < rows * cols; i += 256) {
        const int row = m0 + i / cols, col = n0 + i % cols;
        const uint16_t *ah = (const uint16_t *)g.a + (size_t)row * g.K, *al = (const uint16_t *)g.a_lo + (size_t)row * g.K;
        float acc = 0.f;
        for (int k = k0; k < k0 + kn && pk_finite(acc); ++k) {
            const size_t e = (size_t)col * g.K + k;
            const int q = Q4 ? (int)((unsigned)((const uint8_t *)g.w)[e / 2] << (28 - 4 * (int)(e & 1))) >> 28
                             : ((const int8_t *)g.w)[e];
            acc = fmaf(bf2f(ah[k]) + bf2f(al[k]), (float)q * g.w_scale[e / 32], acc);
        }
        const float v[1] = {acc};
        pk_store<EPI, 1>(g, ws, z, row, col, v, EPI != PK_PARTIAL && g.bias ? g.bias[col] : 0.f);
    }
}

// ---------------------------------------------------------------------------
// Skinny form, M <= 16 * R rows: the packed weights are the stream. A block
// of four waves owns 128 (gate/up: 64) weight columns and one k range. The
// activation planes of 512 or 256 keys at a time sit in LDS, so the waves meet
// only when the next chunk is brought in, and each streams the packed bytes
// and scales of its own two 16-column units (two column groups, or one of
// each matrix) global -> registers one group ahead.
//
// A group is four 32-key blocks of each weight row, 128 (q4: 64) contiguous
// bytes, a block per 16-lane row of the wave, so a line is fetched once and
// used at once; loading 32 (16) bytes of each row per stage instead fetched
// each line four (eight) times through the L1 and ran at the L2's rate. The
// lane rows then transpose what they loaded (v_permlane32_swap, 16_swap): row
// q ends with keys 8 q .. 8 q + 8 of every block, the B operand of
// v_mfma_f32_16x16x32_bf16. (q4 groups of a whole line need 128 registers of
// values and scales in flight and spilled.) 8B-shape gate/up at 9 rows: q8
// 61 -> 37 us (3.6 TB/s), q4 52 -> 28 us; dequantizing and multiplying the
// bf16 halves took 250. Bound by the vector ALU's share of each block (widen,
// scale, sum) and the latency of its chain.
// Activation keys resident in LDS. Three planes of them (the output head) take
// half the keys, so that a CU keeps as many blocks: a 128256 x 4096 head, us
// with as many keys as two planes -> with half: q8 9 rows 205 -> 171, 64 rows
// 593 -> 381, q4 9 rows 144 -> 120 (two planes: 161, 270, 107).
template <int R, int P> constexpr int ps_keys() { return P == 3 ? (R == 1 ? 256 : 128) : R == 1 ? 512 : 256; }

constexpr int PS_G = 4, PS_GK = 32 * PS_G;  // blocks and keys of a group

__device__ __forceinline__ void pk_swap32(uint32_t &a, uint32_t &b) {
    const u32x2p_t r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r.x;
    b = r.y;
}
__device__ __forceinline__ void pk_swap16(uint32_t &a, uint32_t &b) {
    const u32x2p_t r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r.x;
    b = r.y;
}
// x[j] of 16-lane row q -> x[q] of row j
__device__ __forceinline__ void pk_transpose(uint32_t &x0, uint32_t &x1, uint32_t &x2, uint32_t &x3) {
    pk_swap32(x0, x2);
    pk_swap32(x1, x3);
    pk_swap16(x0, x1);
    pk_swap16(x2, x3);
}

template <int EPI, int NB, int R, bool Q4, int P>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(R == 1 ? 4 : 2)))
    gemm_pk_skinny_k(GemmArgs g, float *ws, int k_per_split) {
    constexpr int G = PS_G, KEYS = PS_GK, NQ = Q4 ? 1 : 2, CK = ps_keys<R, P>(), GPC = CK / KEYS;
    constexpr int NC = 2 / NB;                       // 16-column groups per wave and matrix
    constexpr int BN = 64 * NC;                      // columns per block
    constexpr int ROWS = 16 * R, APL = ROWS * PK_ROWB, AST = P * APL;  // a stage: its planes
    extern __shared__ __attribute__((aligned(16))) char lds_p[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int M = g.M, N = g.N, K = g.K;
    const int n0 = blockIdx.x * BN, kbeg = blockIdx.z * k_per_split;
    const int kn = min(K, kbeg + k_per_split) - kbeg, NG = kn / KEYS;

    // unit u: matrix u / NC, columns n0 + 16 (wave NC + u % NC) ..; columns
    // past N repeat the last one
    const char *wsrc[2];
    const float *ssrc[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int b = u / NC, n = min(n0 + 16 * (wave * NC + u % NC) + (lane & 15), N - 1);
        const size_t e = (size_t)n * K + kbeg;
        wsrc[u] = (const char *)(b ? g.w2 : g.w) + (Q4 ? e / 2 : e) + (lane >> 4) * 16 * NQ;
        ssrc[u] = (b ? g.w2_scale : g.w_scale) + (size_t)n * (K / 32) + kbeg / 32;
    }
    struct Wt {
        u32x4p_t v[2][NQ];
        f32x4p_t s[2];
    };
    auto issue_w = [&](int gi, Wt &w) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
#pragma unroll
            for (int q = 0; q < NQ; ++q) w.v[u][q] = *(const u32x4p_t *)(wsrc[u] + (size_t)gi * 64 * NQ + q * 16);
            w.s[u] = *(const f32x4p_t *)(ssrc[u] + gi * G);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // activation chunk: instruction q brings 16 rows of one stage and plane
    // (slot sl: row sl / 4, 16-byte chunk (sl % 4) ^ swz); rows past M repeat
    // the last, stages past the range are skipped
    auto bring_a = [&](int k0) {
        const int n_ins = min(CK, kn - k0) / 32 * P * R;
        const int r16 = lane >> 2, kc = (lane & 3) ^ pk_swz(r16);
        for (int q = wave; q < n_ins; q += 4) {
            const int st = q / (P * R), p = q / R % P, rb = q % R;
            const uint16_t *src = pk_plane(g, p) + (size_t)min(rb * 16 + r16, M - 1) * K +
                                  kbeg + k0 + st * 32 + kc * 8;
            __builtin_amdgcn_global_load_lds((gpptr_t)src, (lpptr_t)(lds_p + q * 1024), 16, 0, 0);
        }
        __builtin_amdgcn_s_waitcnt(pk_vm(0));
        __syncthreads();
    };
    f32x4p_t acc[2][R];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < R; ++i) acc[u][i] = (f32x4p_t)(0.f);

    auto group = [&](Wt &w, Wt &nw, int gi) {
        if (gi % GPC == 0) {
            if (gi) __syncthreads();  // every wave is done with the previous chunk
            bring_a(gi * KEYS);
        }
        issue_w(min(gi + 1, NG - 1), nw);  // always, so that the wait for w is exact
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            if constexpr (Q4) {  // block q of row q -> dword s: block s
                u32x4p_t &v = w.v[u][0];
                uint32_t a0 = v.x, a1 = v.y, a2 = v.z, a3 = v.w;
                pk_transpose(a0, a1, a2, a3);
                v = u32x4p_t{a0, a1, a2, a3};
            } else {  // dword pairs (0,1) (2,3) of v0, then of v1: block q of row q
                u32x4p_t &v0 = w.v[u][0], &v1 = w.v[u][1];
                uint32_t a0 = v0.x, a1 = v0.z, a2 = v1.x, a3 = v1.z;
                uint32_t b0 = v0.y, b1 = v0.w, b2 = v1.y, b3 = v1.w;
                pk_transpose(a0, a1, a2, a3);
                pk_transpose(b0, b1, b2, b3);
                v0 = u32x4p_t{a0, b0, a1, b1};  // blocks 0, 1
                v1 = u32x4p_t{a2, b2, a3, b3};  // blocks 2, 3
            }
        }
        const char *base = lds_p + gi % GPC * G * AST;
        bf16x8p_t fa[2][P][R];  // [stage parity][plane]
        auto read_a = [&](int st, bf16x8p_t (&o)[P][R]) {
#pragma unroll
            for (int i = 0; i < R; ++i) {
                const int r = lane & 15, off = i * 1024 + r * PK_ROWB + (((lane >> 4) ^ pk_swz(r)) << 4);
#pragma unroll
                for (int p = 0; p < P; ++p) o[p][i] = *(const bf16x8p_t *)(base + st * AST + p * APL + off);
            }
        };
        read_a(0, fa[0]);
#pragma unroll
        for (int st = 0; st < G; ++st) {
            // one stage at a time, the next one's rows already on their way:
            // left alone the compiler widens the whole group first and spills
            __builtin_amdgcn_sched_barrier(0);
            if (st + 1 < G) read_a(st + 1, fa[(st + 1) & 1]);
            const bf16x8p_t (&fs)[P][R] = fa[st & 1];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                bf16x8p_t f;
                if constexpr (Q4) {
                    const uint32_t x = w.v[u][0][st];
                    f = pk_bytes((x << 4) & 0xF0F0F0F0u, x & 0xF0F0F0F0u, true);
                } else {
                    const u32x4p_t &v = w.v[u][st >> 1];
                    f = st & 1 ? pk_bytes(v.z, v.w, false) : pk_bytes(v.x, v.y, false);
                }
                const float s = Q4 ? w.s[u][st] * 0.0625f : w.s[u][st];
#pragma unroll
                for (int i = 0; i < R; ++i) {
                    f32x4p_t t = (f32x4p_t)(0.f);
#pragma unroll
                    for (int p = 0; p < P; ++p) t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fs[p][i], f, t, 0, 0, 0);
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[u][i][e] = fmaf(t[e], s, acc[u][i][e]);
                }
            }
        }
    };
    Wt w0, w1;
    issue_w(0, w0);
    for (int gi = 0; gi < NG; gi += 2) {
        group(w0, w1, gi);
        if (gi + 1 < NG) group(w1, w0, gi + 1);
    }
    if constexpr (pk_may_overflow<EPI, NB, P>()) {
        bool bad = false;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int i = 0; i < R; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) bad |= !pk_finite(acc[u][i][e]);
        if (__syncthreads_or(bad)) {
            pk_plain<EPI, Q4>(g, ws, blockIdx.z, 0, M, n0, BN, kbeg, kn);
            return;
        }
    }

    // a 16 x 16 block: column lane & 15, rows 4 (lane >> 4) + e
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int col = n0 + 16 * (wave * NC + c) + (lane & 15);
        if (col >= N) continue;
        const float bias = EPI != PK_PARTIAL && EPI != GEMM_SWIGLU && g.bias ? g.bias[col] : 0.f;
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = i * 16 + (lane >> 4) * 4 + e;
                if (row >= M) continue;
                float v[NB];
#pragma unroll
                for (int b = 0; b < NB; ++b) v[b] = acc[b * NC + c][i][e];
                pk_store<EPI, NB>(g, ws, blockIdx.z, row, col, v, bias);
            }
    }
}

// ---------------------------------------------------------------------------
// Tiled form: 128 rows x 256 weight rows (NB matrices of 256 / NB columns),
// four waves of 64 rows x 128 weight rows, two blocks per CU. Per 32-key
// stage (two LDS buffers) the activation planes go global -> LDS directly;
// the packed bytes of stage kt + 2 are loaded to registers while stage kt is
// multiplied, and those of kt + 1 are widened to bf16 into LDS at its start,
// so each weight is widened once per block. Scales ride along (one per weight
// row and stage). 8B shape, 2048 rows: gate/up 1046 us (920 TFLOP/s issued,
// as the bf16 streamed form), where three products and a dequantized copy
// took 1500; 1100 rows, four projections of a layer: 2.25 -> 1.15 ms.
constexpr int PT_BM = 128, PT_BR = 256;
constexpr int PT_A = PT_BM * PK_ROWB;  // one plane of a stage
template <int P> constexpr int pt_stage() { return P * PT_A + PT_BR * PK_ROWB + PT_BR * 4; }
template <int P> constexpr size_t pt_lds() { return 2 * pt_stage<P>(); }

// three planes: one block per CU (82 KB of LDS; a 128256 x 4096 q8 head of 100
// rows 361 -> 540 us against two planes, 3375 dequantized in f32)
template <int EPI, int NB, bool Q4, int P>
__global__ void __launch_bounds__(256, P == 2 ? 2 : 1) gemm_pk_tile_k(GemmArgs g, float *ws, int k_per_split, int mt, int nt) {
    typedef typename PkLoad<Q4>::T W;
    constexpr int BN = PT_BR / NB, NJ = BN / 64;  // 32-column blocks per wave and matrix
    constexpr int PT_STAGE = pt_stage<P>();
    extern __shared__ __attribute__((aligned(16))) char lds_p[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int wm = wave >> 1, wn = wave & 1;
    // XCD-major tile ranges in bands of g.band column tiles, row tiles within
    // a column group, as the bf16 streamed form
    const int total = mt * nt, per = (total + PK_XCDS - 1) / PK_XCDS;
    const int tile = (blockIdx.x % PK_XCDS) * per + blockIdx.x / PK_XCDS;
    if (tile >= total) return;
    const int bw = min(g.band, nt), bsz = mt * bw, bnd = tile / bsz, idx = tile - bnd * bsz;
    const int cw = min(bw, nt - bnd * bw), m0 = idx / cw * PT_BM, n0 = (bnd * bw + idx % cw) * BN;
    const int M = g.M, N = g.N, K = g.K;
    const int kbeg = blockIdx.z * k_per_split;
    const int KT = (min(K, kbeg + k_per_split) - kbeg) / 32;
    if (KT <= 0) return;

    // activation rows: 8 instructions of 16 rows per plane, two per wave;
    // rows past M repeat the last
    const uint16_t *asrc[P][2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int sl = (wave * 2 + q) * 64 + lane, r = sl >> 2, kc = (sl & 3) ^ pk_swz(r);
        const size_t off = (size_t)min(m0 + r, M - 1) * K + kbeg + kc * 8;
#pragma unroll
        for (int p = 0; p < P; ++p) asrc[p][q] = pk_plane(g, p) + off;
    }
    // packed values: thread = (weight row tid / 2 + 128 i, keys 16 (tid & 1)
    // .. + 16); scale: weight row tid
    const int half = tid & 1;
    const char *wsrc[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int r = (tid >> 1) + 128 * i, n = min(n0 + r % BN, N - 1);
        const size_t e = (size_t)n * K + kbeg + half * 16;
        wsrc[i] = (const char *)(r / BN ? g.w2 : g.w) + (Q4 ? e / 2 : e);
    }
    const float *ssrc = (tid / BN ? g.w2_scale : g.w_scale) + (size_t)min(n0 + tid % BN, N - 1) * (K / 32) + kbeg / 32;

    W wr[2];
    float sr;
    auto issue_a = [&](int kt) {
        char *base = lds_p + (kt & 1) * PT_STAGE;
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
            for (int q = 0; q < 2; ++q)
                __builtin_amdgcn_global_load_lds((gpptr_t)(asrc[p][q] + kt * 32),
                                                 (lpptr_t)(base + p * PT_A + (wave * 2 + q) * 1024), 16, 0, 0);
    };
    auto issue_w = [&](int kt) {
#pragma unroll
        for (int i = 0; i < 2; ++i) wr[i] = *(const W *)(wsrc[i] + kt * (Q4 ? 16 : 32));
        sr = ssrc[kt];
    };
    auto put_w = [&](int kt) {  // registers -> LDS, widened
        char *bb = lds_p + (kt & 1) * PT_STAGE + P * PT_A;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int r = (tid >> 1) + 128 * i;
            bf16x8p_t f[2];
            pk_widen(wr[i], f);
#pragma unroll
            for (int c = 0; c < 2; ++c)
                *(bf16x8p_t *)(bb + r * PK_ROWB + (((2 * half + c) ^ pk_swz(r)) << 4)) = f[c];
        }
        *(float *)(bb + PT_BR * PK_ROWB + tid * 4) = Q4 ? sr * 0.0625f : sr;
    };

    f32x16p_t acc[NB][2][NJ];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[b][i][j] = (f32x16p_t)(0.f);

    issue_w(0);
    put_w(0);
    issue_a(0);
    __builtin_amdgcn_sched_barrier(0);
    if (KT > 1) issue_w(1);
    for (int kt = 0; kt < KT; ++kt) {
        // stage kt's planes have landed (only the three loads of kt + 1's
        // packed bytes were issued after them) and its weights are in LDS
        if (kt + 1 < KT) __builtin_amdgcn_s_waitcnt(pk_vm(3) & ~(15 << 8));
        else __builtin_amdgcn_s_waitcnt(pk_vm(0) & ~(15 << 8));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        if (kt + 1 < KT) {
            put_w(kt + 1);
            __builtin_amdgcn_sched_barrier(0);
            issue_a(kt + 1);
            __builtin_amdgcn_sched_barrier(0);
            if (kt + 2 < KT) issue_w(kt + 2);
        }
        __builtin_amdgcn_sched_barrier(0);
        const char *ab = lds_p + (kt & 1) * PT_STAGE, *bb = ab + P * PT_A;
        const float *sc = (const float *)(bb + PT_BR * PK_ROWB);
        bf16x8p_t fs[P][2][2];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int c = 2 * ks + (lane >> 5), r = wm * 64 + i * 32 + (lane & 31);
                const int off = r * PK_ROWB + ((c ^ pk_swz(r)) << 4);
#pragma unroll
                for (int p = 0; p < P; ++p) fs[p][ks][i] = *(const bf16x8p_t *)(ab + p * PT_A + off);
            }
        // Units of one 32 x 32 block: a unit's 2 P products are issued with
        // the previous unit's sixteen sums between them, so the vector ALU
        // works in the shadow of the matrix core, and two product blocks are
        // live at a time.
        constexpr int CB = NB * NJ;
        bf16x8p_t f[2][2];
        float sv[2];
        f32x16p_t t[2];
        auto read_w = [&](int jb, bf16x8p_t (&o)[2], float &sc_o) {
            const int r = jb / NJ * BN + wn * (BN / 2) + jb % NJ * 32 + (lane & 31);
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
                o[ks] = *(const bf16x8p_t *)(bb + r * PK_ROWB + (((2 * ks + (lane >> 5)) ^ pk_swz(r)) << 4));
            sc_o = sc[r];
        };
        auto sums = [&](int u) {
            const int jb = u >> 1, i = u & 1;
#pragma unroll
            for (int e = 0; e < 16; ++e)
                acc[jb / NJ][i][jb % NJ][e] = fmaf(t[u & 1][e], sv[jb & 1], acc[jb / NJ][i][jb % NJ][e]);
        };
        read_w(0, f[0], sv[0]);
#pragma unroll
        for (int u = 0; u < 2 * CB; ++u) {
            const int jb = u >> 1, i = u & 1;
            __builtin_amdgcn_sched_barrier(0);
            f32x16p_t x = (f32x16p_t)(0.f);
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int p = 0; p < P; ++p)
                    x = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fs[p][ks][i], f[jb & 1][ks], x, 0, 0, 0);
            if (u > 0) sums(u - 1);
            t[u & 1] = x;
            if (i == 1 && jb + 1 < CB) read_w(jb + 1, f[(jb + 1) & 1], sv[(jb + 1) & 1]);
            if (u > 0) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
                }
            }
        }
        sums(2 * CB - 1);
    }
    if constexpr (pk_may_overflow<EPI, NB, P>()) {
        bool bad = false;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) bad |= !pk_finite(acc[0][i][j][e]);
        if (__syncthreads_or(bad)) {
            pk_plain<EPI, Q4>(g, ws, blockIdx.z, m0, PT_BM, n0, BN, kbeg, KT * 32);
            return;
        }
    }

#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int col = n0 + wn * (BN / 2) + j * 32 + (lane & 31);
            if (col >= N) continue;
            const float bias = EPI != PK_PARTIAL && EPI != GEMM_SWIGLU && g.bias ? g.bias[col] : 0.f;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int row = m0 + wm * 64 + i * 32 + (e >> 2) * 8 + (lane >> 5) * 4 + (e & 3);
                if (row >= M) continue;
                float v[NB];
#pragma unroll
                for (int b = 0; b < NB; ++b) v[b] = acc[b][i][j][e];
                pk_store<EPI, NB>(g, ws, blockIdx.z, row, col, v, bias);
            }
        }
}

static int pk_cus() {
    static int cus = 0;
    if (!cus) {
        int dev = 0;
        ESP_HIP(hipGetDevice(&dev));
        ESP_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    }
    return cus;
}

static void pk_finish(GemmEpi epi, const GemmArgs &a, int splits, hipStream_t s) {
    if (a.defer_splits) *a.defer_splits = splits;
    else launch_gemm_reduce(epi, a, a.ws, splits, s);
}

template <int EPI, int NB, int R, bool Q4, int P> static void pk_skinny(const GemmArgs &a, hipStream_t s) {
    constexpr int KU = PS_GK, BN = 128 / NB;
    constexpr size_t LDSB = (size_t)ps_keys<R, P>() * 16 * R * 2 * P;
    static bool attr = false;
    if (!attr) {
        for (const void *k : {reinterpret_cast<const void *>(gemm_pk_skinny_k<EPI, NB, R, Q4, P>),
                              reinterpret_cast<const void *>(gemm_pk_skinny_k<PK_PARTIAL, NB, R, Q4, P>)})
            ESP_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDSB));
        attr = true;
    }
    const int gx = (a.N + BN - 1) / BN, want = 2 * pk_cus();
    int splits = 1;
    while (gx * splits < want && a.K / (splits * 2) >= 256 && a.ws &&
           (size_t)(splits * 2) * NB * a.M * a.N * 4 <= a.ws_bytes)
        splits *= 2;
    const int kps = ((a.K + splits - 1) / splits + KU - 1) / KU * KU;
    splits = (a.K + kps - 1) / kps;
    if (splits == 1) {
        gemm_pk_skinny_k<EPI, NB, R, Q4, P><<<dim3(gx), 256, LDSB, s>>>(a, nullptr, a.K);
        return;
    }
    gemm_pk_skinny_k<PK_PARTIAL, NB, R, Q4, P><<<dim3(gx, 1, splits), 256, LDSB, s>>>(a, a.ws, kps);
    pk_finish((GemmEpi)EPI, a, splits, s);
}

template <int EPI, int NB, bool Q4, int P> static void pk_tile(GemmArgs a, hipStream_t s) {
    static bool attr = false;
    if (!attr) {
        for (const void *k : {reinterpret_cast<const void *>(gemm_pk_tile_k<EPI, NB, Q4, P>),
                              reinterpret_cast<const void *>(gemm_pk_tile_k<PK_PARTIAL, NB, Q4, P>)})
            ESP_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)pt_lds<P>()));
        attr = true;
    }
    constexpr int BN = PT_BR / NB;
    a.band = 4;
    const int nt = (a.N + BN - 1) / BN, mt = (a.M + PT_BM - 1) / PT_BM;
    const int blocks = PK_XCDS * ((nt * mt + PK_XCDS - 1) / PK_XCDS);
    // Two blocks sharing a CU work through a 32-key stage each in ~2.3 us, one
    // alone in ~1.7 (measured at 200 - 2048 rows, q8 and q4), and a launch
    // takes as long as the CU with most blocks: K is split, by any count, where
    // that evens the blocks out by more than the partial sums (written and
    // read once at ~4 TB/s) and their reduction cost.
    const long long tiles = (long long)nt * mt;
    int splits = 1;
    double best = 0;
    for (int sp = 1; sp == 1 || (sp <= 16 && a.K / sp >= 256 && a.ws &&
                                 (size_t)sp * NB * a.M * a.N * 4 <= a.ws_bytes); ++sp) {
        const long long n = (tiles * sp + pk_cus() - 1) / pk_cus();
        const double c = (double)(n / 2 * 2.34 + n % 2 * 1.7) * ((a.K / 32 + sp - 1) / sp) +
                         (sp > 1 ? 4.0 + (double)sp * NB * a.M * a.N * 2e-6 : 0.0);
        if (sp == 1 || c < best) best = c, splits = sp;
    }
    const int kps = ((a.K + splits - 1) / splits + 31) / 32 * 32;
    splits = (a.K + kps - 1) / kps;
    if (splits == 1) {
        gemm_pk_tile_k<EPI, NB, Q4, P><<<dim3(blocks), 256, pt_lds<P>(), s>>>(a, nullptr, a.K, mt, nt);
        return;
    }
    gemm_pk_tile_k<PK_PARTIAL, NB, Q4, P><<<dim3(blocks, 1, splits), 256, pt_lds<P>(), s>>>(a, a.ws, kps, mt, nt);
    pk_finish((GemmEpi)EPI, a, splits, s);
}

template <int EPI, bool Q4, int P = 2> static void pk_dispatch(const GemmArgs &a, hipStream_t s) {
    constexpr int NB = EPI == GEMM_SWIGLU ? 2 : 1;
    const bool line = a.K % PS_GK == 0;  // whole groups of every weight row
    if (a.M <= 16 && line) pk_skinny<EPI, NB, 1, Q4, P>(a, s);
    else if (a.M <= 32 && line) pk_skinny<EPI, NB, 2, Q4, P>(a, s);
    else if (a.M <= 64 && line) pk_skinny<EPI, NB, 4, Q4, P>(a, s);
    else pk_tile<EPI, NB, Q4, P>(a, s);
}

void launch_gemm_packed(Dt wt, GemmEpi epi, const GemmArgs &a, hipStream_t s) {
    auto al16 = [](const void *p) { return ((uintptr_t)p & 15) == 0; };
    if (!a.a_lo || !a.w_scale || a.K % 32 || a.grp_offs || !al16(a.a) || !al16(a.a_lo) || !al16(a.w) ||
        (epi == GEMM_SWIGLU && (!a.w2_scale || !al16(a.w2))) || (a.a_lo2 && (epi != GEMM_STORE || !al16(a.a_lo2))))
        fail(ESP_BACKEND, "packed GEMM: operands outside the block-32 form");
    const bool q4 = wt == DT_Q4;
    if (a.a_lo2) q4 ? pk_dispatch<GEMM_STORE, true, 3>(a, s) : pk_dispatch<GEMM_STORE, false, 3>(a, s);
    else if (epi == GEMM_STORE) q4 ? pk_dispatch<GEMM_STORE, true>(a, s) : pk_dispatch<GEMM_STORE, false>(a, s);
    else if (epi == GEMM_RESIDUAL) q4 ? pk_dispatch<GEMM_RESIDUAL, true>(a, s) : pk_dispatch<GEMM_RESIDUAL, false>(a, s);
    else q4 ? pk_dispatch<GEMM_SWIGLU, true>(a, s) : pk_dispatch<GEMM_SWIGLU, false>(a, s);
}

}  // namespace esp
