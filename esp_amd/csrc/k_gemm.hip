// Projection GEMM dispatch: C[M,N] = A[M,K] . W[N,K]^T.
#include "common.hpp"
#include "kernels_extra.hpp"

namespace esp {

bool gemm_mfma_ok(Dt wt, const GemmArgs &a);
void launch_gemm_mfma(GemmEpi epi, const GemmArgs &a, float *ws, size_t ws_bytes, hipStream_t s);
bool gemm_rows_ok(const GemmArgs &a);
void launch_gemm_rows(GemmEpi epi, const GemmArgs &a, hipStream_t s);
bool gemm_f32_ok(Dt wt, const GemmArgs &a);
void launch_gemm_f32(GemmEpi epi, const GemmArgs &a, hipStream_t s);
void launch_gemm_packed(Dt wt, GemmEpi epi, const GemmArgs &a, hipStream_t s);

bool gemm_takes_rows(Dt wt, const GemmArgs &a) { return gemm_mfma_ok(wt, a) && gemm_rows_ok(a); }

// bf16 and packed weights go to the bf16 matrix cores (activations split into
// bf16 hi + lo), f32 weights to the f32 ones. The vector-ALU kernel takes what
// they do not: f32 with K no multiple of 16, bf16 with K no multiple of 8 or
// below 32, unaligned operands.
void launch_gemm(Dt wt, GemmEpi epi, const GemmArgs &a, hipStream_t s) {
    if (a.defer_splits) *a.defer_splits = 0;
    if (a.M <= 0 || a.N <= 0) return;
    if (dt_packed(wt)) launch_gemm_packed(wt, epi, a, s);
    else if (a.a_lo2) fail(ESP_BACKEND, "GEMM: three activation planes outside the packed form");
    else if (gemm_takes_rows(wt, a)) launch_gemm_rows(epi, a, s);
    else if (a.a_rows) fail(ESP_BACKEND, "GEMM: row table outside the few-row form");
    else if (gemm_mfma_ok(wt, a)) launch_gemm_mfma(epi, a, a.ws, a.ws ? a.ws_bytes : 0, s);
    else if (gemm_f32_ok(wt, a)) launch_gemm_f32(epi, a, s);
    else launch_gemm_simple(wt, epi, a, s);
}

}  // namespace esp
