// C entry points of the GEMM family: argument checks, then the launch function of the type (gemm_typed.h).
#include "gemm_typed.h"

using namespace tnn_rocm;

extern "C" {

int tnn_rocm_gemm(void *stream, int dtype, int b_is_nk, const void *A, const void *B, void *C, int M, int N, int K,
                  int lda, int ldb, int ldc, int batch, int batch_a, int batch_b, int epilogue, const float *bias,
                  const void *residual, int ldr) {
    TR_REQUIRE(M >= 0 && N >= 0 && K >= 0 && batch >= 0, TNN_ROCM_ESHAPE, "gemm: negative size");
    if (M == 0 || N == 0 || batch == 0)
        return 0;
    TR_REQUIRE(A && B && C, TNN_ROCM_EINVAL, "gemm: null matrix pointer");
    TR_REQUIRE(K > 0, TNN_ROCM_ESHAPE, "gemm: K must be positive");
    TR_REQUIRE(batch_a >= 1 && batch_b >= 1 && batch_a <= batch && batch_b <= batch, TNN_ROCM_ESHAPE,
               "gemm: batch_a=%d batch_b=%d must lie in [1, batch=%d]", batch_a, batch_b, batch);
    TR_REQUIRE(lda >= K && ldc >= N && ldb >= (b_is_nk ? K : N), TNN_ROCM_ESHAPE,
               "gemm: leading dimension smaller than the row length");
    TR_REQUIRE((epilogue & ~7) == 0, TNN_ROCM_EINVAL, "gemm: unknown epilogue bits 0x%x", epilogue);
    TR_REQUIRE(!(epilogue & TNN_ROCM_EPI_BIAS) || bias, TNN_ROCM_EINVAL, "gemm: bias epilogue without bias");
    TR_REQUIRE(!(epilogue & TNN_ROCM_EPI_RESIDUAL) || (residual && ldr >= N), TNN_ROCM_EINVAL,
               "gemm: residual epilogue without residual / ldr");
    TR_REQUIRE(batch <= 65535, TNN_ROCM_ESHAPE, "gemm: batch %d exceeds 65535", batch);
    hipStream_t s = (hipStream_t)stream;
    auto run = dtype == TNN_ROCM_F32 ? &GemmTyped<TNN_ROCM_F32>::plain
               : dtype == TNN_ROCM_F16 ? &GemmTyped<TNN_ROCM_F16>::plain
               : dtype == TNN_ROCM_BF16 ? &GemmTyped<TNN_ROCM_BF16>::plain : nullptr;
    TR_REQUIRE(run, TNN_ROCM_EDTYPE, "gemm: unsupported dtype %d", dtype);
    return run(s, b_is_nk != 0, A, B, C, M, N, K, lda, ldb, ldc, batch, batch_a, batch_b, epilogue, bias, residual, ldr);
}

static int gemm_i8_impl(void *stream, const int8_t *A, const int8_t *W, const int32_t *bias, const float *scale,
                        int8_t *out_i8, int32_t *acc_i32, int M, int N, int K, int lda, int ldw, int ldo, void *out_f,
                        int out_f_dtype, float dequant_scale, const void *residual, const int8_t *lut = nullptr) {
    TR_REQUIRE(M >= 0 && N >= 0 && K >= 0, TNN_ROCM_ESHAPE, "gemm_i8: negative size");
    if (M == 0 || N == 0)
        return 0;
    TR_REQUIRE(A && W, TNN_ROCM_EINVAL, "gemm_i8: null matrix pointer");
    TR_REQUIRE(K > 0, TNN_ROCM_ESHAPE, "gemm_i8: K must be positive");
    TR_REQUIRE(out_i8 || acc_i32 || out_f, TNN_ROCM_EINVAL, "gemm_i8: no output requested");
    TR_REQUIRE(!(out_i8 || out_f) || scale, TNN_ROCM_EINVAL, "gemm_i8: requantised output needs scale[N]");
    TR_REQUIRE(lda >= K && ldw >= K && ldo >= N, TNN_ROCM_ESHAPE, "gemm_i8: leading dimension too small");
    TR_REQUIRE(!out_f || out_f_dtype == TNN_ROCM_F32 || out_f_dtype == TNN_ROCM_F16, TNN_ROCM_EDTYPE,
               "gemm_i8: dequantised output must be F32 or F16");
    TR_REQUIRE(!residual || out_f, TNN_ROCM_EINVAL, "gemm_i8: a residual needs the dequantised output");
    TR_REQUIRE(!lut || (out_i8 && !out_f && (((uintptr_t)lut) & 3u) == 0), TNN_ROCM_EINVAL,
               "gemm_i8: a lookup table applies to the int8 output only and must be 4-byte aligned");
    return GemmI8::gemm((hipStream_t)stream, A, W, bias, scale, out_i8, acc_i32, M, N, K, lda, ldw, ldo, out_f, out_f_dtype,
                        dequant_scale, residual, lut);
}

int tnn_rocm_gemm_i8(void *stream, const int8_t *A, const int8_t *W, const int32_t *bias, const float *scale,
                     int8_t *out_i8, int32_t *acc_i32, int M, int N, int K, int lda, int ldw, int ldo, void *out_f,
                     int out_f_dtype, float dequant_scale) {
    return gemm_i8_impl(stream, A, W, bias, scale, out_i8, acc_i32, M, N, K, lda, ldw, ldo, out_f, out_f_dtype,
                        dequant_scale, nullptr);
}

int tnn_rocm_gemm_i8_lut(void *stream, const int8_t *A, const int8_t *W, const int32_t *bias, const float *scale,
                         int8_t *out_i8, int M, int N, int K, int lda, int ldw, int ldo, const int8_t *lut) {
    TR_REQUIRE(out_i8 && lut, TNN_ROCM_EINVAL, "gemm_i8_lut: null pointer");
    return gemm_i8_impl(stream, A, W, bias, scale, out_i8, nullptr, M, N, K, lda, ldw, ldo, nullptr, 0, 0.f, nullptr, lut);
}

int tnn_rocm_gemm_i8_dequant_residual(void *stream, const int8_t *A, const int8_t *W, const int32_t *bias,
                                      const float *scale, int M, int N, int K, int lda, int ldw, void *out_f,
                                      int out_f_dtype, int ldo, float dequant_scale, const void *residual) {
    TR_REQUIRE(out_f, TNN_ROCM_EINVAL, "gemm_i8_dequant_residual: null output");
    return gemm_i8_impl(stream, A, W, bias, scale, nullptr, nullptr, M, N, K, lda, ldw, ldo, out_f, out_f_dtype,
                        dequant_scale, residual);
}

int tnn_rocm_gemm_i8_qkv_split(void *stream, int out_dtype, const int8_t *x, const int8_t *wqkv, const int32_t *bias,
                               const float *scale, const float *dequant, void *qk, void *vt, int B, int S, int heads,
                               int K, int vt_key_order) {
    TR_REQUIRE(vt_key_order == 0 || (vt_key_order == 1 && S % 16 == 0), TNN_ROCM_EINVAL,
               "gemm_i8_qkv_split: V^T key order %d (0 or 1; 1 needs S %% 16 == 0, S=%d)", vt_key_order, S);
    TR_REQUIRE(B >= 0 && S >= 0 && heads >= 0 && K >= 0, TNN_ROCM_ESHAPE, "gemm_i8_qkv_split: negative size");
    if (B == 0 || S == 0 || heads == 0)
        return 0;
    TR_REQUIRE(x && wqkv && scale && dequant && qk && vt, TNN_ROCM_EINVAL, "gemm_i8_qkv_split: null pointer");
    TR_REQUIRE(out_dtype == TNN_ROCM_F16 || out_dtype == TNN_ROCM_BF16, TNN_ROCM_EDTYPE,
               "gemm_i8_qkv_split: F16 or BF16 outputs only");
    TR_REQUIRE(K > 0 && K % 64 == 0, TNN_ROCM_ESHAPE, "gemm_i8_qkv_split: K=%d must be a positive multiple of 64", K);
    TR_REQUIRE((long)B * S < (1l << 24) && (long)B * S * 3 * heads * 64 < (1l << 31), TNN_ROCM_ESHAPE,
               "gemm_i8_qkv_split: problem too large for 32-bit panel offsets");
    TR_REQUIRE(al16(x) && al16(wqkv) && al16(qk) && al16(vt) && (!bias || al16(bias)) && al16(scale) && al16(dequant),
               TNN_ROCM_EALIGN, "gemm_i8_qkv_split: pointers must be 16-byte aligned");
    auto run = out_dtype == TNN_ROCM_F16 ? &GemmI8::qkv_split<TNN_ROCM_F16> : &GemmI8::qkv_split<TNN_ROCM_BF16>;
    return run((hipStream_t)stream, x, wqkv, bias, scale, dequant, qk, vt, B, S, heads, K, vt_key_order);
}

int tnn_rocm_gemm_qkv_split(void *stream, int dtype, const void *x, const void *wqkv, const float *bqkv, void *qk,
                            void *vt, int B, int S, int heads, int K, int vt_key_order) {
    TR_REQUIRE(vt_key_order == 0 || (vt_key_order == 1 && S % 16 == 0), TNN_ROCM_EINVAL,
               "gemm_qkv_split: V^T key order %d (0 or 1; 1 needs S %% 16 == 0, S=%d)", vt_key_order, S);
    TR_REQUIRE(B >= 0 && S >= 0 && heads >= 0 && K >= 0, TNN_ROCM_ESHAPE, "gemm_qkv_split: negative size");
    if (B == 0 || S == 0 || heads == 0)
        return 0;
    TR_REQUIRE(x && wqkv && qk && vt, TNN_ROCM_EINVAL, "gemm_qkv_split: null pointer");
    TR_REQUIRE(dtype == TNN_ROCM_F16 || dtype == TNN_ROCM_BF16, TNN_ROCM_EDTYPE, "gemm_qkv_split: F16 or BF16 only");
    TR_REQUIRE(K > 0 && K % 64 == 0, TNN_ROCM_ESHAPE, "gemm_qkv_split: K=%d must be a positive multiple of 64", K);
    TR_REQUIRE((long)B * S < (1l << 24) && (long)B * S * 3 * heads * 64 < (1l << 31), TNN_ROCM_ESHAPE,
               "gemm_qkv_split: problem too large for 32-bit panel offsets");
    TR_REQUIRE(al16(x) && al16(wqkv) && al16(qk) && al16(vt) && (!bqkv || al16(bqkv)), TNN_ROCM_EALIGN,
               "gemm_qkv_split: pointers must be 16-byte aligned");
    auto run = dtype == TNN_ROCM_F16 ? &GemmTyped<TNN_ROCM_F16>::qkv_split : &GemmTyped<TNN_ROCM_BF16>::qkv_split;
    return run((hipStream_t)stream, x, wqkv, bqkv, qk, vt, B, S, heads, K, vt_key_order);
}

int tnn_rocm_gemm_ln(void *stream, int dtype, const void *t, const void *w_folded, const float *bias_folded,
                     const float *colsum, const float *gamma, const float *beta, float eps, void *C, void *y,
                     float *row_stats, const float *row_sums, int row_sum_blocks, int M, int N, int K, int flags,
                     const void *residual) {
    TR_REQUIRE(M >= 0 && N >= 0 && K >= 0, TNN_ROCM_ESHAPE, "gemm_ln: negative size");
    if (M == 0 || N == 0)
        return 0;
    TR_REQUIRE(t && w_folded && bias_folded && colsum && C, TNN_ROCM_EINVAL, "gemm_ln: null pointer");
    TR_REQUIRE(!y || (gamma && beta), TNN_ROCM_EINVAL, "gemm_ln: the LayerNorm output needs gamma and beta");
    TR_REQUIRE(dtype == TNN_ROCM_F16 || dtype == TNN_ROCM_BF16, TNN_ROCM_EDTYPE, "gemm_ln: F16 or BF16 only");
    TR_REQUIRE(K > 0 && K % 128 == 0 && N % 8 == 0, TNN_ROCM_ESHAPE,
               "gemm_ln: K=%d must be a positive multiple of 128 and N=%d a multiple of 8", K, N);
    TR_REQUIRE((long)M < (1l << 24) && (long)N < (1l << 24) && (long)M * K < (1l << 31) && (long)N * K < (1l << 31) &&
                   (long)M * N < (1l << 31),
               TNN_ROCM_ESHAPE, "gemm_ln: problem too large for 32-bit panel offsets");
    TR_REQUIRE(!(flags & TNN_ROCM_EPI_RESIDUAL) || residual, TNN_ROCM_EINVAL, "gemm_ln: residual flag without a residual");
    TR_REQUIRE(!row_sums || (row_sum_blocks >= 1 && row_sum_blocks <= kMaxRowSumBlocks && (((uintptr_t)row_sums) & 7u) == 0),
               TNN_ROCM_EINVAL, "gemm_ln: row sums come in 1..%d blocks, 8-byte aligned", kMaxRowSumBlocks);
    TR_REQUIRE(al16(t) && al16(w_folded) && al16(C) && al16(bias_folded) && al16(colsum) && (!residual || al16(residual)) &&
                   (!y || (al16(y) && al16(gamma) && al16(beta))) && (((uintptr_t)row_stats) & 7u) == 0,
               TNN_ROCM_EALIGN, "gemm_ln: pointers must be 16-byte aligned (row_stats: 8-byte)");
    auto run = dtype == TNN_ROCM_F16 ? &GemmTyped<TNN_ROCM_F16>::ln : &GemmTyped<TNN_ROCM_BF16>::ln;
    return run((hipStream_t)stream, t, w_folded, bias_folded, colsum, gamma, beta, eps, C, y, row_stats, row_sums,
               row_sum_blocks, M, N, K, flags, residual);
}

int tnn_rocm_gemm_qkv_split_ln(void *stream, int dtype, const void *t, const void *wqkv_folded, const float *bqkv_folded,
                               const float *colsum, const float *gamma, const float *beta, float eps, void *qk, void *vt,
                               void *y, float *row_stats, const float *row_sums, int row_sum_blocks, int B, int S, int heads,
                               int K, int vt_key_order) {
    TR_REQUIRE(vt_key_order == 0 || (vt_key_order == 1 && S % 16 == 0), TNN_ROCM_EINVAL,
               "gemm_qkv_split_ln: V^T key order %d (0 or 1; 1 needs S %% 16 == 0, S=%d)", vt_key_order, S);
    TR_REQUIRE(B >= 0 && S >= 0 && heads >= 0 && K >= 0, TNN_ROCM_ESHAPE, "gemm_qkv_split_ln: negative size");
    if (B == 0 || S == 0 || heads == 0)
        return 0;
    TR_REQUIRE(t && wqkv_folded && bqkv_folded && colsum && qk && vt, TNN_ROCM_EINVAL, "gemm_qkv_split_ln: null pointer");
    TR_REQUIRE(!y || (gamma && beta), TNN_ROCM_EINVAL, "gemm_qkv_split_ln: the LayerNorm output needs gamma and beta");
    TR_REQUIRE(dtype == TNN_ROCM_F16 || dtype == TNN_ROCM_BF16, TNN_ROCM_EDTYPE, "gemm_qkv_split_ln: F16 or BF16 only");
    TR_REQUIRE(K > 0 && K % 128 == 0 && S % 8 == 0, TNN_ROCM_ESHAPE,
               "gemm_qkv_split_ln: K=%d must be a positive multiple of 128 and S=%d a multiple of 8", K, S);
    TR_REQUIRE((long)B * S < (1l << 24) && (long)heads * 192 < (1l << 24) && (long)B * S * 3 * heads * 64 < (1l << 31),
               TNN_ROCM_ESHAPE, "gemm_qkv_split_ln: problem too large for 32-bit panel offsets");
    TR_REQUIRE(al16(t) && al16(wqkv_folded) && al16(qk) && al16(vt) && al16(bqkv_folded) && al16(colsum) &&
                   (!y || (al16(y) && al16(gamma) && al16(beta))) && (((uintptr_t)row_stats) & 7u) == 0,
               TNN_ROCM_EALIGN, "gemm_qkv_split_ln: pointers must be 16-byte aligned (row_stats: 8-byte)");
    TR_REQUIRE(!row_sums || (row_sum_blocks >= 1 && row_sum_blocks <= kMaxRowSumBlocks && (((uintptr_t)row_sums) & 7u) == 0),
               TNN_ROCM_EINVAL, "gemm_qkv_split_ln: row sums come in 1..%d blocks, 8-byte aligned", kMaxRowSumBlocks);
    auto run = dtype == TNN_ROCM_F16 ? &GemmTyped<TNN_ROCM_F16>::qkv_split_ln : &GemmTyped<TNN_ROCM_BF16>::qkv_split_ln;
    return run((hipStream_t)stream, t, wqkv_folded, bqkv_folded, colsum, gamma, beta, eps, qk, vt, y, row_stats, row_sums,
               row_sum_blocks, B, S, heads, K, vt_key_order);
}

int tnn_rocm_gemm_residual_ln(void *stream, int dtype, const void *x, const void *w, const float *bias, void *C,
                              const void *t, const float *row_stats, const float *gamma, const float *beta, int M, int N,
                              int K, int flags, float *row_sums, int *row_sum_blocks) {
    TR_REQUIRE(M >= 0 && N >= 0 && K >= 0, TNN_ROCM_ESHAPE, "gemm_residual_ln: negative size");
    if (M == 0 || N == 0)
        return 0;
    TR_REQUIRE(x && w && C && t && row_stats && gamma && beta, TNN_ROCM_EINVAL, "gemm_residual_ln: null pointer");
    TR_REQUIRE(!(flags & TNN_ROCM_EPI_BIAS) || bias, TNN_ROCM_EINVAL, "gemm_residual_ln: bias flag without a bias");
    TR_REQUIRE(!(flags & ~(TNN_ROCM_EPI_BIAS | TNN_ROCM_EPI_GELU)), TNN_ROCM_EINVAL,
               "gemm_residual_ln: flags may name bias and GELU only (the residual is the rebuilt LayerNorm)");
    TR_REQUIRE(dtype == TNN_ROCM_F16 || dtype == TNN_ROCM_BF16, TNN_ROCM_EDTYPE, "gemm_residual_ln: F16 or BF16 only");
    TR_REQUIRE(K > 0 && K % 64 == 0 && N % 8 == 0, TNN_ROCM_ESHAPE,
               "gemm_residual_ln: K=%d must be a positive multiple of 64 and N=%d a multiple of 8", K, N);
    TR_REQUIRE((long)M < (1l << 24) && (long)N < (1l << 24) && (long)M * K < (1l << 31) && (long)N * K < (1l << 31) &&
                   (long)M * N < (1l << 31),
               TNN_ROCM_ESHAPE, "gemm_residual_ln: problem too large for 32-bit panel offsets");
    TR_REQUIRE(al16(x) && al16(w) && al16(C) && al16(t) && al16(gamma) && al16(beta) && (!bias || al16(bias)) &&
                   (((uintptr_t)row_stats) & 7u) == 0,
               TNN_ROCM_EALIGN, "gemm_residual_ln: pointers must be 16-byte aligned (row_stats: 8-byte)");
    TR_REQUIRE(!row_sums || (row_sum_blocks && (((uintptr_t)row_sums) & 7u) == 0), TNN_ROCM_EINVAL,
               "gemm_residual_ln: the row sums need an 8-byte aligned buffer and a place for their block count");
    if (row_sum_blocks)
        *row_sum_blocks = 0;
    auto run = dtype == TNN_ROCM_F16 ? &GemmTyped<TNN_ROCM_F16>::residual_ln : &GemmTyped<TNN_ROCM_BF16>::residual_ln;
    return run((hipStream_t)stream, x, w, bias, C, t, row_stats, gamma, beta, M, N, K, flags, row_sums, row_sum_blocks);
}

// Experiment hook (not part of the documented ABI): 0 restores the shape heuristic, -1 forces the baseline
// kernel, other values select a configuration code of the tiled kernel.
__attribute__((visibility("default"))) int tnn_rocm_debug_set_gemm_config(int cfg) {
    g_gemm_force_cfg = cfg;
    return 0;
}
__attribute__((visibility("default"))) int tnn_rocm_debug_set_gemm_tune(const char *spec) {
    std::lock_guard<std::mutex> hold(g_tune_lock);
    parse_tune(spec);
    return 0;
}
__attribute__((visibility("default"))) int tnn_rocm_debug_set_ln_y_ahead(int on) {
    g_ln_y_ahead = on ? 1 : 0;
    return 0;
}
__attribute__((visibility("default"))) int tnn_rocm_debug_set_gemm_group_m(int group_m) {
    g_gemm_group_m = group_m;
    return 0;
}

}  // extern "C"
