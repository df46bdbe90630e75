// GEMM kernels for int8 operands.
#include "gemm_kernels.h"

namespace tnn_rocm {

int GemmI8::gemm(hipStream_t s, const int8_t *A, const int8_t *W, const int32_t *bias, const float *scale,
                        int8_t *out_i8, int32_t *acc_i32, int M, int N, int K, int lda, int ldw, int ldo, void *out_f,
                        int out_f_dtype, float dequant_scale, const void *residual, const int8_t *lut) {
    const bool aligned = al16(A) && al16(W) && lda % 16 == 0 && ldw % 16 == 0 && K % 16 == 0;
    Int8Epilogue epi;
    epi.lut         = lut;
    epi.bias        = bias;
    epi.scale       = scale;
    epi.out         = out_i8;
    epi.acc_out     = acc_i32;
    epi.ldo         = ldo;
    epi.out_f       = out_f;
    epi.out_f_dtype = out_f_dtype;
    epi.dq          = dequant_scale;
    epi.residual    = residual;
    const bool vec_out = ldo % 8 == 0 && (!bias || al16(bias)) && (!scale || al16(scale)) &&
                         (!out_i8 || (((uintptr_t)out_i8) & 7u) == 0) && (!acc_i32 || al16(acc_i32)) && (!out_f || al16(out_f)) &&
                         (!residual || al16(residual));
    if (aligned && vec_out && g_gemm_force_cfg >= 0 && K % 64 == 0)
        return launch_gemm_fast<TNN_ROCM_I8, Int8Epilogue>(s, A, W, M, N, K, lda, ldw, epi);
    return launch_gemm<TNN_ROCM_I8, Int8Epilogue>(s, true, aligned, A, W, M, N, K, lda, ldw, 1, 1, 1, 0, 0, epi);
}

template <int DT>
int GemmI8::qkv_split(hipStream_t s, const int8_t *x, const int8_t *wqkv, const int32_t *bias, const float *scale,
                      const float *dequant, void *qk, void *vt, int B, int S, int heads, int K, int vt_key_order) {
    const int H = heads * 64, T = B * S;
    Int8QkvSplitEpilogue<DT> epi;
    epi.bias    = bias;
    epi.scale   = scale;
    epi.dequant = dequant;
    epi.qk      = (typename Elem<DT>::type *)qk;
    epi.vt      = (typename Elem<DT>::type *)vt;
    epi.H       = H;
    epi.S       = S;
    epi.heads   = heads;
    epi.vt_sh   = vt_key_order;
    return launch_gemm_fast<TNN_ROCM_I8, Int8QkvSplitEpilogue<DT>>(s, x, wqkv, T, 3 * H, K, K, K, epi);
}

template int GemmI8::qkv_split<TNN_ROCM_F16>(hipStream_t, const int8_t *, const int8_t *, const int32_t *, const float *,
    const float *, void *, void *, int, int, int, int, int);
template int GemmI8::qkv_split<TNN_ROCM_BF16>(hipStream_t, const int8_t *, const int8_t *, const int32_t *, const float *,
    const float *, void *, void *, int, int, int, int, int);

}  // namespace tnn_rocm
