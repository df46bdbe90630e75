// GEMM kernels for bf16 operands: plain epilogues, the QKV split, the rebuilt LayerNorm residual.
#include "gemm_kernels.h"

namespace tnn_rocm {
template int GemmTyped<TNN_ROCM_BF16>::plain(hipStream_t, bool, const void *, const void *, void *, int, int, int, int,
    int, int, int, int, int, int, const float *, const void *, int);
template int GemmTyped<TNN_ROCM_BF16>::qkv_split(hipStream_t, const void *, const void *, const float *, void *, void *,
    int, int, int, int, int);
template int GemmTyped<TNN_ROCM_BF16>::residual_ln(hipStream_t, const void *, const void *, const float *, void *, const
    void *, const float *, const float *, const float *, int, int, int, int, float *, int *);
}  // namespace tnn_rocm
