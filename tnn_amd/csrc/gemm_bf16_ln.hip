// GEMM kernels for bf16 operands with a LayerNorm folded in.
#include "gemm_kernels.h"

namespace tnn_rocm {
template int GemmTyped<TNN_ROCM_BF16>::ln(hipStream_t, const void *, const void *, const float *, const float *, const
    float *, const float *, float, void *, void *, float *, const float *, int, int, int, int, int, const void *);
template int GemmTyped<TNN_ROCM_BF16>::qkv_split_ln(hipStream_t, const void *, const void *, const float *, const float
    *, const float *, const float *, float, void *, void *, void *, float *, const float *, int, int, int, int, int,
    int);
}  // namespace tnn_rocm
