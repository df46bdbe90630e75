// GEMM kernels for fp32 operands.
#include "gemm_kernels.h"

namespace tnn_rocm {
template int GemmTyped<TNN_ROCM_F32>::plain(hipStream_t, bool, const void *, const void *, void *, int, int, int, int,
    int, int, int, int, int, int, const float *, const void *, int);
}  // namespace tnn_rocm
