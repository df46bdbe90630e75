// What the GEMM translation units share: the launch functions of one type (each defined in a file of its own, so that the
// kernels of the different types and epilogue families compile side by side) and the tuning hooks.
#ifndef TNN_ROCM_CSRC_GEMM_TYPED_H_
#define TNN_ROCM_CSRC_GEMM_TYPED_H_

#include <atomic>
#include <cstdlib>
#include <cstring>
#include <mutex>

#include "common.h"

namespace tnn_rocm {

constexpr int kMaxRowSumBlocks = TNN_ROCM_MAX_ROW_SUM_BLOCKS;
inline bool al16(const void *p) { return (((uintptr_t)p) & 15u) == 0; }

inline std::atomic<int> g_ln_y_ahead{1};  // experiment hook, see tnn_rocm_debug_set_ln_y_ahead
// tuning override for experiments: 0 = heuristic, otherwise a configuration code of the tiled kernel
// the hooks may be set while other threads launch: atomics, and a lock around the tuning table
inline std::atomic<int> g_gemm_force_cfg{0};
inline std::atomic<int> g_gemm_group_m{0};  // 0 = derived from the tile count; otherwise forced

// Experiment hook: "N:K:code,N:K:code,..." forces a configuration code for given (N, K); set from the environment
// variable TNN_ROCM_GEMM_TUNE at first use, or through tnn_rocm_debug_set_gemm_tune().
struct TuneEntry { int n, k, cfg, group_m; };
inline TuneEntry g_tune_table[16];
inline int g_tune_count = -1;
inline std::mutex g_tune_lock;
inline void parse_tune(const char *e) {  // caller holds g_tune_lock
    g_tune_count = 0;
    while (e && *e && g_tune_count < 16) {
        TuneEntry t;
        t.group_m = 0;
        if (sscanf(e, "%d:%d:%d:%d", &t.n, &t.k, &t.cfg, &t.group_m) >= 3)
            g_tune_table[g_tune_count++] = t;
        e = strchr(e, ',');
        if (e)
            ++e;
    }
}
inline int tune_override(int N, int K, int *group_m) {
    static std::once_flag env_read;  // instances on several threads may launch their first GEMM together
    std::call_once(env_read, [] {
        std::lock_guard<std::mutex> hold(g_tune_lock);
        if (g_tune_count < 0)
            parse_tune(getenv("TNN_ROCM_GEMM_TUNE"));
    });
    std::lock_guard<std::mutex> hold(g_tune_lock);
    for (int i = 0; i < g_tune_count; ++i)
        if (g_tune_table[i].n == N && g_tune_table[i].k == K) {
            if (group_m)
                *group_m = g_tune_table[i].group_m;
            return g_tune_table[i].cfg;
        }
    return 0;
}

// fp32 (plain only), fp16, bf16
template <int DT> struct GemmTyped {
    static int plain(hipStream_t s, bool b_is_nk, const void *A, const void *B, void *C, int M, int N, int K, int lda, int ldb,
                     int ldc, int batch, int batch_a, int batch_b, int epilogue, const float *bias, const void *residual,
                     int ldr);
    static int qkv_split(hipStream_t s, const void *x, const void *wqkv, const float *bqkv, void *qk, void *vt, int B, int S,
                         int heads, int K, int vt_key_order);
    static int ln(hipStream_t s, const void *t, const void *w_folded, const float *bias_folded, const float *colsum,
                  const float *gamma, const float *beta, float eps, void *C, void *y, float *row_stats, const float *row_sums,
                  int row_sum_blocks, int M, int N, int K, int flags, const void *residual);
    static int qkv_split_ln(hipStream_t s, const void *t, const void *wqkv_folded, const float *bqkv_folded,
                            const float *colsum, const float *gamma, const float *beta, float eps, void *qk, void *vt, void *y,
                            float *row_stats, const float *row_sums, int row_sum_blocks, int B, int S, int heads, int K,
                            int vt_key_order);
    static int residual_ln(hipStream_t s, const void *x, const void *w, const float *bias, void *C, const void *t,
                           const float *row_stats, const float *gamma, const float *beta, int M, int N, int K, int flags,
                           float *row_sums, int *row_sum_blocks);
};

struct GemmI8 {
    static int gemm(hipStream_t s, const int8_t *A, const int8_t *W, const int32_t *bias, const float *scale, int8_t *out_i8,
                    int32_t *acc_i32, int M, int N, int K, int lda, int ldw, int ldo, void *out_f, int out_f_dtype,
                    float dequant_scale, const void *residual, const int8_t *lut);
    template <int DT>  // the type of qk and vt
    static int qkv_split(hipStream_t s, const int8_t *x, const int8_t *wqkv, const int32_t *bias, const float *scale,
                         const float *dequant, void *qk, void *vt, int B, int S, int heads, int K, int vt_key_order);
};

}  // namespace tnn_rocm
#endif
