// Row-wise HBM-bound kernels: LayerNorm (+residual, +int8 quantised copy) and Softmax.
//
// One 64-lane wavefront owns one row (LayerNorm rows of at most 128 vectors: half a wavefront): the row is read
// once with 16-byte accesses, kept in registers, reduced with cross-lane shuffles (no LDS), and written once.
// Four waves per workgroup, so a launch over T rows issues T/4 or T/8 workgroups (>> 256 CUs for encoder shapes).
#include "common.h"

using namespace tnn_rocm;

namespace {

constexpr int kBlock       = 256;
constexpr int kRowsPerBlk  = kBlock / kWave;
constexpr int kMaxVecPerLn = 8;  // row cached in registers when cols <= 64 * VEC * 8

__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        v += __shfl_xor(v, o, 64);
    return v;
}

// sum over each aligned group of LPR lanes (32: the two halves of a wave hold different rows)
template <int LPR> __device__ __forceinline__ double lanes_sum_f64(double v) {
    if constexpr (LPR == 64)
        v = add_lane_xor<32>(v);
    v = add_lane_xor<16>(v);
    v = add_lane_xor<8>(v);
    v = add_lane_xor<4>(v);
    v = add_lane_xor<2>(v);
    return add_lane_xor<1>(v);
}

// ---- LayerNorm ----------------------------------------------------------------------------------
// Statistics follow the reference's one-pass form var = E[x^2] - E[x]^2 with its types: the square
// is an fp32 product, both sums, the mean, the variance and rstd are double.  An all-fp32
// E[x^2]-E[x]^2 loses the variance to cancellation when |mean| >> std.
// Optional row sources of the embedding front end: row r of the input is word_table[ids[r]] (x is the table),
// the residual is pos_table[r % period] (res is the table) and a second addend type_table[type_ids[r]]; the sum is
// ((word + pos) + type), the order of the Add layers it replaces.
struct EmbedRows {
    const int32_t *ids      = nullptr;  // null: plain LayerNorm
    const int32_t *type_ids = nullptr;
    const void *type_table  = nullptr;
    int vocab = 0, n_types = 0, period = 0;
    // optional third lookup: row r takes position row pos_ids[r % n_pos_ids] of a table of pos_rows rows
    const int32_t *pos_ids = nullptr;
    int n_pos_ids = 0, pos_rows = 0;
    int32_t *error_flag = nullptr;
};

// LPR lanes own one row (64: a wave per row; 32: a wave holds two rows, which keeps every lane busy and twice the
// bytes in flight for rows of at most 128 vectors); NV = 16-byte vectors a lane can hold.
// AHEAD: everything the row needs is requested at once, scale and shift among it.  Requested where they are used they are a
// second latency behind the reduction; the registers they take meanwhile cost resident waves.
// VB: bytes of a vector, 16 or, for half types, 8.
template <int DT, bool VECTOR, int LPR, int NV, bool AHEAD, int VB = 16>
__global__ void __launch_bounds__(kBlock) layernorm_kernel(const typename Elem<DT>::type *__restrict__ x,
                                                           const typename Elem<DT>::type *__restrict__ res,
                                                           const float *__restrict__ gamma,
                                                           const float *__restrict__ beta,
                                                           typename Elem<DT>::type *__restrict__ y, int rows, int cols,
                                                           float eps, int8_t *__restrict__ out_q, float q_inv,
                                                           EmbedRows emb, StoreThrough mode) {
    typedef typename Elem<DT>::type T;
    touch_kernel_args<7 * 8 + 3 * 8 + sizeof(EmbedRows)>();
    typedef typename std::conditional<VB == 16, uint4, uint2>::type Raw;
    constexpr int VEC = VECTOR ? (int)(VB / sizeof(T)) : 1;
    const int lane    = threadIdx.x & (LPR - 1);
    const int row     = (blockIdx.x * kRowsPerBlk + (threadIdx.x >> 6)) * (kWave / LPR) + ((threadIdx.x & (kWave - 1)) / LPR);
    if (row >= rows)
        return;  // the lanes of a row exit together; no workgroup barrier is used below and shuffles stay inside a row
    const T *px  = x + (size_t)row * cols;
    const T *pr  = res ? res + (size_t)row * cols : nullptr;
    const T *pr2 = nullptr;
    if (VECTOR && emb.ids) {
        // negative indices wrap, an index outside the table raises the flag and reads row 0
        // (cpu_gather_layer_acc.cc:27-86)
        int wi = emb.ids[row], ti = emb.type_ids[row];
        int pi = emb.pos_ids ? emb.pos_ids[row % emb.n_pos_ids] : row % emb.period;
        wi += wi < 0 ? emb.vocab : 0;
        ti += ti < 0 ? emb.n_types : 0;
        bool bad = wi < 0 || wi >= emb.vocab || ti < 0 || ti >= emb.n_types;
        if (emb.pos_ids) {
            pi += pi < 0 ? emb.pos_rows : 0;
            bad |= pi < 0 || pi >= emb.pos_rows;
        }
        if (bad) {
            if (lane == 0 && emb.error_flag)
                *emb.error_flag = 1;
            wi = 0, ti = 0, pi = 0;
        }
        px  = x + (size_t)wi * cols;
        pr  = res + (size_t)pi * cols;
        pr2 = reinterpret_cast<const T *>(emb.type_table) + (size_t)ti * cols;
    }
    T *py        = y + (size_t)row * cols;
    int8_t *pq   = out_q ? out_q + (size_t)row * cols : nullptr;
    const int nv = cols / VEC;  // VECTOR launches guarantee cols % VEC == 0

    float v[NV][VEC];
    double s1 = 0.0, s2 = 0.0;
    Raw raw[NV], rraw[NV], rraw2[NV];
    float gam[NV][VEC], bet[NV][VEC];
    auto request = [&](int j, int vi) __attribute__((always_inline)) {
        raw[j] = reinterpret_cast<const Raw *>(px)[vi];
        if (pr)
            rraw[j] = reinterpret_cast<const Raw *>(pr)[vi];
        if (pr2)
            rraw2[j] = reinterpret_cast<const Raw *>(pr2)[vi];
    };
    auto request_affine = [&](int j, int vi) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < VEC; ++t)
            gam[j][t] = gamma[vi * VEC + t], bet[j][t] = beta[vi * VEC + t];
    };
    if constexpr (AHEAD) {  // what lies behind the row is clamped and not used
#pragma unroll
        for (int j = 0; j < NV; ++j)
            request(j, lane + j * LPR < nv ? lane + j * LPR : nv - 1);
#pragma unroll
        for (int j = 0; j < NV; ++j)
            request_affine(j, lane + j * LPR < nv ? lane + j * LPR : nv - 1);
    }
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        int vi = lane + j * LPR;
        if (vi < nv) {
            if (VECTOR) {
                if constexpr (!AHEAD)
                    request(j, vi);
                const T *e = reinterpret_cast<const T *>(&raw[j]);
                const T *re = reinterpret_cast<const T *>(&rraw[j]), *re2 = reinterpret_cast<const T *>(&rraw2[j]);
#pragma unroll
                for (int t = 0; t < VEC; ++t) {
                    float f = Elem<DT>::ld(&e[t]);
                    if (pr)
                        f = __fadd_rn(f, Elem<DT>::ld(&re[t]));
                    if (pr2)
                        f = __fadd_rn(f, Elem<DT>::ld(&re2[t]));
                    v[j][t] = f;
                }
            } else {
                float f = Elem<DT>::ld(&px[vi]);
                if (pr)
                    f = __fadd_rn(f, Elem<DT>::ld(&pr[vi]));
                v[j][0] = f;
            }
#pragma unroll
            for (int t = 0; t < VEC; ++t) {
                s1 += (double)v[j][t];
                s2 += (double)__fmul_rn(v[j][t], v[j][t]);  // fp32 square, double sum (as the reference)
            }
        }
    }
    double d1    = lanes_sum_f64<LPR>(s1);
    double d2    = lanes_sum_f64<LPR>(s2);
    double mean  = d1 / cols;
    double var   = d2 / cols - mean * mean;
    double rstdd;
    if (DT == TNN_ROCM_F32) {
        rstdd = 1.0 / sqrt(var + (double)eps);  // the reference's expression, correctly rounded
    } else {
        // only the fp32 roundings of rstd and mean*rstd are used below: the hardware estimate (about 2^-26 relative)
        // refined by one Newton step is within a few double ulps, far inside what those roundings can see
        const double a = var + (double)eps;
        double r       = __builtin_amdgcn_rsq(a);
        rstdd          = r + r * (0.5 - 0.5 * a * r * r);
    }
    float rstd   = (float)rstdd;
    float mrs    = (float)(mean * rstdd);

#pragma unroll
    for (int j = 0; j < NV; ++j) {
        int vi = lane + j * LPR;
        if (vi < nv) {
            if constexpr (!AHEAD)
                request_affine(j, vi);
            float o[VEC];
#pragma unroll
            for (int t = 0; t < VEC; ++t) {
                float k = gam[j][t];
                if (DT == TNN_ROCM_F32) {
                    // the reference's operand order and widths (cpu_layer_norm_layer_acc.cc:126-131): the shifted
                    // bias is formed in double and rounded to float, the affine combination is evaluated in double
                    float b = (float)((double)bet[j][t] - mean * rstdd * (double)k);
                    o[t]    = (float)((double)v[j][t] * rstdd * (double)k + (double)b);
                } else {
                    float b = bet[j][t] - mrs * k;
                    o[t]    = v[j][t] * rstd * k + b;
                }
            }
            if (VECTOR) {
                Raw out;
                T *e = reinterpret_cast<T *>(&out);
#pragma unroll
                for (int t = 0; t < VEC; ++t)
                    Elem<DT>::st(&e[t], o[t]);
                if constexpr (VB == 16)
                    store_out16(mode.through, reinterpret_cast<uint4 *>(py) + vi, store_u32x4{out.x, out.y, out.z, out.w});
                else
                    store_out8(mode.through, reinterpret_cast<uint2 *>(py) + vi, store_u32x2{out.x, out.y});
                if (pq) {  // the VEC (4 or 8) quantised values of this lane leave as one 4- or 8-byte store
                    uint32_t w[2] = {0u, 0u};
#pragma unroll
                    for (int t = 0; t < VEC; ++t) {
                        const int8_t q = float2int8_ref(__fmul_rn(Elem<DT>::ld(&e[t]), q_inv));
                        w[t >> 2] |= (uint32_t)(uint8_t)q << (8 * (t & 3));
                    }
                    if (VEC == 8)
                        store_out8(mode.through, pq + (size_t)vi * VEC, store_u32x2{w[0], w[1]});
                    else
                        store_out4(mode.through, pq + (size_t)vi * VEC, w[0]);
                }
            } else {
                T tmp;
                Elem<DT>::st(&tmp, o[0]);
                py[vi] = tmp;
                if (pq)
                    pq[vi] = float2int8_ref(__fmul_rn(Elem<DT>::ld(&tmp), q_inv));
            }
        }
    }
}

// Rows too long for the register cache: three passes over the row (statistics, then output).
template <int DT>
__global__ void __launch_bounds__(kBlock) layernorm_long_kernel(const typename Elem<DT>::type *__restrict__ x,
                                                                const typename Elem<DT>::type *__restrict__ res,
                                                                const float *__restrict__ gamma,
                                                                const float *__restrict__ beta,
                                                                typename Elem<DT>::type *__restrict__ y, int rows,
                                                                int cols, float eps, int8_t *__restrict__ out_q,
                                                                float q_inv) {
    typedef typename Elem<DT>::type T;
    const int lane = threadIdx.x & (kWave - 1);
    const int row  = blockIdx.x * kRowsPerBlk + (threadIdx.x >> 6);
    if (row >= rows)
        return;
    const T *px = x + (size_t)row * cols;
    const T *pr = res ? res + (size_t)row * cols : nullptr;
    T *py       = y + (size_t)row * cols;
    int8_t *pq  = out_q ? out_q + (size_t)row * cols : nullptr;
    double s1 = 0, s2 = 0;
    for (int c = lane; c < cols; c += kWave) {
        float f = Elem<DT>::ld(&px[c]);
        if (pr)
            f = __fadd_rn(f, Elem<DT>::ld(&pr[c]));
        s1 += (double)f;
        s2 += (double)__fmul_rn(f, f);
    }
    s1           = wave_sum_f64(s1);
    s2           = wave_sum_f64(s2);
    double mean  = s1 / cols;
    double var   = s2 / cols - mean * mean;
    double rstdd = 1.0 / sqrt(var + (double)eps);
    float rstd   = (float)rstdd;
    float mrs    = (float)(mean * rstdd);
    for (int c = lane; c < cols; c += kWave) {
        float f = Elem<DT>::ld(&px[c]);
        if (pr)
            f = __fadd_rn(f, Elem<DT>::ld(&pr[c]));
        float k = gamma[c];
        float o;
        if (DT == TNN_ROCM_F32) {
            float b = (float)((double)beta[c] - mean * rstdd * (double)k);
            o       = (float)((double)f * rstdd * (double)k + (double)b);
        } else {
            o = f * rstd * k + (beta[c] - mrs * k);
        }
        T tmp;
        Elem<DT>::st(&tmp, o);
        py[c] = tmp;
        if (pq)
            pq[c] = float2int8_ref(__fmul_rn(Elem<DT>::ld(&tmp), q_inv));
    }
}

template <int DT>
int launch_layernorm(hipStream_t s, const void *x, const void *res, const float *gamma, const float *beta, void *y,
                     int rows, int cols, float eps, int8_t *out_q, float q_inv, const EmbedRows &emb = EmbedRows()) {
    typedef typename Elem<DT>::type T;
    constexpr int VEC = 16 / sizeof(T);
    dim3 grid((rows + kRowsPerBlk - 1) / kRowsPerBlk), block(kBlock);
    const int nv = cols / VEC;
    bool al = ((((uintptr_t)x) | ((uintptr_t)y) | ((uintptr_t)res) | ((uintptr_t)emb.type_table) | ((uintptr_t)out_q)) & 15u) == 0 &&
              cols % VEC == 0;
    if (emb.ids && !(al && cols <= kWave * VEC * kMaxVecPerLn)) {
        set_error("embed_layernorm: hidden size %d needs 16-byte aligned rows of at most %d elements", cols,
                  kWave * VEC * kMaxVecPerLn);
        return TNN_ROCM_ESHAPE;
    }
    if (al && cols <= kWave * VEC * kMaxVecPerLn) {
        // Everything requested ahead where all rows are resident at once: the launch is as long as one row's chain.  More rows, and
        // other waves cover it, of which the registers taken leave fewer: 196608 rows of 1024 with a residual 158 us, 222 requested
        // ahead.  How many rows that is follows from the registers of the form: HALF / F32 workgroups a CU (of eight rows, or of
        // four where a wave owns one).  us with a residual, requested where used -> ahead, at the last rows that are resident and
        // at more of them:
        //   fp16  768 columns 6144 rows 6.1 -> 6.0, 12288 9.9 -> 11.5     1536 4096 7.2 -> 7.1, 6144 9.6 -> 11.0
        //        2048 3072 7.2 -> 7.1, 4096 8.7 -> 10.0                   2304 1024 5.9 -> 6.0, 2048 7.4 -> 11.2, 4096 10.6 -> 23.5
        //   fp32 1024 4096 7.2 -> 6.6, 5120 10.8 -> 11.5                  2048 2048 10.0 -> 7.2, 4096 16.4 -> 18.0
#define TR_LN_LAUNCH(LPR, NV, AHEAD)                                                                                  \
    hipLaunchKernelGGL((layernorm_kernel<DT, true, LPR, NV, AHEAD>),                                                  \
                       dim3((rows + kRowsPerBlk * (kWave / LPR) - 1) / (kRowsPerBlk * (kWave / LPR))), block, 0, s,   \
                       (const T *)x, (const T *)res, gamma, beta, (T *)y, rows, cols, eps, out_q, q_inv, emb,     \
                       StoreThrough())
#define TR_LN(LPR, NV, HALF, F32)                                                                                     \
    do {                                                                                                              \
        constexpr int resident = kNumCU * kRowsPerBlk * (kWave / LPR) * (DT == TNN_ROCM_F32 ? F32 : HALF);            \
        if (rows <= resident)                                                                                         \
            TR_LN_LAUNCH(LPR, NV, true);                                                                              \
        else                                                                                                          \
            TR_LN_LAUNCH(LPR, NV, false);                                                                             \
    } while (0)
        // Few half rows of 257 to 1024 columns: a wave a row and vectors of eight bytes, so that a lane adds up 8 to 16 values in
        // double, not 16 to 32; that chain is most of such a launch.  Up to three workgroups a CU; from there on the waves, twice
        // as many, cost more than the shorter chain gives.  The sums in double differ from those of the form below by their order alone, some 2^-50
        // of a sum, which the roundings to fp32 behind them leave nothing of but in a rare tie.  us with a residual and an int8 copy, half a wave a row -> this:
        //   768 columns  128 rows 4.68 -> 4.06, 1024 4.98 -> 4.10, 3072 5.88 -> 5.43, 4096 6.09 -> 6.31
        //   1024         128      5.51 -> 4.49, 3072 7.04 -> 6.40, 4096 7.48 -> 7.35 (without the copy 6.35 -> 6.56)
        //   256          1024     3.10 -> 3.00, 2048 3.37 -> 3.51          embedding, 768, 128 rows 6.61 -> 6.09, 4096 7.67 -> 8.07
        if constexpr (DT != TNN_ROCM_F32) {
            if (cols > 256 && cols <= 1024 && rows <= 3 * kNumCU * kRowsPerBlk) {
#define TR_LN_FEW(NV)                                                                                                 \
    hipLaunchKernelGGL((layernorm_kernel<DT, true, 64, NV, true, 8>), grid, block, 0, s, (const T *)x, (const T *)res, gamma, \
                       beta, (T *)y, rows, cols, eps, out_q, q_inv, emb, StoreThrough())
                if (cols <= 512)
                    TR_LN_FEW(2);
                else if (cols <= 768)
                    TR_LN_FEW(3);
                else
                    TR_LN_FEW(4);
#undef TR_LN_FEW
                TR_CHECK_LAUNCH();
                return 0;
            }
        }
        if (nv <= 32)  // a second vector of a lane would be requested twice: 8192 embedded rows of 256 halves 6.6 us with it
            TR_LN(32, 1, 8, 8);
        else if (nv <= 64)
            TR_LN(32, 2, 5, 8);
        else if (nv <= 96)
            TR_LN(32, 3, 4, 6);
        else if (nv <= 128)
            TR_LN(32, 4, 3, 4);
        else if (nv <= 192)
            TR_LN(64, 3, 4, 6);
        else if (nv <= 256)
            TR_LN(64, 4, 3, 4);
        else
            TR_LN(64, 8, 1, 2);
#undef TR_LN
#undef TR_LN_LAUNCH
    } else if (cols <= kWave * kMaxVecPerLn) {
        hipLaunchKernelGGL((layernorm_kernel<DT, false, kWave, kMaxVecPerLn, false>), grid, block, 0, s, (const T *)x,
                           (const T *)res, gamma, beta, (T *)y, rows, cols, eps, out_q, q_inv, emb, StoreThrough());
    } else {
        hipLaunchKernelGGL((layernorm_long_kernel<DT>), grid, block, 0, s, (const T *)x, (const T *)res, gamma, beta,
                           (T *)y, rows, cols, eps, out_q, q_inv);
    }
    TR_CHECK_LAUNCH();
    return 0;
}

// ---- Softmax ------------------------------------------------------------------------------------
constexpr int kSmMaxPerLane = 16;  // last-axis rows up to 1024 values stay in registers

// inner == 1: one wave per row.
template <int DT>
__global__ void __launch_bounds__(kBlock) softmax_lastaxis_kernel(const typename Elem<DT>::type *__restrict__ x,
                                                                  typename Elem<DT>::type *__restrict__ y, int rows,
                                                                  int channel) {
    const int lane = threadIdx.x & (kWave - 1);
    const int row  = blockIdx.x * kRowsPerBlk + (threadIdx.x >> 6);
    if (row >= rows)
        return;
    const typename Elem<DT>::type *px = x + (size_t)row * channel;
    typename Elem<DT>::type *py       = y + (size_t)row * channel;
    if (channel <= kWave * kSmMaxPerLane) {
        float v[kSmMaxPerLane];
        float mx = -INFINITY;
#pragma unroll
        for (int j = 0; j < kSmMaxPerLane; ++j) {
            int c = lane + j * kWave;
            v[j]  = c < channel ? Elem<DT>::ld(&px[c]) : -INFINITY;
            mx    = fmaxf(mx, v[j]);
        }
        mx        = wave_max(mx);
        float sum = 0.f;
#pragma unroll
        for (int j = 0; j < kSmMaxPerLane; ++j) {
            int c = lane + j * kWave;
            v[j]  = c < channel ? expf(v[j] - mx) : 0.f;
            sum += v[j];
        }
        sum       = wave_sum(sum);
        float inv = 1.0f / sum;
#pragma unroll
        for (int j = 0; j < kSmMaxPerLane; ++j) {
            int c = lane + j * kWave;
            if (c < channel)
                Elem<DT>::st(&py[c], v[j] * inv);
        }
    } else {
        float mx = -INFINITY;
        for (int c = lane; c < channel; c += kWave)
            mx = fmaxf(mx, Elem<DT>::ld(&px[c]));
        mx        = wave_max(mx);
        float sum = 0.f;
        for (int c = lane; c < channel; c += kWave)
            sum += expf(Elem<DT>::ld(&px[c]) - mx);
        sum       = wave_sum(sum);
        float inv = 1.0f / sum;
        for (int c = lane; c < channel; c += kWave)
            Elem<DT>::st(&py[c], expf(Elem<DT>::ld(&px[c]) - mx) * inv);
    }
}

// inner > 1: one lane per (outer, inner) column; consecutive lanes touch consecutive addresses.
template <int DT>
__global__ void __launch_bounds__(kBlock) softmax_strided_kernel(const typename Elem<DT>::type *__restrict__ x,
                                                                 typename Elem<DT>::type *__restrict__ y, int outer,
                                                                 int channel, int inner) {
    size_t total  = (size_t)outer * inner;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
        size_t n = i / inner, e = i % inner;
        const typename Elem<DT>::type *px = x + n * channel * inner + e;
        typename Elem<DT>::type *py       = y + n * channel * inner + e;
        float mx                          = -INFINITY;
        for (int c = 0; c < channel; ++c)
            mx = fmaxf(mx, Elem<DT>::ld(&px[(size_t)c * inner]));
        float sum = 0.f;
        for (int c = 0; c < channel; ++c)
            sum += expf(Elem<DT>::ld(&px[(size_t)c * inner]) - mx);
        float inv = 1.0f / sum;
        for (int c = 0; c < channel; ++c)
            Elem<DT>::st(&py[(size_t)c * inner], expf(Elem<DT>::ld(&px[(size_t)c * inner]) - mx) * inv);
    }
}

template <int DT>
int launch_softmax(hipStream_t s, const void *x, void *y, int outer, int channel, int inner) {
    typedef typename Elem<DT>::type T;
    if (inner == 1) {
        dim3 grid((outer + kRowsPerBlk - 1) / kRowsPerBlk);
        hipLaunchKernelGGL((softmax_lastaxis_kernel<DT>), grid, dim3(kBlock), 0, s, (const T *)x, (T *)y, outer,
                           channel);
    } else {
        size_t total = (size_t)outer * inner;
        size_t g     = (total + kBlock - 1) / kBlock;
        if (g > 4096)
            g = 4096;
        hipLaunchKernelGGL((softmax_strided_kernel<DT>), dim3((unsigned)g), dim3(kBlock), 0, s, (const T *)x, (T *)y,
                           outer, channel, inner);
    }
    TR_CHECK_LAUNCH();
    return 0;
}

}  // namespace

extern "C" {
int tnn_rocm_layernorm(void *stream, int dtype, const void *x, const void *residual, const float *gamma,
                       const float *beta, void *y, int rows, int cols, float eps, int8_t *out_q, float q_inv_scale) {
    TR_REQUIRE(rows >= 0 && cols >= 0, TNN_ROCM_ESHAPE, "layernorm: negative size");
    // the reference rejects an empty reduction (cpu_layer_norm_layer_acc.cc:87-90)
    TR_REQUIRE(rows > 0 && cols > 0, TNN_ROCM_ESHAPE, "layernorm: blob count is zero");
    TR_REQUIRE(x && y && gamma && beta, TNN_ROCM_EINVAL, "layernorm: null pointer");
    hipStream_t s = (hipStream_t)stream;
    switch (dtype) {
        case TNN_ROCM_F32:
            return launch_layernorm<TNN_ROCM_F32>(s, x, residual, gamma, beta, y, rows, cols, eps, out_q, q_inv_scale);
        case TNN_ROCM_F16:
            return launch_layernorm<TNN_ROCM_F16>(s, x, residual, gamma, beta, y, rows, cols, eps, out_q, q_inv_scale);
        case TNN_ROCM_BF16:
            return launch_layernorm<TNN_ROCM_BF16>(s, x, residual, gamma, beta, y, rows, cols, eps, out_q,
                                                   q_inv_scale);
        default: set_error("layernorm: unsupported dtype %d", dtype); return TNN_ROCM_EDTYPE;
    }
}

static int embed_layernorm_impl(void *stream, int dtype, const int32_t *ids, const int32_t *type_ids, const void *word_table,
                                int vocab, const void *type_table, int n_types, const void *pos_table, int period,
                                const int32_t *pos_ids, int n_pos_ids, int pos_rows, const float *gamma, const float *beta,
                                float eps, void *y, int rows, int cols, int32_t *error_flag);

int tnn_rocm_embed_layernorm(void *stream, int dtype, const int32_t *ids, const int32_t *type_ids, const void *word_table,
                             int vocab, const void *type_table, int n_types, const void *pos_table, int period,
                             const float *gamma, const float *beta, float eps, void *y, int rows, int cols,
                             int32_t *error_flag) {
    return embed_layernorm_impl(stream, dtype, ids, type_ids, word_table, vocab, type_table, n_types, pos_table, period,
                                nullptr, 0, 0, gamma, beta, eps, y, rows, cols, error_flag);
}

int tnn_rocm_embed_layernorm_pos(void *stream, int dtype, const int32_t *ids, const int32_t *type_ids,
                                 const int32_t *pos_ids, int n_pos_ids, const void *word_table, int vocab,
                                 const void *type_table, int n_types, const void *pos_table, int pos_rows,
                                 const float *gamma, const float *beta, float eps, void *y, int rows, int cols,
                                 int32_t *error_flag) {
    TR_REQUIRE(pos_ids && n_pos_ids > 0 && pos_rows > 0, TNN_ROCM_EINVAL, "embed_layernorm_pos: position ids and table rows required");
    return embed_layernorm_impl(stream, dtype, ids, type_ids, word_table, vocab, type_table, n_types, pos_table, 1, pos_ids,
                                n_pos_ids, pos_rows, gamma, beta, eps, y, rows, cols, error_flag);
}

static int embed_layernorm_impl(void *stream, int dtype, const int32_t *ids, const int32_t *type_ids, const void *word_table,
                                int vocab, const void *type_table, int n_types, const void *pos_table, int period,
                                const int32_t *pos_ids, int n_pos_ids, int pos_rows, const float *gamma, const float *beta,
                                float eps, void *y, int rows, int cols, int32_t *error_flag) {
    TR_REQUIRE(rows >= 0 && cols > 0 && vocab > 0 && n_types > 0 && period > 0, TNN_ROCM_ESHAPE,
               "embed_layernorm: sizes must be positive");
    if (rows == 0)
        return 0;
    TR_REQUIRE(ids && type_ids && word_table && type_table && pos_table && gamma && beta && y, TNN_ROCM_EINVAL,
               "embed_layernorm: null pointer");
    EmbedRows emb;
    emb.pos_ids   = pos_ids;
    emb.n_pos_ids = n_pos_ids;
    emb.pos_rows  = pos_rows;
    emb.ids        = ids;
    emb.type_ids   = type_ids;
    emb.type_table = type_table;
    emb.vocab      = vocab;
    emb.n_types    = n_types;
    emb.period     = period;
    emb.error_flag = error_flag;
    hipStream_t s  = (hipStream_t)stream;
    switch (dtype) {
        case TNN_ROCM_F32:
            return launch_layernorm<TNN_ROCM_F32>(s, word_table, pos_table, gamma, beta, y, rows, cols, eps, nullptr, 0.f, emb);
        case TNN_ROCM_F16:
            return launch_layernorm<TNN_ROCM_F16>(s, word_table, pos_table, gamma, beta, y, rows, cols, eps, nullptr, 0.f, emb);
        case TNN_ROCM_BF16:
            return launch_layernorm<TNN_ROCM_BF16>(s, word_table, pos_table, gamma, beta, y, rows, cols, eps, nullptr, 0.f, emb);
        default: set_error("embed_layernorm: unsupported dtype %d", dtype); return TNN_ROCM_EDTYPE;
    }
}

int tnn_rocm_softmax(void *stream, int dtype, const void *x, void *y, int outer, int channel, int inner) {
    TR_REQUIRE(outer >= 0 && channel >= 0 && inner >= 0, TNN_ROCM_ESHAPE, "softmax: negative size");
    if (outer == 0 || channel == 0 || inner == 0)
        return 0;
    TR_REQUIRE(x && y, TNN_ROCM_EINVAL, "softmax: null pointer");
    hipStream_t s = (hipStream_t)stream;
    switch (dtype) {
        case TNN_ROCM_F32: return launch_softmax<TNN_ROCM_F32>(s, x, y, outer, channel, inner);
        case TNN_ROCM_F16: return launch_softmax<TNN_ROCM_F16>(s, x, y, outer, channel, inner);
        case TNN_ROCM_BF16: return launch_softmax<TNN_ROCM_BF16>(s, x, y, outer, channel, inner);
        default: set_error("softmax: unsupported dtype %d", dtype); return TNN_ROCM_EDTYPE;
    }
}

}  // extern "C"
