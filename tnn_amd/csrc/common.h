// Shared helpers for the gfx950 kernels: error plumbing, dtype traits, wavefront reductions.
#ifndef TNN_ROCM_CSRC_COMMON_H_
#define TNN_ROCM_CSRC_COMMON_H_

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#include <atomic>
#include <type_traits>

#include "tnn_rocm.h"

namespace tnn_rocm {

constexpr int kWave = 64;  // CDNA wavefront width

void set_error(const char *fmt, ...);

#define TR_CHECK_HIP(expr)                                                                     \
    do {                                                                                       \
        hipError_t _e = (expr);                                                                \
        if (_e != hipSuccess) {                                                                \
            ::tnn_rocm::set_error("%s failed: %s (%s:%d)", #expr, hipGetErrorString(_e),       \
                                  __FILE__, __LINE__);                                         \
            return (int)_e;                                                                    \
        }                                                                                      \
    } while (0)

#define TR_REQUIRE(cond, code, ...)                                                            \
    do {                                                                                       \
        if (!(cond)) {                                                                         \
            ::tnn_rocm::set_error(__VA_ARGS__);                                                \
            return (code);                                                                     \
        }                                                                                      \
    } while (0)

// Launch check: reports configuration errors of the launch just issued.
#define TR_CHECK_LAUNCH() TR_CHECK_HIP(hipGetLastError())

typedef _Float16 half_t;
typedef uint16_t bf16_bits;

__device__ __forceinline__ float bf16_to_float(bf16_bits v) {
    return __uint_as_float(((uint32_t)v) << 16);
}
// round to nearest even, a NaN stays a (quiet) NaN: v_cvt_pk_bf16_f32, where the integer sequence for it takes six instructions
__device__ __forceinline__ bf16_bits float_to_bf16(float f) { return __builtin_bit_cast(bf16_bits, (__bf16)f); }
__device__ __forceinline__ uint32_t floats_to_bf16_pair(float lo, float hi) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2{lo, hi}), b2));
}

// Element load/store as float for the three floating dtypes.
// ---- result stores --------------------------------------------------------------------------------------------------
// When a kernel ends, the dirty lines of the eight L2s are written back before the next kernel of the stream may start
// (the L2s are not coherent with each other, so this is what makes one kernel's results visible to the next).  A GEMM
// that leaves 18 MB of results dirty pays about 1.8 us for that between its last instruction and its successor's first.
// Stores issued at device scope (sc1) go through the L2 to the memory side as they are made, under the kernel's own
// remaining work, and leave nothing to write back; they still allocate in the memory-side cache, where the consumer
// finds them (stores with the non-temporal hint do not, which costs the consumer more than the write-back saved).
// The compiler has no spelling for a 16-byte store at device scope, hence the assembly; a store of more than 8 bytes
// needs two wait states before its data registers may be overwritten, which the hazard recognizer cannot see through
// an asm statement, so they are part of it.  No memory clobber: nothing in these kernels reads what they store.
// Whether they do is a kernel argument (StoreThrough, set by tnn_rocm_debug_set_store_through for A/B runs): as a variable in
// device memory the switch cost every kernel two dependent scalar loads of cold lines in front of its first store, 0.2 us.
typedef unsigned int store_u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int store_u32x2 __attribute__((ext_vector_type(2)));
inline std::atomic<int> g_store_through{1};
struct StoreThrough {
    int through = g_store_through.load(std::memory_order_relaxed);
};

__device__ __forceinline__ void store_out16(int through, void *p, store_u32x4 v) {
    if (through)
        asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" ::"v"(p), "v"(v));
    else
        *reinterpret_cast<store_u32x4 *>(p) = v;
}
__device__ __forceinline__ void store_out8(int through, void *p, store_u32x2 v) {
    if (through)
        asm volatile("global_store_dwordx2 %0, %1, off sc1" ::"v"(p), "v"(v));
    else
        *reinterpret_cast<store_u32x2 *>(p) = v;
}
__device__ __forceinline__ void store_out8(int through, float2 *p, float2 v) {
    store_out8(through, (void *)p, store_u32x2{__float_as_uint(v.x), __float_as_uint(v.y)});
}
__device__ __forceinline__ void store_out4(int through, void *p, uint32_t v) {
    if (through)
        asm volatile("global_store_dword %0, %1, off sc1" ::"v"(p), "v"(v));
    else
        *reinterpret_cast<uint32_t *>(p) = v;
}
__device__ __forceinline__ void store_out2(int through, void *p, uint16_t v) {
    if (through)
        asm volatile("global_store_short %0, %1, off sc1" ::"v"(p), "v"((uint32_t)v));
    else
        *reinterpret_cast<uint16_t *>(p) = v;
}

template <int DT> struct Elem;
template <> struct Elem<TNN_ROCM_F32> {
    typedef float type;
    static __device__ __forceinline__ float ld(const float *p) { return *p; }
    static __device__ __forceinline__ void st(float *p, float v) { *p = v; }
    static __device__ __forceinline__ void st_out(int through, float *p, float v) { store_out4(through, p, __float_as_uint(v)); }
};
template <> struct Elem<TNN_ROCM_F16> {
    typedef half_t type;
    static __device__ __forceinline__ float ld(const half_t *p) { return (float)*p; }
    static __device__ __forceinline__ void st(half_t *p, float v) { *p = (half_t)v; }
    static __device__ __forceinline__ void st_out(int through, half_t *p, float v) {
        const half_t h = (half_t)v;
        store_out2(through, p, *reinterpret_cast<const uint16_t *>(&h));
    }
};
template <> struct Elem<TNN_ROCM_BF16> {
    typedef bf16_bits type;
    static __device__ __forceinline__ float ld(const bf16_bits *p) { return bf16_to_float(*p); }
    static __device__ __forceinline__ void st(bf16_bits *p, float v) { *p = float_to_bf16(v); }
    static __device__ __forceinline__ void st_out(int through, bf16_bits *p, float v) { store_out2(through, p, float_to_bf16(v)); }
};

// Round half away from zero exactly as the reference's float2int8: add +-0.5f in fp32 (one
// rounding), clamp in fp32, truncate.  The translation units are compiled with -ffp-contract=off
// so the add is never fused with the multiply that produced v.
// (+-0.5 taken from the sign bit and the clamp as one med3 give the same result for every value that is not a NaN --
// -0.0 lands on 0 either way -- in three instructions instead of seven.  A NaN comes out as -128: the median of three
// with a NaN operand is the minimum of the other two, and -128 is also what the reference's x86 path makes of a NaN,
// whose truncating conversion yields INT_MIN before the saturating pack, x86_compute_int8.cc:31-39.)
__device__ __forceinline__ int8_t float2int8_ref(float v) {
    float t = __fadd_rn(v, __builtin_copysignf(0.5f, v));
    t       = __builtin_amdgcn_fmed3f(t, -128.0f, 127.0f);
    return (int8_t)(int)t;
}

// erf GELU for fp32 results, evaluated as the reference's CPU path compiles (cpu_gelu_layer_acc.cc:42-45 includes
// only <cmath>, so its unqualified erf is the double one): x*0.7071f and 0.5f*x are fp32 products, erf, the +1 and the
// final product are double, and the store rounds once to fp32.  erff would differ in the last ulp, which is enough
// to move a value across a rounding boundary of a quantiser that follows.
__device__ __forceinline__ float gelu_erf(float x) {
    const float hv = __fmul_rn(0.5f, x);
    const double e = erf((double)__fmul_rn(x, 0.707106793288165f)) + 1.0;
    return (float)((double)hv * e);
}

// erf GELU for results that are rounded to fp16/bf16.  With a = |x| and Phi(-a) = erfc(a/sqrt2)/2:
// gelu(x) = x*Phi(x) = max(x, 0) - a*Phi(-a) for either sign (no cancellation in the negative tail).
// -log2(Phi(-a)) is smooth and nearly quadratic, so Phi(-a) = exp2(-q(a)) with a degree-6 polynomial q, q(0) = 1
// (minimax fit of the relative error on [0, 9]: 2e-5, i.e. 3e-6 absolute in a*Phi(-a); beyond 9 the term is below
// 1e-18 and a is clamped so the polynomial stays inside its fitted range).  Six fused multiply-adds, one clamp, one
// exp2, one max and the final multiply-add: 13 issue slots against 19 for the rational form 7.1.26 of Abramowitz &
// Stegun used before and ~40 for erff.  Against the correctly rounded fp16 result 0.4 % of the values differ, by one
// ulp (2.8 % for the rational form).  fp32 products take gelu_erf_wide below, the fp32 layer gelu_erf above.
// max(x, 0) is formed as x/2 + |x/2|: exact for every finite x above twice the smallest normal value (halving and the sum of
// equal or opposite halves do not round there), and unlike the maximum instruction, which returns its other operand for a
// NaN, it hands a NaN through, as the reference's GELU does (and gives NaN for -inf, where the reference's 0.5 x (erf + 1) is
// -inf times 0).  An overflow upstream therefore stays visible in the output instead of turning into zeros.
__device__ __forceinline__ float max_with_zero(float x) {
    const float h = __fmul_rn(0.5f, x);
    return __fadd_rn(h, fabsf(h));
}

__device__ __forceinline__ float gelu_erf_fast(float x) {
    // med3 instead of fmin / fmax: one instruction each, where the minimum / maximum forms first quiet their operand
    const float a = __builtin_amdgcn_fmed3f(fabsf(x), 0.f, 9.0f);
    float q       = -2.8009472064e-05f;
    q             = fmaf(q, a, 6.8930927528e-04f);
    q             = fmaf(q, a, -7.6513012845e-03f);
    q             = fmaf(q, a, 5.2408451099e-02f);
    q             = fmaf(q, a, 4.5977897954e-01f);
    q             = fmaf(q, a, 1.1508630942e+00f);
    q             = fmaf(q, a, 1.0f);
    const float e = __builtin_amdgcn_exp2f(-q);  // Phi(-a)
    // the clamped a: a*Phi(-a) is below 1e-18 past 9, and +inf stays +inf
    return fmaf(-a, e, max_with_zero(x));
}

// The same function for fp32 results, without the double erf's branches and range reductions: Phi(-a) = 2^-q(a) as above, q as a
// polynomial of degree 16 in a/4.5 - 1 (minimax fit on [0, 9], 2e-9 relative in Phi up to a = 4, growing as a^2 / 16 beyond,
// where an ulp of x moves Phi by more), 2^f on [-1/2, 1/2] of degree 7 (4e-11), all in double: within 0.57 ulp of
// the exact value for |x| < 6 (260 000 points) (gelu_erf: 45 ulp, its x * 0.7071f is rounded to fp32).  31 instructions and no branch; in the
// GEMM epilogue of [1536,768] x [768,3072] GELU took 30 of 82 us with gelu_erf and takes 5 with this.  The stand-alone layer and
// the int8 tables keep gelu_erf: what they write may go into a quantiser that has to meet the reference's bits.
__device__ __forceinline__ float gelu_erf_wide(float x) {
    const float a  = __builtin_amdgcn_fmed3f(fabsf(x), 0.f, 9.0f);
    const double u = fma((double)a, 1.0 / 4.5, -1.0);
    double q      = -0.00029480396093531765;
    q             = fma(q, u, -0.0002237530950128007);
    q             = fma(q, u, 0.0018946046748763853);
    q             = fma(q, u, -0.0008031934073889893);
    q             = fma(q, u, -0.0016600184100701802);
    q             = fma(q, u, 0.0004907614109894859);
    q             = fma(q, u, -0.0002371595308020806);
    q             = fma(q, u, 0.005366156345686441);
    q             = fma(q, u, -0.01374846949674306);
    q             = fma(q, u, 0.027259356200940412);
    q             = fma(q, u, -0.05217673527433646);
    q             = fma(q, u, 0.09565246244411721);
    q             = fma(q, u, -0.17006105027347934);
    q             = fma(q, u, 0.3022702751305858);
    q             = fma(q, u, 14.040319310540893);
    q             = fma(q, u, 30.54104511153);
    q             = fma(q, u, 18.167021500535277);
    const double n = rint(q), f = n - q;
    double e      = 1.520191909887254e-05;
    e             = fma(e, f, 0.0001546929118398554);
    e             = fma(e, f, 0.0013333922575706968);
    e             = fma(e, f, 0.009618027253502241);
    e             = fma(e, f, 0.055504103534314266);
    e             = fma(e, f, 0.24022651198159448);
    e             = fma(e, f, 0.6931471807284522);
    e             = fma(e, f, 0.9999999999616818);
    const double h = 0.5 * (double)x;  // max(x, 0) as above, in double: there half of the smallest floats is exact too
    return (float)fma(-(double)a, ldexp(e, -(int)n), h + fabs(h));
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        v += __shfl_xor(v, o, 64);
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}

// v plus the v of lane ^ O, for O = 32, 16, 8, 4, 2, 1 in turn (from 4 on down the lanes of a row that differ in higher bits
// hold the same value already, so that a rotation serves): register moves between lanes, where a shuffle goes through LDS at
// some hundred clocks
template <int O> __device__ __forceinline__ double add_lane_xor(double v) {
    typedef uint32_t pair __attribute__((ext_vector_type(2)));
    const pair u = __builtin_bit_cast(pair, v);
    if constexpr (O >= 16) {
        const auto lo = O == 32 ? __builtin_amdgcn_permlane32_swap(u.x, u.x, false, false) : __builtin_amdgcn_permlane16_swap(u.x, u.x, false, false);
        const auto hi = O == 32 ? __builtin_amdgcn_permlane32_swap(u.y, u.y, false, false) : __builtin_amdgcn_permlane16_swap(u.y, u.y, false, false);
        return __builtin_bit_cast(double, pair{lo[0], hi[0]}) + __builtin_bit_cast(double, pair{lo[1], hi[1]});
    } else {
        constexpr int CTRL = O == 8 ? 0x128 : O == 4 ? 0x124 : O == 2 ? 0x4E : 0xB1;  // row_ror:8, row_ror:4, quad_perm
        const pair w = {(uint32_t)__builtin_amdgcn_update_dpp(0, (int)u.x, CTRL, 0xf, 0xf, false),
                        (uint32_t)__builtin_amdgcn_update_dpp(0, (int)u.y, CTRL, 0xf, 0xf, false)};
        return v + __builtin_bit_cast(double, w);
    }
}

// the v of another lane of the same eight, by a DPP control word
template <int CTRL> __device__ __forceinline__ float lane_of_eight(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
template <int CTRL> __device__ __forceinline__ double lane_of_eight(double v) {
    typedef float pair __attribute__((ext_vector_type(2)));
    const pair u = __builtin_bit_cast(pair, v);
    return __builtin_bit_cast(double, pair{lane_of_eight<CTRL>(u.x), lane_of_eight<CTRL>(u.y)});
}

// the sum over N = 2, 4 or 8 neighbouring lanes, in every one of them
template <int N, typename V> __device__ __forceinline__ V add_neighbours(V v) {
    v = v + lane_of_eight<0xB1>(v);  // quad_perm: lane ^ 1
    if constexpr (N >= 4)
        v = v + lane_of_eight<0x4E>(v);  // quad_perm: lane ^ 2
    if constexpr (N >= 8)
        v = v + lane_of_eight<0x141>(v);  // row_half_mirror: the other four of eight
    return v;
}

// 1 / sqrt(v), of zero, infinities and NaN too: the instruction's estimate (2^-26) and two Newton steps, the second with the exact
// rest of v r, so that the result is the rounded root nearly everywhere (over 4 million values from 1e-12 to 1e8 0.5005 ulp at most;
// 1.0 / sqrt(v) 1.48, one step 19.9) in nine double instructions.
__device__ __forceinline__ double reciprocal_root(double v) {
    const double e = __builtin_amdgcn_rsq(v);
    const double r = fma(0.5 * e, fma(-v * e, e, 1.0), e);
    const double h = v * r, rest = fma(v, r, -h);
    const double root = fma(0.5 * r, fma(-rest, r, fma(-h, r, 1.0)), r);
    return e > 0.0 && e < (double)INFINITY ? root : e;
}

constexpr int kNumCU = 256;  // compute units of the chip, in eight XCDs

// A kernel's arguments lie in cache lines that nothing on the chip has read yet.  The compiler loads them as it comes to them,
// one miss after the other (1700 clocks to a GEMM's first slab request, with five lines); touched together they cost one.
// request_kernel_args only asks for them: the wait is where the caller uses the result.
template <size_t BYTES> __device__ __forceinline__ uint32_t request_kernel_args() {
    typedef const __attribute__((address_space(4))) uint32_t *KernArg;
    const KernArg args = (KernArg)__builtin_amdgcn_kernarg_segment_ptr();
    uint32_t touched   = 0;
#pragma unroll
    for (int w = 0; w < (int)(BYTES / 4); w += 16)
        touched |= args[w];
    return touched;
}
template <size_t BYTES> __device__ __forceinline__ void touch_kernel_args() {
    asm volatile("" ::"s"(request_kernel_args<BYTES>()));
}

// Division by a number the host knows, as a product: three scalar instructions where the compiler's sequence for an unknown
// divisor takes some forty dependent ones, in front of everything else a workgroup does.  With s = ceil(log2 d) and
// magic = ceil(2^(31+s) / d) the quotient is exact for every n below 2^31.
struct FixedDivisor {
    uint32_t magic, shift;
    __device__ __forceinline__ int quotient(int n) const { return (int)(((uint64_t)(uint32_t)n * magic) >> shift); }
    static FixedDivisor of(uint32_t d) {
        uint32_t s = 0;
        d          = d < 1 ? 1 : d;
        while ((1ull << s) < d)
            ++s;
        return {(uint32_t)(((1ull << (31 + s)) + d - 1) / d), 31 + s};
    }
};
static inline bool is_float_dtype(int dt) {
    return dt == TNN_ROCM_F32 || dt == TNN_ROCM_F16 || dt == TNN_ROCM_BF16;
}
static inline size_t dtype_bytes(int dt) {
    switch (dt) {
        case TNN_ROCM_F32: return 4;
        case TNN_ROCM_F16: return 2;
        case TNN_ROCM_I8: return 1;
        case TNN_ROCM_I32: return 4;
        case TNN_ROCM_BF16: return 2;
        default: return 0;
    }
}

}  // namespace tnn_rocm
#endif
