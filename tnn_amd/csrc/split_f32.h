// fp32 products on the bf16 matrix cores.
//
// An fp32 value has 24 significant bits, a bfloat16 eight of its own and the same exponent range, so a value is exactly the
// sum of three of them: x = x1 + x2 + x3 with x1 = bf16(x), x2 = bf16(x - x1), x3 = bf16(x - x1 - x2), each rounded to
// nearest (both differences are exact in fp32), as long as x3's last place is one that bfloat16 has.  Below 2^-109 it has not
// (its smallest step is 2^-133), so the planes are those of 2^24 x: exact for every x down to the smallest there is, and a
// sum of products comes out 2^48 times too large, which its reader takes back.  What the factor costs at the other end shows:
// x from 2^104 on, or a sum from 2^80 on, gives an infinity or a NaN, as an operand that is infinite or NaN does; the readers
// look for those and form such a sum again with the fp32 matrix instruction.  The multiplication makes 4.5 instructions per
// value of 3.5; most go into issue slots that the matrix instructions leave (fp32 request of 4 x 384 tokens, 2887 us without,
// 2901 with).  A product is then the sum of nine bf16 products, each exact in the fp32 accumulator; the six down to x1*y3 /
// x2*y2 / x3*y1 are formed.  The three left out are below 2^-26 |x y| together, a quarter of the rounding error that an fp32
// product itself carries.  (The scheme is that of Henry, Tang and Heinecke,
// "Leveraging the bfloat16 Artificial Intelligence Datatype For Higher-Precision Computations", ARITH 2019.)
//
// Why: the fp32 matrix instruction does 256 operations per CU and clock, the bf16 one 4096, i.e. 683 after six products.
// Sums over K are also rounded less often, once per 16 products instead of once per two.  Measured at kTilesF32 in
// gemm_kernels.h: up to 1.5 times the rate, a third to two thirds of the error against float64.
#ifndef TNN_ROCM_CSRC_SPLIT_F32_H_
#define TNN_ROCM_CSRC_SPLIT_F32_H_

#include <type_traits>

#include "common.h"

namespace tnn_rocm {

typedef __bf16 split_bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 split_bf16x8 __attribute__((ext_vector_type(8)));
typedef float split_f32x2 __attribute__((ext_vector_type(2)));
typedef float split_f32x4 __attribute__((ext_vector_type(4)));
typedef float split_f32x16 __attribute__((ext_vector_type(16)));

constexpr float kSplitScale   = 16777216.0f;                 // 2^24, of every operand
constexpr float kSplitUnscale = 1.0f / 281474976710656.0f;   // 2^-48, of every sum of products

// eight values of k of one row or column: one operand of v_mfma_f32_32x32x16_bf16 per plane
struct Split3 {
    uint32_t p[3][4];
};

// The residuals x - bf16(x) of a packed pair as dot products {lo, hi} . {-1, 0} + x and {lo, hi} . {0, -1} + y: one
// instruction each instead of two (7.4 against 9.3 clocks per value and level, measured), and exact, because the result is
// representable.  The two constants are held in registers: as an immediate the pair {-1, 0} becomes the inline constant
// -1.0, which this instruction does not read as that pair.
struct SplitConst {
    uint32_t lo, hi;
    __device__ __forceinline__ SplitConst() : lo(0x0000bf80u), hi(0xbf800000u) {
        asm("" : "+s"(lo));
        asm("" : "+s"(hi));
    }
};

__device__ __forceinline__ uint32_t split_pack(float x, float y) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((split_f32x2{x, y}), split_bf16x2));
}
__device__ __forceinline__ float split_rest(uint32_t pair, uint32_t minus_one, float x) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(split_bf16x2, pair), __builtin_bit_cast(split_bf16x2, minus_one), x, false);
}

__device__ __forceinline__ Split3 split3(const float (&x)[8], const SplitConst &c) {
    Split3 s;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float a = x[2 * i] * kSplitScale, b = x[2 * i + 1] * kSplitScale;
        s.p[0][i]      = split_pack(a, b);
        const float ra = split_rest(s.p[0][i], c.lo, a), rb = split_rest(s.p[0][i], c.hi, b);
        s.p[1][i]      = split_pack(ra, rb);
        s.p[2][i]      = split_pack(split_rest(s.p[1][i], c.lo, ra), split_rest(s.p[1][i], c.hi, rb));
    }
    return s;
}

// the planes of the six products, the smallest first
constexpr int kSplitProducts       = 6;
constexpr int kSplitOrder[6][2]    = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};

__device__ __forceinline__ void split_mma(const Split3 &a, const Split3 &b, int product, split_f32x16 &c) {
    const int pa = kSplitOrder[product][0], pb = kSplitOrder[product][1];  // constants once the caller's loop is unrolled
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const u32x4 va = {a.p[pa][0], a.p[pa][1], a.p[pa][2], a.p[pa][3]}, vb = {b.p[pb][0], b.p[pb][1], b.p[pb][2], b.p[pb][3]};
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(split_bf16x8, va), __builtin_bit_cast(split_bf16x8, vb), c,
                                                0, 0, 0);
}
__device__ __forceinline__ void split_mma(const Split3 &a, const Split3 &b, int product, split_f32x4 &c) {  // of 16 x 16 blocks
    const int pa = kSplitOrder[product][0], pb = kSplitOrder[product][1];
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const u32x4 va = {a.p[pa][0], a.p[pa][1], a.p[pa][2], a.p[pa][3]}, vb = {b.p[pb][0], b.p[pb][1], b.p[pb][2], b.p[pb][3]};
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(split_bf16x8, va), __builtin_bit_cast(split_bf16x8, vb), c, 0, 0, 0);
}

// is x, a value without sign, neither infinite nor a NaN?  On the bits: of a sum of magnitudes "< INFINITY" the compiler makes
// "!= INFINITY", which a NaN passes.
__device__ __forceinline__ bool split_finite(float x) { return (__float_as_uint(x) & 0x7fffffffu) < 0x7f800000u; }

}  // namespace tnn_rocm
#endif
