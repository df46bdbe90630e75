// MFMA GEMM for gfx950: C = A * op(B) with fused epilogues, for fp32 / fp16 / bf16 / int8 inputs.
//
// Tiling (64-wide wavefronts): a workgroup of WM x WN waves computes a BM x BN macro tile; each
// wave owns a (BM/WM) x (BN/WN) sub-tile made of 32x32 MFMA blocks.  Operand panels are staged
// through LDS in k-slabs of 64 bytes per row, double buffered: the global loads of slab k+1 are
// issued into registers before the MFMAs of slab k and written to the other LDS buffer afterwards,
// so one barrier per slab suffices.  Both LDS panels are stored "row x k" (k contiguous), which is
// the order the MFMA operands want: a lane supplies 16 contiguous bytes of k for one row/column.
//
//   fp16 : v_mfma_f32_32x32x16_f16   (8 halfs per lane per operand)
//   bf16 : v_mfma_f32_32x32x16_bf16
//   int8 : v_mfma_i32_32x32x32_i8    (16 bytes per lane per operand), exact int32 accumulation
//   fp32 : 4 x v_mfma_f32_32x32x2f32 per 16-byte operand read (general kernel and slabs staged through registers); the
//          direct-to-LDS kernels split every value into three bf16 planes, see split_f32.h
//
// The contraction index inside one MFMA is symmetric between the two operands, so any fixed
// assignment of k-values to (lane half, vector element) gives the same sum; both panels use the
// same one.
//
// Output layout of a 32x32 block: lane l holds column (l % 32); accumulator register r holds row
// 8*(r/4) + 4*(l/32) + (r%4).
#ifndef TNN_ROCM_CSRC_GEMM_KERNELS_H_
#define TNN_ROCM_CSRC_GEMM_KERNELS_H_

#include <type_traits>
#include <utility>

#include "gemm_typed.h"
#include "split_f32.h"

// Hook for scratch builds that include this file to time the tiled kernel from inside: TR_TL(i) marks point i of a
// workgroup's life (0 entry, 5 first slabs requested, 6 row sums added up, 1 first slab landed, 2 main loop done,
// 3 C stored, 4 kernel end).  The library itself compiles it to nothing.
#ifndef TR_TL
#define TR_TL(i)
#endif

namespace tnn_rocm {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int kSlabBytes  = 64;               // bytes of k per row per LDS slab
constexpr int kLdsStride  = kSlabBytes + 16;  // padded row stride in bytes (bank spread for b128 reads)

// FRAGS: 16-byte LDS reads per operand and step of the tiled kernel
template <int DT> struct GemmTraits;
template <> struct GemmTraits<TNN_ROCM_F16> {
    static constexpr int FRAGS = 1;
    typedef half_t elem;
    typedef f32x16 acc;
    typedef f32x4 acc_small;  // of a 16 x 16 block
    static __device__ __forceinline__ void mma(const uint4 &a, const uint4 &b, acc &c) {
        c = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                   0);
    }
    static __device__ __forceinline__ void mma(const uint4 &a, const uint4 &b, acc_small &c) {
        c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    }
};
template <> struct GemmTraits<TNN_ROCM_BF16> {
    static constexpr int FRAGS = 1;
    typedef bf16_bits elem;
    typedef f32x16 acc;
    typedef f32x4 acc_small;
    static __device__ __forceinline__ void mma(const uint4 &a, const uint4 &b, acc &c) {
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                    0, 0);
    }
    static __device__ __forceinline__ void mma(const uint4 &a, const uint4 &b, acc_small &c) {
        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    }
};
template <> struct GemmTraits<TNN_ROCM_I8> {
    static constexpr int FRAGS = 1;
    typedef int8_t elem;
    typedef i32x16 acc;
    typedef i32x4 acc_small;
    static __device__ __forceinline__ void mma(const uint4 &a, const uint4 &b, acc &c) {
        c = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, a), __builtin_bit_cast(i32x4, b), c, 0, 0,
                                                  0);
    }
    static __device__ __forceinline__ void mma(const uint4 &a, const uint4 &b, acc_small &c) {
        c = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, a), __builtin_bit_cast(i32x4, b), c, 0, 0, 0);
    }
};
template <> struct GemmTraits<TNN_ROCM_F32> {
    typedef float elem;
    typedef f32x16 acc;
    typedef f32x4 acc_small;
    // the tiled kernel: two reads make one 16-wide step of three bf16 planes (split_f32.h)
    static constexpr int FRAGS = 2;
    static __device__ __forceinline__ Split3 prepare(const uint4 (&f)[2], const SplitConst &c) {
        const float x[8] = {__uint_as_float(f[0].x), __uint_as_float(f[0].y), __uint_as_float(f[0].z), __uint_as_float(f[0].w),
                            __uint_as_float(f[1].x), __uint_as_float(f[1].y), __uint_as_float(f[1].z), __uint_as_float(f[1].w)};
        return split3(x, c);
    }
    // the general kernel: fp32 matrix instructions
    static __device__ __forceinline__ void mma(const uint4 &a, const uint4 &b, acc &c) {
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a.x), __uint_as_float(b.x), c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a.y), __uint_as_float(b.y), c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a.z), __uint_as_float(b.z), c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a.w), __uint_as_float(b.w), c, 0, 0, 0);
    }
    static __device__ __forceinline__ void mma(const uint4 &a, const uint4 &b, acc_small &c) {
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.x), __uint_as_float(b.x), c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.y), __uint_as_float(b.y), c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.z), __uint_as_float(b.z), c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.w), __uint_as_float(b.w), c, 0, 0, 0);
    }
};
// fp32, pipelined: the planes of the operands of the STEPS steps that a wave takes from one slab.  turn() multiplies one
// slab's planes while it makes the next one's from their LDS reads.  Of the conversion's 36 vector instructions per operand and step
// the 20 that scale and round go behind the matrix instructions, which leave the vector ALU free for about 28 of their 33 clocks (five
// of them fit).  The 16 dot products do not: one waits until the matrix instruction in front of it is done (33 clocks -> 52, every
// further one 5; a wave alone on its SIMD), so they stand together, twice in a turn, where only the first of each pays that.
// Spread over all slots with the others (as they were) a turn took the sum of both kinds: K slabs of 96 x 64 tiles 0.61 us (of 256
// bytes a row, 96 of them 49.7 us), now 0.55 (45.4), of 128 x 128 1.09 -> 0.96, of 192 x 96 1.21 -> 1.09.  A subtraction of the
// widened plane in place of a dot product would hide, but takes two instructions: 2 .. 3 % less for tiles of 3 x 3 blocks on few CUs,
// nothing with all of them at work, 5 .. 10 % more for smaller tiles.  Reading the next slab's values from LDS a turn ahead gave nothing.
// The order is pinned: left to itself the compiler issues the two kinds one after the other, with the wait states that a
// dot product's result needs standing empty.  With every CU at work the matrix pipe's power holds the clock near 1.6 GHz, which
// is then the bound; on few CUs the vector instructions are.
template <int TM, int TN, int STEPS> struct SplitSlab {
    static constexpr int OPS    = TM + TN;
    static constexpr int MFMAS  = STEPS * kSplitProducts * TM * TN;
    static constexpr int PAIRS  = STEPS * OPS * 4;  // of values
    Split3 op[STEPS][OPS];                           // A's operands, then B's
    struct Reads {
        uint4 f[STEPS][OPS][2];
    };

    __device__ __forceinline__ void convert(const Reads &rd, const SplitConst &sc) {
#pragma unroll
        for (int ks = 0; ks < STEPS; ++ks)
#pragma unroll
            for (int o = 0; o < OPS; ++o)
                op[ks][o] = GemmTraits<TNN_ROCM_F32>::prepare(rd.f[ks][o], sc);
    }
    template <typename Acc> __device__ __forceinline__ void mfma(int q, Acc (&acc)[TM][TN]) const {
        const int ks = q / (kSplitProducts * TM * TN), r = q % (kSplitProducts * TM * TN);
        const int product = r / (TM * TN), i = r % (TM * TN) / TN, j = r % TN;
        split_mma(op[ks][TM + j], op[ks][i], product, acc[i][j]);
    }
    template <typename Acc> __device__ __forceinline__ void multiply(Acc (&acc)[TM][TN]) const {
#pragma unroll
        for (int q = 0; q < MFMAS; ++q)
            mfma(q, acc);
    }
    // One level of a pair of values: scale and first plane, rest, second plane, rest, third plane
    static __device__ __forceinline__ void level(int pair_index, int l, SplitSlab &next, float (&rest)[STEPS][OPS][8], const SplitConst &sc) {
        const int ks = pair_index / (OPS * 4), o = pair_index / 4 % OPS, g = pair_index % 4;
        float &x = rest[ks][o][2 * g], &y = rest[ks][o][2 * g + 1];
        if (l == 0)
            x *= kSplitScale, y *= kSplitScale;
        uint32_t &pair = next.op[ks][o].p[l / 2][g];
        if (l % 2 == 0) {
            pair = split_pack(x, y);
        } else {
            x = split_rest(pair, sc.lo, x);
            y = split_rest(pair, sc.hi, y);
        }
    }
    // Multiplies this slab's planes while it makes the next one's, whose LDS reads are under way; load(k) requests the k-th of
    // LOADS loads of the slab after, as early as their place is free, one a slot: the next turn waits for them.
    // AFTER_READS: they go where the reads come from.
    // Levels 0, 2 and 4 go behind the matrix instructions, in proportion to their instructions (three, one and one a pair), levels 1
    // and 3 in one piece each behind the last slot of the level in front.
    template <int LOADS, bool AFTER_READS, typename Acc, typename Load>
    __device__ __forceinline__ void turn(const Reads &rd, SplitSlab &next, Acc (&acc)[TM][TN], const SplitConst &sc, Load load) const {
        constexpr int LEAD   = MFMAS >= 24 ? 4 : 2;  // the first matrix instructions alone: the LDS reads arrive meanwhile
        constexpr int SLOTS  = MFMAS - LEAD, SECOND = SLOTS >= 5 ? SLOTS / 5 : 1, FIRST = SLOTS - 2 * SECOND;
        constexpr int L0     = AFTER_READS ? LEAD : 0;
        constexpr int LSLOTS = LOADS > 0 && LOADS < MFMAS - L0 ? LOADS : MFMAS - L0;
        float rest[STEPS][OPS][8];
        each(std::make_integer_sequence<int, MFMAS>(), [&](auto slot) __attribute__((always_inline)) {
            constexpr int q = decltype(slot)::value, i = q - LEAD;
            mfma(q, acc);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (i == -1) {
#pragma unroll
                for (int ks = 0; ks < STEPS; ++ks)
#pragma unroll
                    for (int o = 0; o < OPS; ++o)
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            rest[ks][o][h * 4 + 0] = __uint_as_float(rd.f[ks][o][h].x);
                            rest[ks][o][h * 4 + 1] = __uint_as_float(rd.f[ks][o][h].y);
                            rest[ks][o][h * 4 + 2] = __uint_as_float(rd.f[ks][o][h].z);
                            rest[ks][o][h * 4 + 3] = __uint_as_float(rd.f[ks][o][h].w);
                        }
            }
            if constexpr (i >= 0) {  // this slot's level, and its share of the level's slots
                constexpr int l  = i < FIRST ? 0 : i < FIRST + SECOND ? 2 : 4;
                constexpr int at = i - (l == 0 ? 0 : l == 2 ? FIRST : FIRST + SECOND), of = l == 0 ? FIRST : SECOND;
#pragma unroll
                for (int k = PAIRS * at / of; k < PAIRS * (at + 1) / of; ++k)
                    level(k, l, next, rest, sc);
                if constexpr (l < 4 && at == of - 1) {
#pragma unroll
                    for (int k = 0; k < PAIRS; ++k)
                        level(k, l + 1, next, rest, sc);
                }
            }
            if constexpr (LOADS > 0 && q >= L0 && q < L0 + LSLOTS) {
                if (AFTER_READS && q == L0)
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
                for (int k = LOADS * (q - L0) / LSLOTS; k < LOADS * (q - L0 + 1) / LSLOTS; ++k)
                    load(k);
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    }
    // (the slots one by one as constants: the unroller gives up on a loop of this size)
    template <int... Q, typename F> static __device__ __forceinline__ void each(std::integer_sequence<int, Q...>, F f) {
        (f(std::integral_constant<int, Q>()), ...);
    }
};

// ---- epilogues ----------------------------------------------------------------------------------
// Optional abilities of an epilogue type, false where the type does not name them:
//   kEmitsRowSums  the epilogue's store8 returns the sum and the sum of squares of the eight values it stored, and the
//                  kernel leaves per tile column and row their totals over the tile's columns (LnResidualEpilogue)
//   kTakesRowSums  a LayerNorm-folding epilogue that is handed such sums by the kernel that produced its A operand,
//                  instead of taking them from the A fragments in the main loop
template <typename E, typename = void> struct EmitsRowSums : std::false_type {};
template <typename E> struct EmitsRowSums<E, typename std::enable_if<E::kEmitsRowSums>::type> : std::true_type {};
template <typename E, typename = void> struct TakesRowSums : std::false_type {};
template <typename E> struct TakesRowSums<E, typename std::enable_if<E::kTakesRowSums>::type> : std::true_type {};
//   kColArrays     the epilogue reads that many per-column float arrays (col_src(k, n)) in store8.  The tiled kernel
//                  copies the tile's columns of each into LDS once, after the main loop, and store8 takes them from
//                  there (cl[k * cs + j] for column j of the item): an item then waits for two LDS reads instead of
//                  for global loads that cannot be moved above the previous item's stores
//   kRowIn         likewise for one float2 per row (row_src(m)), handed to store8 by value
template <typename E, typename = void> struct ColArrays : std::integral_constant<int, 0> {};
template <typename E> struct ColArrays<E, typename std::enable_if<(E::kColArrays > 0)>::type> : std::integral_constant<int, E::kColArrays> {};
template <typename E, typename = void> struct RowIn : std::false_type {};
template <typename E> struct RowIn<E, typename std::enable_if<E::kRowIn>::type> : std::true_type {};
//   kAheadVecs     the epilogue reads that many 16-byte vectors of another matrix (a residual) per item: ahead_src(m, n) is
//                  where they are, or null.  A shape whose threads have one item each requests them before its first slab
template <typename E, typename = void> struct AheadVecs : std::integral_constant<int, 0> {};
template <typename E> struct AheadVecs<E, typename std::enable_if<(E::kAheadVecs > 0)>::type> : std::integral_constant<int, E::kAheadVecs> {};
//   wide_us()      what the epilogue adds to every round of 256 x 256 tiles, in the cost model's microseconds: its 128 values a thread
//                  stand behind the last product of a CU's only tile, and nothing covers them
template <typename E, typename = void> struct WideEpilogue {
    static float us(const E &) { return 0.f; }
};
template <typename E> struct WideEpilogue<E, std::void_t<decltype(std::declval<const E &>().wide_us())>> {
    static float us(const E &e) { return e.wide_us(); }
};
template <typename E, typename = void> struct SumBlocks : std::integral_constant<int, 1> {};
template <typename E> struct SumBlocks<E, typename std::enable_if<E::kTakesRowSums>::type> : std::integral_constant<int, E::kSumBlocks> {};  // tile columns of a producer a consumer can add up (at most 24: 768 columns of 32, 384 of 16)


// GELU of a product, in every kernel and at every column the same function of the sum
template <int DT> __device__ __forceinline__ float gelu_of_product(float v) {
    return DT == TNN_ROCM_F32 ? gelu_erf_wide(v) : gelu_erf_fast(v);
}

template <int DT> struct FloatEpilogue : StoreThrough {
    typedef typename Elem<DT>::type T;
    static constexpr bool kRowStats = false;
    int flags;
    const float *bias;
    const T *residual;
    long ldr;
    T *C;
    long ldc;
    long batch_stride_c;
    long batch_stride_r;
    float wide_us() const { return (flags & TNN_ROCM_EPI_GELU) ? 2.5f : 0.f; }
    __device__ __forceinline__ void set_batch(int b) {
        C += (size_t)b * batch_stride_c;
        if (residual)
            residual += (size_t)b * batch_stride_r;
    }
    __device__ __forceinline__ float col_const(int n) const { return (flags & TNN_ROCM_EPI_BIAS) ? bias[n] : 0.f; }
    __device__ __forceinline__ void store(int m, int n, float acc, float bias_n) const {
        float v = acc;
        if (flags & TNN_ROCM_EPI_BIAS)
            v = v + bias_n;
        if (flags & TNN_ROCM_EPI_GELU)
            v = gelu_of_product<DT>(v);
        if (flags & TNN_ROCM_EPI_RESIDUAL)
            v = v + Elem<DT>::ld(&residual[(size_t)m * ldr + n]);
        Elem<DT>::st(&C[(size_t)m * ldc + n], v);
    }
    // true: this workgroup's columns go to a transposed layout, so the epilogue hands out rows to consecutive lanes
    __device__ __forceinline__ bool direct(int) const { return false; }
    // eight consecutive columns n..n+7 of row m (n % 8 == 0, n + 7 < N, rows 16-byte aligned): whole 16-byte
    // (half) / 32-byte (fp32) pieces, so that the lanes of one row together write full cache lines
    static constexpr int kColArrays = 1;  // bias
    __device__ __forceinline__ float col_src(int, int n) const { return (flags & TNN_ROCM_EPI_BIAS) ? bias[n] : 0.f; }
    static constexpr int kAheadVecs = 8 * sizeof(T) / 16;
    __device__ __forceinline__ const void *ahead_src(int m, int n) const {
        return (flags & TNN_ROCM_EPI_RESIDUAL) ? residual + (size_t)m * ldr + n : nullptr;
    }
    // cl = the item's eight columns of the bias in LDS; ahead = the residual's vectors where they have been requested already
    __device__ __forceinline__ void store8(int m, int n, const float (&acc)[8], const float *cl, int, const u32x4 *ahead) const {
        float v[8];
#pragma unroll
        for (int t = 0; t < 8; ++t)
            v[t] = acc[t];
        if (flags & TNN_ROCM_EPI_BIAS) {
            float4 b0 = *reinterpret_cast<const float4 *>(cl), b1 = *reinterpret_cast<const float4 *>(cl + 4);
            v[0] += b0.x, v[1] += b0.y, v[2] += b0.z, v[3] += b0.w;
            v[4] += b1.x, v[5] += b1.y, v[6] += b1.z, v[7] += b1.w;
        }
        if (flags & TNN_ROCM_EPI_GELU) {
#pragma unroll
            for (int t = 0; t < 8; ++t)
                v[t] = gelu_of_product<DT>(v[t]);
        }
        constexpr int NV = 8 * sizeof(T) / 16;  // 16-byte vectors per eight elements
        u32x4 packed[NV];
        T *pe = reinterpret_cast<T *>(packed);
        if (flags & TNN_ROCM_EPI_RESIDUAL) {
            const u32x4 *rp = reinterpret_cast<const u32x4 *>(residual + (size_t)m * ldr + n);
#pragma unroll
            for (int q = 0; q < NV; ++q)
                packed[q] = ahead ? ahead[q] : rp[q];
#pragma unroll
            for (int t = 0; t < 8; ++t)
                v[t] += Elem<DT>::ld(&pe[t]);
        }
#pragma unroll
        for (int t = 0; t < 8; ++t)
            Elem<DT>::st(&pe[t], v[t]);
        u32x4 *cp = reinterpret_cast<u32x4 *>(C + (size_t)m * ldc + n);
#pragma unroll
        for (int q = 0; q < NV; ++q)
            store_out16(through, &cp[q], packed[q]);
    }
};

// Where key s goes inside its V^T row.  sh = 0: at s.  sh = 1: inside every group of 16 keys the blocks of four
// k4-7 and k8-11 change places ([k0-3 | k8-11 | k4-7 | k12-15]), the order in which the lane halves of the attention
// kernel hold a tile's probabilities, so that kernel feeds them to its second MFMA without exchanging registers.
__device__ __forceinline__ int key_slot(int s, int sh) { return (s & ~12) | ((s & 4) << sh) | ((s & 8) >> sh); }

// QKV projection epilogue: columns [0,2H) -> qk[T,2H]; columns [2H,3H) -> V^T[b][head][d][s]
template <int DT> struct QkvSplitEpilogue : StoreThrough {
    typedef typename Elem<DT>::type T;
    static constexpr bool kRowStats = false;
    const float *bias;
    T *qk;
    T *vt;
    int H, S, heads;
    int vt_sh;  // 0: V^T keys in natural order; 1: bits 2 and 3 of the key index change places (see key_slot)
    float wide_us() const { return 1.5f; }  // V^T
    __device__ __forceinline__ void set_batch(int) {}
    __device__ __forceinline__ float col_const(int n) const { return bias ? bias[n] : 0.f; }
    __device__ __forceinline__ void store(int m, int n, float acc, float bias_n) const {
        float v = acc + bias_n;
        if (n < 2 * H) {
            Elem<DT>::st(&qk[(size_t)m * 2 * H + n], v);
        } else {
            int c = n - 2 * H, b = m / S, s = key_slot(m - b * S, vt_sh);
            Elem<DT>::st(&vt[(((size_t)b * heads + (c >> 6)) * 64 + (c & 63)) * S + s], v);
        }
    }
    // the V^T columns are written with consecutive lanes along s; Q|K rows with consecutive lanes along the row
    __device__ __forceinline__ bool direct(int n0) const { return n0 >= 2 * H; }
    static constexpr int kColArrays = 1;  // bias
    __device__ __forceinline__ float col_src(int, int n) const { return bias ? bias[n] : 0.f; }
    __device__ __forceinline__ void store8(int m, int n, const float (&acc)[8], const float *cl, int, const u32x4 *) const {
        float v[8];
#pragma unroll
        for (int t = 0; t < 8; ++t)
            v[t] = acc[t];
        if (bias) {
            float4 b0 = *reinterpret_cast<const float4 *>(cl), b1 = *reinterpret_cast<const float4 *>(cl + 4);
            v[0] += b0.x, v[1] += b0.y, v[2] += b0.z, v[3] += b0.w;
            v[4] += b1.x, v[5] += b1.y, v[6] += b1.z, v[7] += b1.w;
        }
        if (n < 2 * H) {
            constexpr int NV = 8 * sizeof(T) / 16;
            u32x4 packed[NV];
            T *pe = reinterpret_cast<T *>(packed);
#pragma unroll
            for (int t = 0; t < 8; ++t)
                Elem<DT>::st(&pe[t], v[t]);
            u32x4 *cp = reinterpret_cast<u32x4 *>(qk + (size_t)m * 2 * H + n);
#pragma unroll
            for (int q = 0; q < NV; ++q)
                store_out16(through, &cp[q], packed[q]);
        } else {
            int c = n - 2 * H, b = m / S, s_ = key_slot(m - b * S, vt_sh);
            T *dst = vt + (((size_t)b * heads + (c >> 6)) * 64 + (c & 63)) * S + s_;
#pragma unroll
            for (int t = 0; t < 8; ++t)
                Elem<DT>::st_out(through, dst + (size_t)t * S, v[t]);
        }
    }
};

// ---- LayerNorm folded into the projection that reads it ------------------------------------------------------------
// y = LayerNorm(t) over the last axis (cpu_layer_norm_layer_acc.cc:86-135: per row mean and variance,
// (t - mean) * rstd * gamma + beta) followed by y W^T + b, as one GEMM on the raw t:
//     y W^T + b = rstd * (t W'^T - mean * colsum) + b',   W' = gamma (.) W,  colsum[n] = sum_k W'[n,k],  b' = b + W beta.
// K is the normalised width, so every workgroup streams whole rows of t through LDS anyway: the row sums and sums of
// squares are taken from the A fragments the waves already hold for the MFMAs (two dot2 instructions per four
// values), reduced over the workgroup after the main loop, and applied to the accumulators in the epilogue.
// Other readers of y (the residual additions) still need the tensor: the workgroup of tile column j writes
// y for the j-th share of the columns of its rows, so the LayerNorm launch disappears without y disappearing.
struct LnFold {
    double cols, inv_cols;      // K and 1 / K: rounded to fp32, 1 / 768 took 3e-8 of the squared mean off the variance
    float eps;
    const float *colsum;        // [N]
    const float *gamma, *beta;  // [K], for the y side output
    void *y;                    // [M, K] in the compute type, or nullptr
    int y_ahead;                // 1: the source vectors of y are requested under the epilogue (0 for experiments)
    float2 *stats;              // [M] {rstd, mean} for a later kernel that rebuilds LayerNorm(t) itself, or nullptr
    const float2 *row_sums;     // kTakesRowSums: [sum_blocks][M] {sum, sum of squares} over a block of columns of t
    int sum_blocks;
};

// Mean, and variance + eps, of a row from its sums.  K s2 - s1^2 is formed exactly before it is rounded, so that rows of little
// spread far from zero keep what the sums themselves know of their variance: with E[x^2] - mean^2 in double a row at 100 is off by
// 2e-12, twice the eps of the models.  The sums are made of fp32 parts and can leave it a hair below zero, where it is cut
// off.  A NaN stays one.
__device__ __forceinline__ double row_moments(const LnFold &ln, double s1, double s2, double *mean) {
    const double square = s1 * s1;
    const double spread = fma(ln.cols, s2, -square) - fma(s1, s1, -square);
    *mean = s1 * ln.inv_cols;
    return (spread < 0.0 ? 0.0 : spread * (ln.inv_cols * ln.inv_cols)) + (double)ln.eps;
}

// row sum and sum of squares of the eight values of an A fragment register quad
template <int DT> __device__ __forceinline__ void ln_accumulate(const uint4 &frag, float &s1, float &s2) {
    const uint32_t w[4] = {frag.x, frag.y, frag.z, frag.w};
    if constexpr (DT == TNN_ROCM_F16) {
        typedef _Float16 h2 __attribute__((ext_vector_type(2)));
        const h2 one = {(_Float16)1.0f, (_Float16)1.0f};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            h2 v = __builtin_bit_cast(h2, w[t]);
            s1   = __builtin_amdgcn_fdot2(v, one, s1, false);
            s2   = __builtin_amdgcn_fdot2(v, v, s2, false);
        }
    } else {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            float lo = __uint_as_float(w[t] << 16), hi = __uint_as_float(w[t] & 0xffff0000u);
            s1 += lo + hi;
            s2 = fmaf(lo, lo, fmaf(hi, hi, s2));
        }
    }
}

// Element offset of (row m, column n) in a row-major matrix of leading dimension ld, for the epilogues whose entry
// points have checked rows < 2^24, ld < 2^24 and rows * ld < 2^31: one full-rate 24-bit multiply where the 64-bit
// product m * ld costs two v_mul_lo_u32 and a v_mad_u64_u32 (quarter rate each) per item.
__device__ __forceinline__ unsigned elem_offset24(int m, unsigned ld, int n) {
    return __umul24((unsigned)m, ld) + (unsigned)n;
}

// SUMS: 0 = the statistics come from the A fragments; else the most row-sum blocks the kernel is handed (12 or 24: that
// many register pairs hold them while they are in flight)
template <int DT, int SUMS = 0> struct LnFloatEpilogue : StoreThrough {
    typedef typename Elem<DT>::type T;
    static constexpr bool kRowStats = true;
    static constexpr bool kTakesRowSums = SUMS > 0;
    static constexpr int kSumBlocks     = SUMS;
    int flags;
    const float *bias;  // b' (always present)
    const T *residual;
    T *C;
    long ldc;
    LnFold ln;
    float wide_us() const { return (flags & TNN_ROCM_EPI_GELU) ? 2.5f : 0.f; }
    __device__ __forceinline__ void set_batch(int) {}
    __device__ __forceinline__ float col_const(int) const { return 0.f; }
    __device__ __forceinline__ void store(int, int, float, float) const {}  // N % 8 == 0 is required at launch
    __device__ __forceinline__ bool direct(int) const { return false; }
    static constexpr int kColArrays = 2;  // colsum, b'
    __device__ __forceinline__ float col_src(int k, int n) const { return k == 0 ? ln.colsum[n] : bias[n]; }
    static constexpr int kAheadVecs = 8 * sizeof(T) / 16;
    __device__ __forceinline__ const void *ahead_src(int m, int n) const {
        return (flags & TNN_ROCM_EPI_RESIDUAL) ? residual + elem_offset24(m, (unsigned)ldc, n) : nullptr;
    }
    // st = {rstd, mean} of row m; cl = the item's eight columns of the two arrays in LDS, cs apart; ahead as in FloatEpilogue
    __device__ __forceinline__ void store8(int m, int n, const float (&acc)[8], float2 st, const float *cl, int cs,
                                           const u32x4 *ahead) const {
        float4 g0 = *reinterpret_cast<const float4 *>(cl), g1 = *reinterpret_cast<const float4 *>(cl + 4);
        float4 b0 = *reinterpret_cast<const float4 *>(cl + cs), b1 = *reinterpret_cast<const float4 *>(cl + cs + 4);
        const float g[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
        const float b[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
        float v[8];
#pragma unroll
        for (int t = 0; t < 8; ++t)
            v[t] = fmaf(st.x, fmaf(-st.y, g[t], acc[t]), b[t]);
        if (flags & TNN_ROCM_EPI_GELU) {
#pragma unroll
            for (int t = 0; t < 8; ++t)
                v[t] = gelu_of_product<DT>(v[t]);
        }
        // the two forms each end in their own conversion and store: joined behind the branch, the form without a
        // residual pays eight register copies per item for the join
        if (flags & TNN_ROCM_EPI_RESIDUAL) {
            constexpr int NV = 8 * sizeof(T) / 16;
            u32x4 packed[NV];
            const T *pe      = reinterpret_cast<const T *>(packed);
            const u32x4 *rp = reinterpret_cast<const u32x4 *>(residual + elem_offset24(m, (unsigned)ldc, n));
#pragma unroll
            for (int q = 0; q < NV; ++q)
                packed[q] = ahead ? ahead[q] : rp[q];
            float w[8];
#pragma unroll
            for (int t = 0; t < 8; ++t)
                w[t] = v[t] + Elem<DT>::ld(&pe[t]);
            convert_and_store(m, n, w);
        } else {
            convert_and_store(m, n, v);
        }
    }
    __device__ __forceinline__ void convert_and_store(int m, int n, const float (&v)[8]) const {
        constexpr int NV = 8 * sizeof(T) / 16;
        u32x4 packed[NV];
        T *pe = reinterpret_cast<T *>(packed);
#pragma unroll
        for (int t = 0; t < 8; ++t)
            Elem<DT>::st(&pe[t], v[t]);
        u32x4 *cp = reinterpret_cast<u32x4 *>(C + elem_offset24(m, (unsigned)ldc, n));
#pragma unroll
        for (int q = 0; q < NV; ++q)
            store_out16(through, &cp[q], packed[q]);
    }
};

// QKV projection of LayerNorm(t): QkvSplitEpilogue's layout with the folded-LayerNorm correction on the accumulators
template <int DT, int SUMS = 0> struct LnQkvSplitEpilogue : StoreThrough {
    typedef typename Elem<DT>::type T;
    static constexpr bool kRowStats = true;
    static constexpr bool kTakesRowSums = SUMS > 0;
    static constexpr int kSumBlocks     = SUMS;
    const float *bias;
    T *qk;
    T *vt;
    int H, S, heads;
    int vt_sh;  // 0: V^T keys in natural order; 1: bits 2 and 3 of the key index change places (see key_slot)
    LnFold ln;
    float wide_us() const { return 1.5f; }  // V^T
    __device__ __forceinline__ void set_batch(int) {}
    __device__ __forceinline__ float col_const(int) const { return 0.f; }
    __device__ __forceinline__ void store(int, int, float, float) const {}
    __device__ __forceinline__ bool direct(int n0) const { return n0 >= 2 * H; }
    static constexpr int kColArrays = 2;  // colsum, b'
    __device__ __forceinline__ float col_src(int k, int n) const { return k == 0 ? ln.colsum[n] : bias[n]; }
    __device__ __forceinline__ void store8(int m, int n, const float (&acc)[8], float2 st, const float *cl, int cs,
                                           const u32x4 *) const {
        float4 g0 = *reinterpret_cast<const float4 *>(cl), g1 = *reinterpret_cast<const float4 *>(cl + 4);
        float4 b0 = *reinterpret_cast<const float4 *>(cl + cs), b1 = *reinterpret_cast<const float4 *>(cl + cs + 4);
        const float g[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
        const float b[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
        float v[8];
#pragma unroll
        for (int t = 0; t < 8; ++t)
            v[t] = fmaf(st.x, fmaf(-st.y, g[t], acc[t]), b[t]);
        if (n < 2 * H) {
            constexpr int NV = 8 * sizeof(T) / 16;
            u32x4 packed[NV];
            T *pe = reinterpret_cast<T *>(packed);
#pragma unroll
            for (int t = 0; t < 8; ++t)
                Elem<DT>::st(&pe[t], v[t]);
            u32x4 *cp = reinterpret_cast<u32x4 *>(qk + elem_offset24(m, 2u * (unsigned)H, n));
#pragma unroll
            for (int q = 0; q < NV; ++q)
                store_out16(through, &cp[q], packed[q]);
        } else {
            // B * S * 3H < 2^31 is checked at launch: 32-bit offsets throughout
            int c = n - 2 * H, bb = m / S, s_ = key_slot(m - bb * S, vt_sh);
            T *dst = vt + (unsigned)(((bb * heads + (c >> 6)) * 64 + (c & 63)) * S + s_);
#pragma unroll
            for (int t = 0; t < 8; ++t)
                Elem<DT>::st_out(through, dst + (unsigned)(t * S), v[t]);
        }
    }
};

// Projection whose residual operand is LayerNorm(t) of a tensor whose row statistics an earlier kernel left behind
// (LnFold::stats): C = act(x W^T + b) + ((t - mean) * rstd * gamma + beta).  The normalised tensor is rebuilt from t in
// registers, in the LayerNorm kernel's half-precision form x * rstd * gamma + (beta - mean * rstd * gamma), and never
// stored.  N is the normalised width.
template <int DT, bool SUMS = false> struct LnResidualEpilogue : StoreThrough {
    typedef typename Elem<DT>::type T;
    static constexpr bool kRowStats = false;
    static constexpr bool kEmitsRowSums = SUMS;
    float2 *row_sums;  // kEmitsRowSums: [blocks of columns][M] {sum, sum of squares} of the stored values of C
    int flags;  // TNN_ROCM_EPI_BIAS, TNN_ROCM_EPI_GELU
    const float *bias;
    const T *t;                 // [M, N]
    const float2 *st;           // [M] {rstd, mean}
    const float *gamma, *beta;  // [N]
    T *C;
    long ldc;
    float wide_us() const { return (flags & TNN_ROCM_EPI_GELU) ? 2.5f : 0.f; }
    __device__ __forceinline__ void set_batch(int) {}
    __device__ __forceinline__ float col_const(int n) const { return (flags & TNN_ROCM_EPI_BIAS) ? bias[n] : 0.f; }
    __device__ __forceinline__ void store(int m, int n, float acc, float bias_n) const {
        float v = acc;
        if (flags & TNN_ROCM_EPI_BIAS)
            v = v + bias_n;
        if (flags & TNN_ROCM_EPI_GELU)
            v = gelu_of_product<DT>(v);
        const float2 s = st[m];
        const float mrs = s.y * s.x;
        v = v + (Elem<DT>::ld(&t[(size_t)m * ldc + n]) * s.x * gamma[n] + (beta[n] - mrs * gamma[n]));
        Elem<DT>::st(&C[(size_t)m * ldc + n], v);
    }
    __device__ __forceinline__ bool direct(int) const { return false; }
    static constexpr int kColArrays = 3;  // bias (zeros without one), gamma, beta
    static constexpr bool kRowIn    = true;  // {rstd, mean} of the rows of t
    __device__ __forceinline__ float col_src(int k, int n) const {
        return k == 0 ? ((flags & TNN_ROCM_EPI_BIAS) ? bias[n] : 0.f) : k == 1 ? gamma[n] : beta[n];
    }
    __device__ __forceinline__ float2 row_src(int m) const { return st[m]; }
    static constexpr int kAheadVecs = 1;
    __device__ __forceinline__ const void *ahead_src(int m, int n) const { return t + elem_offset24(m, (unsigned)ldc, n); }
    // cl = the item's eight columns of the three arrays in LDS, cs apart; s = {rstd, mean} of row m; ahead as in FloatEpilogue
    __device__ __forceinline__ float2 store8(int m, int n, const float (&acc)[8], const float *cl, int cs, float2 s,
                                             const u32x4 *ahead) const {
        static_assert(sizeof(T) == 2, "half-precision blobs only");
        const unsigned off = elem_offset24(m, (unsigned)ldc, n);
        u32x4 packed = ahead ? *ahead : *reinterpret_cast<const u32x4 *>(t + off);
        float v[8];
        {
            float4 b0 = *reinterpret_cast<const float4 *>(cl), b1 = *reinterpret_cast<const float4 *>(cl + 4);
            v[0] = acc[0] + b0.x, v[1] = acc[1] + b0.y, v[2] = acc[2] + b0.z, v[3] = acc[3] + b0.w;
            v[4] = acc[4] + b1.x, v[5] = acc[5] + b1.y, v[6] = acc[6] + b1.z, v[7] = acc[7] + b1.w;
        }
        if (flags & TNN_ROCM_EPI_GELU) {
#pragma unroll
            for (int q = 0; q < 8; ++q)
                v[q] = gelu_of_product<DT>(v[q]);
        }
        T *pe = reinterpret_cast<T *>(&packed);
        const float mrs = s.y * s.x;
        float4 k0 = *reinterpret_cast<const float4 *>(cl + cs), k1 = *reinterpret_cast<const float4 *>(cl + cs + 4);
        float4 e0 = *reinterpret_cast<const float4 *>(cl + 2 * cs), e1 = *reinterpret_cast<const float4 *>(cl + 2 * cs + 4);
        const float kk[8] = {k0.x, k0.y, k0.z, k0.w, k1.x, k1.y, k1.z, k1.w};
        const float ee[8] = {e0.x, e0.y, e0.z, e0.w, e1.x, e1.y, e1.z, e1.w};
#pragma unroll
        for (int q = 0; q < 8; ++q)
            v[q] += Elem<DT>::ld(&pe[q]) * s.x * kk[q] + (ee[q] - mrs * kk[q]);
#pragma unroll
        for (int q = 0; q < 8; ++q)
            Elem<DT>::st(&pe[q], v[q]);
        store_out16(through, C + off, packed);
        float2 sums = make_float2(0.f, 0.f);
        if constexpr (SUMS) {  // of the values as stored (rounded to the blob type): what the next GEMM reads
            ln_accumulate<DT>(__builtin_bit_cast(uint4, packed), sums.x, sums.y);
        }
        return sums;
    }
};

struct Int8Epilogue : StoreThrough {
    static constexpr bool kRowStats = false;
    // optional 256-entry table applied to the requantised value (index q + 128): an int8 -> int8 function that
    // followed the layer (dequantise, GELU, quantise) folded into this epilogue.  The tiled kernel keeps a copy in LDS.
    const int8_t *lut;
    const int32_t *bias;
    const float *scale;
    int8_t *out;
    int32_t *acc_out;
    long ldo;
    void *out_f;
    int out_f_dtype;
    float dq;
    const void *residual;  // optional, type and leading dimension of out_f: out_f = q * dq + residual
    __device__ __forceinline__ void set_batch(int) {}
    struct ColConst {
        int32_t bias;
        float scale;
    };
    __device__ __forceinline__ ColConst col_const(int n) const {
        ColConst c;
        c.bias  = bias ? bias[n] : 0;
        c.scale = scale ? scale[n] : 0.f;
        return c;
    }
    __device__ __forceinline__ void store(int m, int n, int acc, const ColConst &cc) const {
        int a = acc + cc.bias;
        if (acc_out)
            acc_out[(size_t)m * ldo + n] = a;
        if (out || out_f) {
            // (float)int32 rounds to nearest even, one fp32 multiply, then the +-0.5 add: three
            // separately rounded steps as on the CPU paths.
            float f  = __fmul_rn((float)a, cc.scale);
            int8_t q = float2int8_ref(f);
            if (lut)
                q = lut[(int)q + 128];
            if (out)
                out[(size_t)m * ldo + n] = q;
            if (out_f) {
                float d = __fmul_rn((float)q, dq);
                if (out_f_dtype == TNN_ROCM_F32) {
                    if (residual)
                        d = __fadd_rn(d, ((const float *)residual)[(size_t)m * ldo + n]);
                    ((float *)out_f)[(size_t)m * ldo + n] = d;
                } else {
                    if (residual)
                        d = __fadd_rn(d, (float)((const half_t *)residual)[(size_t)m * ldo + n]);
                    ((half_t *)out_f)[(size_t)m * ldo + n] = (half_t)d;
                }
            }
        }
    }
    __device__ __forceinline__ bool direct(int) const { return false; }
    // eight consecutive columns (n % 8 == 0, n + 7 < N, ldo % 8 == 0): same arithmetic as store(), vector accesses
    static constexpr int kColArrays = 2;  // bias (its int32 bits), scale
    __device__ __forceinline__ float col_src(int k, int n) const {
        return k == 0 ? (bias ? __int_as_float(bias[n]) : 0.f) : (scale ? scale[n] : 0.f);
    }
    static constexpr int kAheadVecs = 1;  // a half residual; an fp32 one is read in its place
    __device__ __forceinline__ const void *ahead_src(int m, int n) const {
        return out_f && residual && out_f_dtype != TNN_ROCM_F32 ? (const half_t *)residual + (size_t)m * ldo + n : nullptr;
    }
    // cl = the item's eight columns of the two arrays in LDS, cs apart; ahead as in FloatEpilogue
    __device__ __forceinline__ void store8(int m, int n, const int (&acc)[8], const int8_t *lut_lds, const float *cl, int cs,
                                           const u32x4 *ahead) const {
        int a[8];
#pragma unroll
        for (int t = 0; t < 8; ++t)
            a[t] = acc[t];
        if (bias) {
            i32x4 b0 = *reinterpret_cast<const i32x4 *>(cl), b1 = *reinterpret_cast<const i32x4 *>(cl + 4);
#pragma unroll
            for (int t = 0; t < 4; ++t)
                a[t] += b0[t], a[4 + t] += b1[t];
        }
        const size_t o = (size_t)m * ldo + n;
        if (acc_out) {
            i32x4 *ap = reinterpret_cast<i32x4 *>(acc_out + o);
            ap[0] = i32x4{a[0], a[1], a[2], a[3]};
            ap[1] = i32x4{a[4], a[5], a[6], a[7]};
        }
        if (out || out_f) {
            float sc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            if (scale) {
                float4 s0 = *reinterpret_cast<const float4 *>(cl + cs), s1 = *reinterpret_cast<const float4 *>(cl + cs + 4);
                sc[0] = s0.x, sc[1] = s0.y, sc[2] = s0.z, sc[3] = s0.w, sc[4] = s1.x, sc[5] = s1.y, sc[6] = s1.z, sc[7] = s1.w;
            }
            int8_t q[8];
#pragma unroll
            for (int t = 0; t < 8; ++t)
                q[t] = float2int8_ref(__fmul_rn((float)a[t], sc[t]));
            if (lut_lds) {
#pragma unroll
                for (int t = 0; t < 8; ++t)
                    q[t] = lut_lds[(int)q[t] + 128];
            }
            if (out)
                store_out8(through, out + o, *reinterpret_cast<const store_u32x2 *>(q));
            if (out_f) {
                float d[8];
#pragma unroll
                for (int t = 0; t < 8; ++t)
                    d[t] = __fmul_rn((float)q[t], dq);
                if (out_f_dtype == TNN_ROCM_F32) {
                    if (residual) {
                        const float4 *rp = reinterpret_cast<const float4 *>((const float *)residual + o);
                        float4 r0 = rp[0], r1 = rp[1];
                        d[0] = __fadd_rn(d[0], r0.x), d[1] = __fadd_rn(d[1], r0.y), d[2] = __fadd_rn(d[2], r0.z),
                        d[3] = __fadd_rn(d[3], r0.w), d[4] = __fadd_rn(d[4], r1.x), d[5] = __fadd_rn(d[5], r1.y),
                        d[6] = __fadd_rn(d[6], r1.z), d[7] = __fadd_rn(d[7], r1.w);
                    }
                    float4 *fp = reinterpret_cast<float4 *>((float *)out_f + o);
                    store_out16(through, fp, store_u32x4{__float_as_uint(d[0]), __float_as_uint(d[1]), __float_as_uint(d[2]),
                                                __float_as_uint(d[3])});
                    store_out16(through, fp + 1, store_u32x4{__float_as_uint(d[4]), __float_as_uint(d[5]), __float_as_uint(d[6]),
                                                    __float_as_uint(d[7])});
                } else {
                    half_t h[8];
                    if (residual) {
                        *reinterpret_cast<u32x4 *>(h) = ahead ? *ahead : *reinterpret_cast<const u32x4 *>((const half_t *)residual + o);
#pragma unroll
                        for (int t = 0; t < 8; ++t)
                            d[t] = __fadd_rn(d[t], (float)h[t]);
                    }
#pragma unroll
                    for (int t = 0; t < 8; ++t)
                        h[t] = (half_t)d[t];
                    store_out16(through, (half_t *)out_f + o, *reinterpret_cast<const u32x4 *>(h));
                }
            }
        }
    }
};

// Quantised QKV projection for the attention layer: the int8 outputs of the three QuantizedInnerProduct layers are
// formed in registers (requantisation with scale[n] = w_scale[n] / o_scale of the column's section) and written
// already dequantised (q * dequant[n], the value the following Reformat layer produces) in the layout of
// QkvSplitEpilogue: columns [0,2H) -> qk[T,2H]; columns [2H,3H) -> V^T[b][head][d][s].
template <int DT> struct Int8QkvSplitEpilogue : StoreThrough {
    typedef typename Elem<DT>::type T;
    static constexpr bool kRowStats = false;
    const int32_t *bias;
    const float *scale;
    const float *dequant;
    T *qk;
    T *vt;
    int H, S, heads;
    int vt_sh;  // 0: V^T keys in natural order; 1: bits 2 and 3 of the key index change places (see key_slot)
    __device__ __forceinline__ void set_batch(int) {}
    struct ColConst {
        int32_t bias;
        float scale, dq;
    };
    __device__ __forceinline__ ColConst col_const(int n) const {
        ColConst c;
        c.bias  = bias ? bias[n] : 0;
        c.scale = scale[n];
        c.dq    = dequant[n];
        return c;
    }
    __device__ __forceinline__ void store(int m, int n, int acc, const ColConst &cc) const {
        int8_t q = float2int8_ref(__fmul_rn((float)(acc + cc.bias), cc.scale));
        float v  = __fmul_rn((float)q, cc.dq);
        if (n < 2 * H) {
            Elem<DT>::st(&qk[(size_t)m * 2 * H + n], v);
        } else {
            int c = n - 2 * H, b = m / S, s = key_slot(m - b * S, vt_sh);
            Elem<DT>::st(&vt[(((size_t)b * heads + (c >> 6)) * 64 + (c & 63)) * S + s], v);
        }
    }
    __device__ __forceinline__ bool direct(int n0) const { return n0 >= 2 * H; }
    static constexpr int kColArrays = 3;  // bias (its int32 bits), scale, dequant
    __device__ __forceinline__ float col_src(int k, int n) const {
        return k == 0 ? (bias ? __int_as_float(bias[n]) : 0.f) : k == 1 ? scale[n] : dequant[n];
    }
    __device__ __forceinline__ void store8(int m, int n, const int (&acc)[8], const float *cl, int cs, const u32x4 *) const {
        // the item's eight columns of the three arrays, from LDS
        const i32x4 b0 = *reinterpret_cast<const i32x4 *>(cl), b1 = *reinterpret_cast<const i32x4 *>(cl + 4);
        const float4 s0 = *reinterpret_cast<const float4 *>(cl + cs), s1 = *reinterpret_cast<const float4 *>(cl + cs + 4);
        const float4 d0 = *reinterpret_cast<const float4 *>(cl + 2 * cs), d1 = *reinterpret_cast<const float4 *>(cl + 2 * cs + 4);
        const int bb[8]   = {b0[0], b0[1], b0[2], b0[3], b1[0], b1[1], b1[2], b1[3]};
        const float sc[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
        const float dq[8] = {d0.x, d0.y, d0.z, d0.w, d1.x, d1.y, d1.z, d1.w};
        float v[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            int8_t q = float2int8_ref(__fmul_rn((float)(acc[t] + bb[t]), sc[t]));
            v[t]     = __fmul_rn((float)q, dq[t]);
        }
        if (n < 2 * H) {
            constexpr int NV = 8 * sizeof(T) / 16;
            u32x4 packed[NV];
            T *pe = reinterpret_cast<T *>(packed);
#pragma unroll
            for (int t = 0; t < 8; ++t)
                Elem<DT>::st(&pe[t], v[t]);
            u32x4 *cp = reinterpret_cast<u32x4 *>(qk + (size_t)m * 2 * H + n);
#pragma unroll
            for (int q = 0; q < NV; ++q)
                store_out16(through, &cp[q], packed[q]);
        } else {
            int c = n - 2 * H, b = m / S, s_ = key_slot(m - b * S, vt_sh);
            T *dst = vt + (((size_t)b * heads + (c >> 6)) * 64 + (c & 63)) * S + s_;
#pragma unroll
            for (int t = 0; t < 8; ++t)
                Elem<DT>::st_out(through, dst + (size_t)t * S, v[t]);
        }
    }
};

// 16-byte panel fetch with zero fill outside [0,rows) x [0,K).  `row_major_k` panels have k
// contiguous in memory.
template <typename T, bool ALIGNED>
__device__ __forceinline__ uint4 fetch_k_contig(const T *__restrict__ base, long ld, int row, int rows, int k, int K) {
    constexpr int VEC = 16 / sizeof(T);
    uint4 r           = make_uint4(0, 0, 0, 0);
    if (row < rows) {
        const T *p = base + (size_t)row * ld + k;
        if (ALIGNED) {
            if (k < K)
                r = *reinterpret_cast<const uint4 *>(p);
        } else {
            T *e = reinterpret_cast<T *>(&r);
#pragma unroll
            for (int t = 0; t < VEC; ++t)
                if (k + t < K)
                    e[t] = p[t];
        }
    }
    return r;
}

// B given as [K,N] (n contiguous): fetch 16 bytes along n at row k.
template <typename T, bool ALIGNED>
__device__ __forceinline__ uint4 fetch_n_contig(const T *__restrict__ base, long ld, int k, int K, int n, int N) {
    constexpr int VEC = 16 / sizeof(T);
    uint4 r           = make_uint4(0, 0, 0, 0);
    if (k < K) {
        const T *p = base + (size_t)k * ld + n;
        if (ALIGNED) {
            if (n < N)
                r = *reinterpret_cast<const uint4 *>(p);
        } else {
            T *e = reinterpret_cast<T *>(&r);
#pragma unroll
            for (int t = 0; t < VEC; ++t)
                if (n + t < N)
                    e[t] = p[t];
        }
    }
    return r;
}

template <int DT, int BM, int BN, int WM, int WN, bool B_NK, bool ALIGNED, typename Epi>
__global__ void __launch_bounds__(WM *WN * 64)
    gemm_kernel(const typename GemmTraits<DT>::elem *__restrict__ A, const typename GemmTraits<DT>::elem *__restrict__ B,
                int M, int N, int K, long lda, long ldb, int batch_a, int batch_b, long stride_a, long stride_b,
                int tiles_m, int tiles_n, Epi epi) {
    typedef typename GemmTraits<DT>::elem T;
    typedef typename GemmTraits<DT>::acc Acc;
    constexpr int NT      = WM * WN * 64;
    constexpr int VEC     = 16 / sizeof(T);
    constexpr int KB      = kSlabBytes / sizeof(T);  // k elements per slab
    constexpr int MT      = BM / WM / 32;
    constexpr int NTL     = BN / WN / 32;
    constexpr int A_VECS  = BM * 4 / NT;  // 16-byte vectors of the A slab per thread
    constexpr int B_VECS  = BN * 4 / NT;
    static_assert(BM * 4 % NT == 0 && BN * 4 % NT == 0, "slab must divide evenly over the workgroup");
    static_assert(BM % (WM * 32) == 0 && BN % (WN * 32) == 0, "wave tile must be a multiple of 32x32");

    __shared__ __attribute__((aligned(16))) unsigned char lds_a[2][BM * kLdsStride];
    __shared__ __attribute__((aligned(16))) unsigned char lds_b[2][BN * kLdsStride];

    const int tid  = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wm   = wave / WN;
    const int wn   = wave % WN;

    // XCD-aware tile order: workgroups are dealt round-robin to the 8 XCDs, so give each XCD a
    // contiguous run of tiles (shared A row panels stay in one L2).
    int pid           = blockIdx.x;
    const int n_tiles = tiles_m * tiles_n;
    if ((n_tiles & 7) == 0) {
        pid = (pid & 7) * (n_tiles >> 3) + (pid >> 3);
    }
    const int tm = pid / tiles_n;
    const int tn = pid % tiles_n;
    const int m0 = tm * BM;
    const int n0 = tn * BN;

    const int bz = blockIdx.y;
    A += (size_t)(bz % batch_a) * stride_a;
    B += (size_t)(bz % batch_b) * stride_b;
    epi.set_batch(bz);

    uint4 ra[A_VECS], rb[B_VECS];

    auto load_global = [&](int k0) {
#pragma unroll
        for (int i = 0; i < A_VECS; ++i) {
            int v   = tid + i * NT;
            int row = v >> 2, kc = (v & 3) * VEC;
            ra[i] = fetch_k_contig<T, ALIGNED>(A, lda, m0 + row, M, k0 + kc, K);
        }
        if (B_NK) {
#pragma unroll
            for (int i = 0; i < B_VECS; ++i) {
                int v   = tid + i * NT;
                int row = v >> 2, kc = (v & 3) * VEC;
                rb[i] = fetch_k_contig<T, ALIGNED>(B, ldb, n0 + row, N, k0 + kc, K);
            }
        } else {
            // slab is KB rows (k) x BN columns (n): BN/VEC vectors per k row
#pragma unroll
            for (int i = 0; i < B_VECS; ++i) {
                int v  = tid + i * NT;
                int kr = v / (BN / VEC), nc = (v % (BN / VEC)) * VEC;
                rb[i] = fetch_n_contig<T, ALIGNED>(B, ldb, k0 + kr, K, n0 + nc, N);
            }
        }
    };

    auto store_lds = [&](int buf) {
#pragma unroll
        for (int i = 0; i < A_VECS; ++i) {
            int v   = tid + i * NT;
            int row = v >> 2, kc = (v & 3);
            *reinterpret_cast<uint4 *>(&lds_a[buf][row * kLdsStride + kc * 16]) = ra[i];
        }
        if (B_NK) {
#pragma unroll
            for (int i = 0; i < B_VECS; ++i) {
                int v   = tid + i * NT;
                int row = v >> 2, kc = (v & 3);
                *reinterpret_cast<uint4 *>(&lds_b[buf][row * kLdsStride + kc * 16]) = rb[i];
            }
        } else {
#pragma unroll
            for (int i = 0; i < B_VECS; ++i) {
                int v  = tid + i * NT;
                int kr = v / (BN / VEC), nc = (v % (BN / VEC)) * VEC;
                const T *e = reinterpret_cast<const T *>(&rb[i]);
#pragma unroll
                for (int t = 0; t < VEC; ++t)
                    *reinterpret_cast<T *>(&lds_b[buf][(nc + t) * kLdsStride + kr * (int)sizeof(T)]) = e[t];
            }
        }
    };

    Acc acc[MT][NTL];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NTL; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                acc[i][j][r] = 0;

    const int nk = (K + KB - 1) / KB;
    load_global(0);
    store_lds(0);
    __syncthreads();

    const int frag_row = lane & 31;
    const int frag_off = (lane >> 5) * 16;

    for (int kt = 0; kt < nk; ++kt) {
        const int buf = kt & 1;
        if (kt + 1 < nk)
            load_global((kt + 1) * KB);
#pragma unroll
        for (int kk = 0; kk < kSlabBytes / 32; ++kk) {
            uint4 fa[MT], fb[NTL];
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                int row = wm * (BM / WM) + i * 32 + frag_row;
                fa[i]   = *reinterpret_cast<const uint4 *>(&lds_a[buf][row * kLdsStride + kk * 32 + frag_off]);
            }
#pragma unroll
            for (int j = 0; j < NTL; ++j) {
                int row = wn * (BN / WN) + j * 32 + frag_row;
                fb[j]   = *reinterpret_cast<const uint4 *>(&lds_b[buf][row * kLdsStride + kk * 32 + frag_off]);
            }
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NTL; ++j)
                    GemmTraits<DT>::mma(fa[i], fb[j], acc[i][j]);
        }
        if (kt + 1 < nk)
            store_lds(buf ^ 1);
        __syncthreads();
    }

    // epilogue: lane = column, registers = rows
#pragma unroll
    for (int j = 0; j < NTL; ++j) {
        int n = n0 + wn * (BN / WN) + j * 32 + (lane & 31);
        if (n < N) {
            auto cc = epi.col_const(n);
#pragma unroll
            for (int i = 0; i < MT; ++i) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    int m = m0 + wm * (BM / WM) + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                    if (m < M)
                        epi.store(m, n, acc[i][j][r], cc);
                }
            }
        }
    }
}


// ---- tiled, pipelined kernel for the aligned x * W^T case ----------------------------------------------
// One workgroup of four or eight waves (one or two per SIMD) per output tile.  The waves form a WGM x WGN x WGK grid: a wave
// owns a (32*TM) x (32*TN) block of the tile and, when WGK > 1, every WGK-th 32-byte k-step of each slab
// (the partial sums of the WGK waves are added in the epilogue).  Tile = (32*TM*WGM) x (32*TN*WGN).
//   * the launcher picks the shape so that the tile count is at most (or a multiple of) the CU count with
//     tiles as large as registers allow: fewer bytes per flop from L2 and LDS, no second partial round;
//   * k-slabs of SLAB bytes per row; two slabs in flight in registers in addition to the one being consumed
//     from LDS (global loads for slab k+2 are issued before the MFMAs of slab k);
//   * the MFMA operands are swapped (the W panel is the "A" operand), so a lane owns one output ROW and
//     four consecutive columns per accumulator group;
//   * the epilogue turns the accumulators through LDS into a row-contiguous layout, so C, bias and residual
//     move as whole cache lines.
// LDS is dynamic: max(2 buffers x (BM + BN) rows x (SLAB + 16) bytes, 4 x 32 x (32*TN + 4) words of staging).
// NSTAGE = 0: slabs travel global -> registers -> LDS (padded rows, two LDS buffers).
// NSTAGE = 2 or 3: slabs travel global -> LDS directly (global_load_lds_dwordx4: no staging registers and no LDS
//     store instructions), into NSTAGE un-padded buffers whose 16-byte chunks are XOR-swizzled per row so that the
//     fragment reads stay free of bank conflicts; loads run NSTAGE-1 slabs ahead of the MFMAs.
// OWN (with WGM = WGN = 1): every k-wave has a ring of NSTAGE slabs of its own and walks a contiguous part of K by itself.
//     A slab is then SLAB bytes of k of ALL rows of the tile for ONE wave, and nothing in the main loop concerns another
//     wave: no barrier, each wave waits for its own loads only.
// BLK = 16 (slabs direct to LDS): the waves' blocks are 16 x 16 instead of 32 x 32 (v_mfma_*_16x16x32, 64 bytes of k a step), TM
//     and TN count those.
// SETS (shared slabs of two steps a wave): sets of sums that a wave's steps take turns on, added up at the end.  A sum in fp32 grows its
//     error with the root of the products that follow one another in it, and the shapes of 32 x 32 blocks that these took the place of
//     had K in two, four or eight parts.  K is in WGK * SETS parts here, as many as those had: 96 x 96 tiles eight, 64 x 64 four, 128 x 128
//     and larger two (three stages deep four: they took the place of some 64 x 64 ones, too).  256 x 256 tiles have no registers for a second
//     set and one part, as they had.  FOLDS (192 x 128 from K = 2048 on): the sets go to totals every 768 products, eight parts of
//     K = 3072, where such tiles took the place of 96 x 96 ones.  (As a kernel of its own: with the totals in one, launches of K = 768
//     and 1024 took 2 .. 5 % more.)  Error of the sums (2-norm over 2-norm), fp16, K = 768 / 3072 / 4096:
//       shapes before: 96 x 96 0.85 / 1.41 / 1.54e-7, 64 x 64 1.00 / 1.82 / 2.03, 128 x 128 1.29 / 2.45 / 2.97
//       one set:       96 x 96 1.28 / 2.56 / 2.91e-7, 64 x 64 1.28 / 2.56 / 2.91, 128 x 128 1.73 / 3.53 / 4.06
//       these:         96 x 96 0.81 / 1.35 / 1.51e-7, 64 x 64 0.99 / 1.83 / 2.10, 128 x 128 1.28 / 2.56 / 2.91
//     A launch takes 0.992 of what it did with one set in the mean (96 of hidden sizes 768 and 1024, 64 to 8192 rows), at most 1.007, with folds
//     1.03 (5600 x 768 x 3072 31.9 -> 32.7).
template <int TM_, int TN_, int WGM_, int WGN_, int WGK_, int SLAB_, int NSTAGE_ = 0, bool OWN_ = false, int BLK_ = 32,
          int SETS_ = 1, bool FOLDS_ = false>
struct TileCfg {
    static constexpr int BLK = BLK_;
    // groups of rows that are staged one after the other, and the rows of a wave position in one: blocks of 32 rows, or the whole tile
    // where it is one of 16 x 16 blocks and fits into LDS at once (256 x 256 tiles do not: halves)
    static constexpr int GROUPS = BLK_ == 32 ? TM_ : WGM_ * WGN_ * WGK_ * TM_ * (4 * TN_ + 1) > 640 ? 2 : 1, GROWS = BLK_ * TM_ / GROUPS;
    static_assert(BLK_ == 32 || (BLK_ == 16 && NSTAGE_ > 0 && (!OWN_ || BLK_ * TM_ <= 32)), "16 x 16 blocks: direct-to-LDS slabs only");
    static constexpr int TM = TM_, TN = TN_, WGM = WGM_, WGN = WGN_, WGK = WGK_, SLAB = SLAB_, NSTAGE = NSTAGE_;
    static constexpr bool OWN = OWN_, FOLDS = FOLDS_;
    static constexpr int SETS = SETS_;
    static constexpr int BM = BLK * TM * WGM, BN = BLK * TN * WGN;
    static constexpr int STRIDE = NSTAGE_ ? SLAB : SLAB + 16;
    static constexpr int SSTR   = BLK * TN + 4;  // staged row stride in 32-bit words
    static constexpr size_t slab_bytes  = (size_t)(NSTAGE_ ? NSTAGE_ : 2) * (BM + BN) * STRIDE * (OWN_ ? WGK_ : 1);
    static constexpr size_t stage_bytes = (size_t)WGM_ * WGN_ * WGK_ * GROWS * SSTR * 4;
    static constexpr size_t lds_bytes   = slab_bytes > stage_bytes ? slab_bytes : stage_bytes;
    // Row sums of what an epilogue stored.  Where all columns are one wave's they are added up over the two to eight lanes that hold a
    // row (32 x 32 tiles, 256 x 768 x 768: 4.60 -> 4.40 us against sums through LDS), and so are those of each wave's 64 columns where the
    // tile is staged in groups; elsewhere an item's pair goes into the place of its own staged values, which takes the whole tile
    // staged at once.
    static constexpr bool sums_by_lanes = OWN_ || (GROUPS > 1 && BLK_ * TN_ == 64);
    static constexpr bool leaves_sums   = sums_by_lanes || GROUPS == 1;
    static constexpr int sum_cols       = sums_by_lanes ? BLK_ * TN_ : BN;  // columns of a pair of row sums
    static constexpr int NW = WGM * WGN * WGK, NT = 64 * NW;  // waves and threads per workgroup
    static_assert(NW == 4 || NW == 8, "four or eight waves per workgroup");
    static_assert(OWN_ || ((BM * (SLAB / 16)) % NT == 0 && (BN * (SLAB / 16)) % NT == 0), "slab must divide over the workgroup");
    static_assert(!OWN_ || (WGM_ == 1 && WGN_ == 1 && NSTAGE_ >= 2 && NSTAGE_ <= 3), "rings of two or three slabs, k-waves only");
    static_assert(OWN_ || NSTAGE_ == 0 || (NSTAGE_ >= 2 && NSTAGE_ <= 3), "register-staged, or two or three direct-to-LDS stages");
};

// Dynamic LDS of one (tile shape, epilogue) pair, for the kernel and its launcher alike: the slab / staging area, what
// the epilogue keeps behind it, and at the very end the tile's columns of the epilogue's per-column arrays followed by
// its per-row pairs.
template <typename CFG, typename Epi> struct EpiLds {
    static constexpr size_t lut_need   = CFG::stage_bytes + 256;  // Int8Epilogue's table behind the staging area
    static constexpr size_t stats_need = CFG::stage_bytes + (size_t)CFG::BM * (8 + 16 * CFG::WGK * CFG::WGN);
    static constexpr size_t base0 = std::is_same<Epi, Int8Epilogue>::value && lut_need > CFG::lds_bytes ? lut_need : CFG::lds_bytes;
    // row statistics and the partial-sum buffer sit behind the staging area; handed-over sums park {rstd, mean} per row
    // behind the slabs before the main loop
    static constexpr size_t base1 = TakesRowSums<Epi>::value ? CFG::lds_bytes + (size_t)CFG::BM * 8
                                    : (Epi::kRowStats && stats_need > base0) ? stats_need : base0;
    static constexpr size_t col_offset = (base1 + 15) & ~(size_t)15;
    static constexpr size_t row_offset = col_offset + (size_t)ColArrays<Epi>::value * CFG::BN * 4;
    static constexpr size_t side_bytes = (size_t)ColArrays<Epi>::value * CFG::BN * 4 + (RowIn<Epi>::value ? (size_t)CFG::BM * 8 : 0);
    static constexpr size_t total      = col_offset + side_bytes;
};

// s_waitcnt that waits only for the vector-memory counter to drop to n (gfx9 encoding: vmcnt in bits 3:0 and
// 15:14, expcnt 6:4 and lgkmcnt 11:8 left at their maxima)
#define TR_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt((((n)&0xF) | ((((n) >> 4) & 3) << 14) | (0x7 << 4) | (0xF << 8)))

// Divisors of the tile order: tiles of a group, tile rows of a group, tile rows of the last, smaller group; and the tile rows of a
// group.  With the panels and the sizes in front of them they are 13 words, which is what the dispatcher has registers for
// (-amdgpu-kernarg-preload-count): a workgroup requests its first slab without a look at the argument memory, which
// nothing on the chip has read yet.  us a launch, all arguments loaded -> these in registers, fp16, twelve weight sets in turn:
//   32 x 768 x 3072 5.41 -> 5.13, 32 x 2304 x 768 4.84 -> 4.65, 985 x 2304 x 768 10.0 -> 9.7
struct TileOrder {
    uint32_t group, rows, last_rows;  // FixedDivisor::magic
    uint32_t packed;                  // their shifts, six bits each, and the tile rows of a group from bit 18 on
    static constexpr int kMaxRows = (1 << 14) - 1;
    static TileOrder of(int tiles_m, int tiles_n, int group_m) {
        const FixedDivisor g = FixedDivisor::of((uint32_t)group_m * (uint32_t)tiles_n), r = FixedDivisor::of((uint32_t)group_m),
                           l = FixedDivisor::of((uint32_t)(tiles_m % group_m));
        return {g.magic, r.magic, l.magic, g.shift | r.shift << 6 | l.shift << 12 | (uint32_t)group_m << 18};
    }
};

// An infinity, a NaN or a finite value from 2^104 on has no planes (split_f32.h), and turns every sum it enters into something
// that is not finite, as a sum beyond 2^80 becomes by itself.  A wave that finds such a sum in one of its 32 x 32 blocks
// multiplies that block again, its own part of K, with the fp32 matrix instruction and operands straight from memory, and
// takes those sums in the place of the ones that are not finite.  pa, pb = this lane's row of A and of B, eight values into the step for the upper
// lanes; steps of 16 k from `first` to `end`, `stride` apart.
// Nothing overlaps here, so a block costs several times what it did: [384,3072] x [3072,768] takes 28 us, with two rows that
// are not finite 74, with every value NaN 91 (one thread per sum: 1.6 ms and 1.9 ms; 96 x 96 tiles 78 -> 350, were 13 ms).
template <typename Acc>
__device__ __forceinline__ void multiply_again(const float *pa, const float *pb, int first, int end, int stride, Acc &acc) {
    constexpr int REGS = sizeof(Acc) / 4;  // 16: a 32 x 32 block, a lane holds 8 of a step's values; 4: 16 x 16, it holds 4
    Acc sum;
#pragma unroll
    for (int r = 0; r < REGS; ++r)
        sum[r] = 0.f;
#pragma unroll 1
    for (int t = first; t < end; t += stride) {
        const uint4 *a = reinterpret_cast<const uint4 *>(pa + (size_t)t * 16), *b = reinterpret_cast<const uint4 *>(pb + (size_t)t * 16);
#pragma unroll
        for (int h = 0; h < REGS / 8 + (REGS < 8); ++h)
            GemmTraits<TNN_ROCM_F32>::mma(b[h], a[h], sum);
    }
#pragma unroll
    for (int r = 0; r < REGS; ++r)
        acc[r] = split_finite(__builtin_fabsf(acc[r])) ? acc[r] : sum[r];
}

template <int DT, typename CFG, typename Epi>
__global__ void __launch_bounds__(CFG::NT)
    gemm_nk_tiled_kernel(const typename GemmTraits<DT>::elem *__restrict__ A,
                         const typename GemmTraits<DT>::elem *__restrict__ B, int M, int N, int K, int lda, int ldb,
                         uint32_t group_magic, uint32_t rows_magic, uint32_t last_magic, uint32_t order_packed, Epi epi) {
    typedef typename GemmTraits<DT>::elem T;
    constexpr int BLK = CFG::BLK, GROUPS = CFG::GROUPS, GROWS = CFG::GROWS;
    typedef typename std::conditional<BLK == 32, typename GemmTraits<DT>::acc, typename GemmTraits<DT>::acc_small>::type Acc;
    constexpr int TM = CFG::TM, TN = CFG::TN, WGN = CFG::WGN, WGK = CFG::WGK, SLAB = CFG::SLAB;
    constexpr int BM = CFG::BM, BN = CFG::BN, STRIDE = CFG::STRIDE;
    constexpr int NT     = CFG::NT;
    constexpr int VEC    = 16 / sizeof(T);
    constexpr int KB     = SLAB / sizeof(T);
    constexpr int VPR    = SLAB / 16;  // 16-byte vectors per slab row
    constexpr int A_VECS = BM * VPR / NT;
    constexpr int B_VECS = BN * VPR / NT;

    extern __shared__ __attribute__((aligned(16))) unsigned char lds_dyn[];

    const int tid  = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wk   = wave % WGK;
    const int wn   = (wave / WGK) % WGN;
    const int wm   = wave / (WGK * WGN);

    // Tile order.  Workgroups are dealt round-robin to the 8 XCDs, each with its own 4 MB L2, and run roughly in
    // launch order.  Every XCD takes a contiguous run of a "grouped" tile order (group_m tile rows at a time, down
    // the rows first, then the next tile column), so the tiles that are resident together on one XCD form a
    // compact block of the tile grid: their A and W panels fit that L2 and are fetched from HBM once, instead of
    // the whole W panel streaming through every L2 once per tile row.
    TR_TL(0);  // entry
    // the epilogue's arguments, needed behind the first slab requests only
    const uint32_t epi_args = request_kernel_args<56 + sizeof(Epi)>();
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    const int n_tiles = tiles_m * tiles_n;
    const int per_xcd = (n_tiles + 7) >> 3;
    const int vid     = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    const int group_m  = (int)(order_packed >> 18);
    const int grp      = FixedDivisor{group_magic, order_packed & 63}.quotient(vid);
    const int first_m  = grp * group_m;
    const bool last_g  = tiles_m - first_m < group_m;
    const int rows_g   = last_g ? tiles_m - first_m : group_m;
    const int in_grp   = vid - grp * group_m * tiles_n;
    const int col_g    = FixedDivisor{last_g ? last_magic : rows_magic, (order_packed >> (last_g ? 12 : 6)) & 63}.quotient(in_grp);
    const int m0       = (first_m + in_grp - col_g * rows_g) * BM;
    const int n0       = col_g * BN;
    if (vid >= n_tiles)
        return;  // the grid is padded to a multiple of 8; whole workgroups leave before any barrier

    // ---- what the epilogue reads, requested with the first slabs where a thread has few items and registers to spare: behind
    // the main loop the same loads are two latencies one after the other (columns and row pairs, then the residual), 0.4 us
    // of a launch of 4
    constexpr int CW    = TN * BLK;      // columns per wave
    constexpr int CPR   = CW / 8;        // 8-column pieces per staged row
    constexpr int POS   = CFG::NW / WGK;  // wave positions (wm, wn) in the tile
    constexpr int ITEMS = POS * GROWS * CPR;
    constexpr int MY_ITEMS = (ITEMS + NT - 1) / NT;  // of a thread
    constexpr bool EARLY = GROUPS == 1 && MY_ITEMS <= 3 && CFG::NSTAGE > 0;
    const bool by_rows   = epi.direct(n0);
    // row and first column (inside the tile) of an item of the first group of rows of every wave position
    auto item_at = [&](int item, int *row, int *col) __attribute__((always_inline)) {
        const int c8  = by_rows ? ((item / GROWS) % CPR) * 8 : (item % CPR) * 8;
        const int r   = by_rows ? (item % GROWS) : (item / CPR) % GROWS;
        const int pos = item / (CPR * GROWS);
        *row          = (pos / WGN) * GROUPS * GROWS + r;
        *col          = (pos % WGN) * CW + c8;
    };
    constexpr int COLQ = (ColArrays<Epi>::value * BN + NT - 1) / NT;
    float early_col[COLQ > 0 ? COLQ : 1];
    float2 early_row = make_float2(0.f, 0.f);
    constexpr int AHEAD = EARLY ? AheadVecs<Epi>::value : 0;
    u32x4 ahead_vec[MY_ITEMS][AHEAD > 0 ? AHEAD : 1];
    auto request_columns = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < COLQ; ++q) {
            // clamped, not guarded: what lies outside is never used, and a branch costs more than the load
            constexpr int LAST = ColArrays<Epi>::value * BN - 1;
            const int e  = q * NT + tid < LAST ? q * NT + tid : LAST, n = n0 + e % BN;
            early_col[q] = epi.col_src(e / BN, n < N ? n : N - 1);
        }
        if constexpr (RowIn<Epi>::value)
            early_row = epi.row_src(m0 + tid % BM < M ? m0 + tid % BM : M - 1);
    };
    // Behind the first slabs: their place in memory is not in a register.  What waits for the first slabs waits for these as well.
    auto request_ahead = [&]() __attribute__((always_inline)) {
        asm volatile("" ::"s"(epi_args));
        if constexpr (EARLY) {
            if constexpr (ColArrays<Epi>::value > 0)
                request_columns();
            if constexpr (AHEAD > 0) {
#pragma unroll
                for (int it = 0; it < MY_ITEMS; ++it) {
                    int row = 0, col = 0;
                    item_at((it * NT + tid) % ITEMS, &row, &col);
                    const int m = m0 + row < M ? m0 + row : M - 1, n = n0 + col + 8 <= N ? n0 + col : N - 8;
                    if (N >= 8) {
                        const u32x4 *src = reinterpret_cast<const u32x4 *>(epi.ahead_src(m, n));
                        if (src) {
#pragma unroll
                            for (int q = 0; q < AHEAD; ++q)
                                ahead_vec[it][q] = src[q];
                        }
                    }
                }
            }
        }
    };

    constexpr int SETS = DT == TNN_ROCM_I8 ? 1 : CFG::SETS;  // sums of whole numbers are exact
    Acc parts[SETS][TM][TN];
    Acc(&acc)[TM][TN] = parts[0];
    auto clear = [](Acc(&sums)[TM][TN]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int r = 0; r < BLK * BLK / 64; ++r)
                    sums[i][j][r] = 0;
    };
    auto add_to = [](Acc(&sums)[TM][TN], const Acc(&more)[TM][TN]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                sums[i][j] += more[i][j];
    };
    if constexpr (SETS == 1)
        clear(parts[0]);

    const int frag_row = lane & (BLK - 1);
    const int frag_off = (lane >> 5) * 16;  // slabs staged through registers: blocks of 32 x 32
    const int nk       = K / KB;
    constexpr int FRAGS = GemmTraits<DT>::FRAGS, KSTEP = (1024 / BLK) * FRAGS;  // bytes of k per row that one step multiplies
    const SplitConst split_const;

    // LayerNorm-folding epilogues: this lane's share of sum / sum of squares of A row (wm * TM + i) * 32 + frag_row.  The
    // eight values of a fragment are added up in fp32, the fragments in double: every tile shape deals the fragments out to
    // its waves in another way, and the statistics should not depend on that.
    double ln_s1[TM], ln_s2[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i)
        ln_s1[i] = ln_s2[i] = 0.0;
    auto ln_take = [&](const uint4 &frag, int i) __attribute__((always_inline)) {
        float s1 = 0.f, s2 = 0.f;
        ln_accumulate<DT>(frag, s1, s2);
        ln_s1[i] += (double)s1;
        ln_s2[i] += (double)s2;
    };

    if constexpr (CFG::OWN) {
        // Every wave streams its own part of K: both panels' rows of one k-slab of SLAB bytes per stage, through a ring that
        // only this wave fills and reads.  Row swizzle as in the shared pipeline below.
        static_assert(!TakesRowSums<Epi>::value, "own-ring shapes take the row statistics from their A fragments");
        constexpr int NS   = CFG::NSTAGE;
        constexpr int RPL  = 1024 / SLAB;  // slab rows per load instruction
        constexpr int R256 = 256 / SLAB;
        constexpr int A_LD = BM / RPL, B_LD = BN / RPL, LPW = A_LD + B_LD;
        constexpr int STAGE = (BM + BN) * SLAB;
        static_assert(SLAB <= 256 && BM % RPL == 0 && BN % RPL == 0 && (NS - 1) * LPW < 64, "ring shape");
        uint32_t a_off[A_LD], b_off[B_LD];
        const int lrow = lane / VPR, lpos = lane % VPR;
#pragma unroll
        for (int i = 0; i < A_LD; ++i) {
            const int r = i * RPL + lrow;
            int row     = m0 + r;
            row         = row < M ? row : M - 1;
            a_off[i]    = ((uint32_t)row * (uint32_t)lda + (uint32_t)((lpos ^ ((r / R256) % VPR)) * VEC)) * (uint32_t)sizeof(T);
        }
#pragma unroll
        for (int i = 0; i < B_LD; ++i) {
            const int r = i * RPL + lrow;
            int row     = n0 + r;
            row         = row < N ? row : N - 1;
            b_off[i]    = ((uint32_t)row * (uint32_t)ldb + (uint32_t)((lpos ^ ((r / R256) % VPR)) * VEC)) * (uint32_t)sizeof(T);
        }
        const int uwave         = __builtin_amdgcn_readfirstlane(wave);
        const uint32_t ring_dst = (uint32_t)(uintptr_t)lds_dyn + (uint32_t)(uwave * NS * STAGE);
        const unsigned char *const ring = lds_dyn + uwave * NS * STAGE;
        // spelled as assembly for the reason given at the shared pipeline's load
        auto load16 = [](const T *base, uint32_t byte_off, uint32_t lds_addr) {
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                         :
                         : "v"(byte_off), "s"(base), "s"(lds_addr)
                         : "memory", "m0");
        };
        // load k of a slab; the weights first: they come from further away
        auto issue_one = [&](int k, int slab, int stage) __attribute__((always_inline)) {
            const uint32_t dst = ring_dst + (uint32_t)(stage * STAGE);
            if (k >= B_LD)
                load16(A + (size_t)slab * KB, a_off[k >= B_LD ? k - B_LD : 0], dst + (k - B_LD) * 1024);
            else
                load16(B + (size_t)slab * KB, b_off[k < B_LD ? k : 0], dst + BM * SLAB + k * 1024);
        };
        auto issue = [&](int slab, int stage) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < LPW; ++k)
                issue_one(k, slab, stage);
        };
        const int fswz = (frag_row / R256) & (VPR - 1);
        const int frow = frag_row * SLAB;
        const int k_lo = nk * uwave / CFG::WGK, k_hi = nk * (uwave + 1) / CFG::WGK;
#pragma unroll
        for (int p = 0; p < NS; ++p)
            if (k_lo + p < k_hi)
                issue(k_lo + p, p);
        TR_TL(5);  // first slabs requested
        request_ahead();
        int stage = 0;
        auto wait_for = [&](int kt) __attribute__((always_inline)) {
            // slab kt is complete once at most the loads of the slabs requested after it are outstanding
            const int behind = k_hi - 1 - kt;
            if (NS > 2 && behind >= 2)
                TR_WAIT_VMCNT(NS > 2 ? 2 * LPW : 0);
            else if (behind >= 1)
                TR_WAIT_VMCNT(LPW);
            else
                TR_WAIT_VMCNT(0);
            asm volatile("" ::: "memory");
        };
        auto read_fragments = [&](uint4 (&f)[SLAB / KSTEP][TM + TN][FRAGS]) __attribute__((always_inline)) {
            const unsigned char *sa = ring + stage * STAGE, *sb = sa + BM * SLAB;
#pragma unroll
            for (int kf = 0; kf < SLAB * BLK / 1024; ++kf) {
                const int chunk = ((kf * (64 / BLK) + lane / BLK) ^ fswz) * 16;
#pragma unroll
                for (int i = 0; i < TM; ++i)
                    f[kf / FRAGS][i][kf % FRAGS] = *reinterpret_cast<const uint4 *>(sa + i * BLK * SLAB + frow + chunk);
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    f[kf / FRAGS][TM + j][kf % FRAGS] = *reinterpret_cast<const uint4 *>(sb + j * BLK * SLAB + frow + chunk);
            }
        };
        if constexpr (DT == TNN_ROCM_F32) {
            if (k_lo < k_hi) {
                typedef SplitSlab<TM, TN, SLAB / KSTEP> Planes;
                Planes p, q;
                auto half = [&](int kt, const Planes &now, Planes &next, auto loads) __attribute__((always_inline)) {
                    typename Planes::Reads rd;
                    wait_for(kt);
                    read_fragments(rd.f);
                    const int here = stage;
                    stage = stage + 1 == NS ? 0 : stage + 1;
                    now.template turn<decltype(loads)::value, true>(
                        rd, next, acc, split_const, [&](int k) __attribute__((always_inline)) { issue_one(k, kt + NS, here); });
                };
                typedef std::integral_constant<int, LPW> WithLoads;
                typedef std::integral_constant<int, 0> NoLoads;
                {
                    typename Planes::Reads rd;
                    wait_for(k_lo);
                    read_fragments(rd.f);
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                    if (k_lo + NS < k_hi)
                        issue(k_lo + NS, 0);
                    stage = 1;
                    p.convert(rd, split_const);
                }
                int kt = k_lo + 1;
                for (; kt + 1 + NS < k_hi; kt += 2) {
                    half(kt, p, q, WithLoads());
                    half(kt + 1, q, p, WithLoads());
                }
                // the last slabs: one more to request at most
                if (kt + NS < k_hi) {
                    half(kt, p, q, WithLoads());
                    p = q;
                    ++kt;
                }
                for (; kt + 1 < k_hi; kt += 2) {
                    half(kt, p, q, NoLoads());
                    half(kt + 1, q, p, NoLoads());
                }
                if (kt < k_hi) {
                    half(kt, p, q, NoLoads());
                    q.multiply(acc);
                } else {
                    p.multiply(acc);
                }
            }
        } else {
            for (int kt = k_lo; kt < k_hi; ++kt) {
                uint4 f[SLAB / KSTEP][TM + TN][FRAGS];
                wait_for(kt);
                read_fragments(f);
                // the fragments are in registers before the slab's place is given to the next load
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                if (kt + NS < k_hi)
                    issue(kt + NS, stage);
                stage = stage + 1 == NS ? 0 : stage + 1;
#pragma unroll
                for (int kk = 0; kk < SLAB / KSTEP; ++kk) {
                    if constexpr (Epi::kRowStats) {
#pragma unroll
                        for (int i = 0; i < TM; ++i)
                            ln_take(f[kk][i][0], i);
                    }
#pragma unroll
                    for (int i = 0; i < TM; ++i)
#pragma unroll
                        for (int j = 0; j < TN; ++j)
                            GemmTraits<DT>::mma(f[kk][TM + j][0], f[kk][i][0], acc[i][j]);
                }
            }
        }
    } else if constexpr (CFG::NSTAGE > 0) {
        // Direct-to-LDS pipeline.  One load instruction of a wave fills 1024 contiguous LDS bytes (lane L writes
        // bytes 16L..16L+15), i.e. RPL whole slab rows; the lane picks WHICH 16 global bytes land there, so the
        // swizzle is applied on the global side: physical chunk p of LDS row r holds logical chunk p ^ f(r),
        // f(r) = (r / rows per 256 bytes) mod VPR.  Sixteen consecutive rows reading the same logical chunk then
        // touch sixteen different 16-byte bank groups.
        constexpr int NS    = CFG::NSTAGE;
        constexpr int RPL   = 1024 / SLAB;        // slab rows per wave-load
        constexpr int R256  = 256 / SLAB > 0 ? 256 / SLAB : 1;
        constexpr int A_LD  = BM / RPL / CFG::NW;  // wave-loads of A per wave and slab
        constexpr int B_LD  = BN / RPL / CFG::NW;
        constexpr int STAGE = (BM + BN) * SLAB;
        static_assert(BM % (RPL * CFG::NW) == 0 && BN % (RPL * CFG::NW) == 0, "slab rows must divide over the waves");
        static_assert((NS - 1) * (A_LD + B_LD) < 64, "look-ahead must fit the vmcnt counter");
        uint32_t a_off[A_LD], b_off[B_LD];
        const int lrow = lane / VPR, lpos = lane % VPR;
#pragma unroll
        for (int i = 0; i < A_LD; ++i) {
            const int r = (wave + i * CFG::NW) * RPL + lrow;
            int row     = m0 + r;
            row         = row < M ? row : M - 1;
            a_off[i]    = (uint32_t)row * (uint32_t)lda + (uint32_t)((lpos ^ ((r / R256) % VPR)) * VEC);
        }
#pragma unroll
        for (int i = 0; i < B_LD; ++i) {
            const int r = (wave + i * CFG::NW) * RPL + lrow;
            int row     = n0 + r;
            row         = row < N ? row : N - 1;
            b_off[i]    = (uint32_t)row * (uint32_t)ldb + (uint32_t)((lpos ^ ((r / R256) % VPR)) * VEC);
        }
        // The load is spelled as inline assembly on purpose: for the compiler's own global_load_lds builtin the
        // wait-count pass puts vmcnt(0) in front of every later LDS read (it cannot tell the stages apart), which
        // serialises the pipeline.  Here the waits are placed by hand (TR_WAIT_VMCNT below): a slab has landed once no more operations
        // are outstanding than the slab loads requested after it.  Any other vector-memory operation behind a slab (the epilogue's
        // early reads between the first slabs and the next, the late row sums behind the last) is one more that is
        // younger, so that a wait lets it stand in a slab load's place and waits longer, never shorter; one in front of a slab
        // (the early row sums) is older and done before it.  m0 carries the wave-uniform LDS address and needs one wait state
        // before the load.
        const uint32_t lds_base = (uint32_t)(uintptr_t)lds_dyn;  // generic -> LDS offset (low 32 bits of the aperture address)
        const uint32_t wave_dst = (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds_base + (uint32_t)wave * 1024u));
        auto load16 = [](const T *base, uint32_t byte_off, uint32_t lds_addr) {
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                         :
                         : "v"(byte_off), "s"(base), "s"(lds_addr)
                         : "memory", "m0");
        };
        auto issue_one = [&](int k, int slab, int stage) __attribute__((always_inline)) {  // load k of a slab
            const uint32_t dst = wave_dst + (uint32_t)(stage * STAGE);
            if (k < A_LD)
                load16(A + (size_t)slab * KB, a_off[k < A_LD ? k : 0] * (uint32_t)sizeof(T), dst + k * CFG::NW * 1024);
            else
                load16(B + (size_t)slab * KB, b_off[k >= A_LD ? k - A_LD : 0] * (uint32_t)sizeof(T),
                       dst + BM * SLAB + (k - A_LD) * CFG::NW * 1024);
        };
        auto issue = [&](int slab, int stage) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < A_LD + B_LD; ++k)
                issue_one(k, slab, stage);
        };
        // byte offset of this lane's fragment chunk inside a slab row, per k-step of the slab
        const int fswz = (frag_row / R256) & (VPR - 1);
        const int frow = frag_row * SLAB;
        // One slab: `between` (the requests for the slab that goes into the stage freed last), then step by step this wave's
        // fragments and their MFMAs
        constexpr int KSTEPS      = SLAB / KSTEP / WGK;
        static_assert((SLAB / KSTEP) % WGK == 0, "k-steps of a slab must split evenly over the k-waves");
        auto compute = [&](int stage, auto between) __attribute__((always_inline)) {
            const unsigned char *sa = lds_dyn + stage * STAGE, *sb = sa + BM * SLAB;
            between();
#pragma unroll
            for (int ks = 0; ks < KSTEPS; ++ks) {
                uint4 fa[TM], fb[TN];
                const int chunk = (((wk + ks * WGK) * (64 / BLK) + lane / BLK) ^ fswz) * 16;
#pragma unroll
                for (int i = 0; i < TM; ++i)
                    fa[i] = *reinterpret_cast<const uint4 *>(sa + (wm * TM + i) * BLK * SLAB + frow + chunk);
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    fb[j] = *reinterpret_cast<const uint4 *>(sb + (wn * TN + j) * BLK * SLAB + frow + chunk);
                if constexpr (Epi::kRowStats && !TakesRowSums<Epi>::value) {
                    // the WGN waves that hold the same A rows take turns over the row groups and k-steps
#pragma unroll
                    for (int i = 0; i < TM; ++i)
                        if ((i + ks) % WGN == wn)
                            ln_take(fa[i], i);
                }
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        GemmTraits<DT>::mma(fb[j], fa[i], acc[i][j]);
            }
        };
        constexpr int LPW = A_LD + B_LD;
        // A folding epilogue that is handed the row sums of A: the rows' sums (8 bytes per tile column of the kernel that wrote
        // A) are requested, added up, and {rstd, mean} parked behind everything else in LDS, where the epilogue finds them.  In the early form the loads are spelled as assembly like the
        // slab loads and the wait is placed by hand: the compiler knows nothing of the slabs in flight, and the wait it
        // would place itself (everything outstanding) would also wait for the slabs requested after the sums.  In the
        // late form they are ordinary loads.  When:
        //   late  (tile shapes that have a CU to themselves, hence registers to spare, and any shape when at most twelve
        //         blocks are handed over: 24 registers): once the last slab is in LDS.
        //         Nothing stands between the kernel's entry and its first slabs, the loads' latency passes under the
        //         last slab's MFMAs, and the sums are added up after the loop while the other waves are on their way
        //         to the barrier that follows it.  They are the youngest loads of the kernel: wait for all.
        //   early (shapes that share a CU, with up to 24 blocks: the 48 registers the sums would occupy through the last
        //         slab would cost a resident workgroup): before the first slabs, added up while those are on their way.  Older than
        //         every slab load, they are complete once at most the slab loads are outstanding.
        // Every wave adds up the sums of BM / NW rows, 64 / that many lanes a row, each with its share of the blocks (where the
        // rows of a tile do not divide so, the first BM threads a row each): one wave with 24 loads and 48 additions in double
        // while the others wait for it took 0.5 us of a launch of 6.5 (256 x 2304 x 768).
        typedef float f32x2 __attribute__((ext_vector_type(2)));
        // Two sets of sums of 3 x 6 blocks leave no 24 registers either (eight of them would go to scratch memory).
        constexpr bool kLateSums = TakesRowSums<Epi>::value &&
                                   ((EpiLds<CFG, Epi>::total > 80 * 1024 && !(SETS > 1 && TM * TN >= 18)) || SumBlocks<Epi>::value <= 12);
        constexpr int ROWS_WAVE = BM / CFG::NW;
        constexpr bool SHARED   = ROWS_WAVE == 8 || ROWS_WAVE == 16 || ROWS_WAVE == 32;
        constexpr int LANES_ROW = SHARED ? 64 / ROWS_WAVE : 1;
        constexpr int NSUM      = (SumBlocks<Epi>::value + LANES_ROW - 1) / LANES_ROW;  // blocks of a lane
        const int sum_row  = SHARED ? wave * ROWS_WAVE + lane % ROWS_WAVE : tid;         // row of the tile
        const int sum_part = SHARED ? lane / ROWS_WAVE : 0;
        f32x2 early[NSUM];
        auto request_sums = [&]() __attribute__((always_inline)) {
            if constexpr (TakesRowSums<Epi>::value) {
                if (SHARED || tid < BM) {
                    const int m = m0 + sum_row < M ? m0 + sum_row : M - 1;
#pragma unroll
                    for (int i = 0; i < NSUM; ++i) {
                        // lanes that differ in their block: clamped, and what lies beyond the blocks is not added (a branch by
                        // lane could copy a register before its load has arrived)
                        const int k = i * LANES_ROW + sum_part, q = k < epi.ln.sum_blocks ? k : epi.ln.sum_blocks - 1;
                        if (!SHARED)
                            early[i] = f32x2{0.f, 0.f};
                        if (!SHARED && k >= epi.ln.sum_blocks)
                            continue;
                        if constexpr (kLateSums)
                            // ordinary loads: they are the youngest of the kernel, so the wait the compiler puts in
                            // front of their first use (everything outstanding) is the wait that is wanted, and
                            // the compiler knows the registers are not valid before it
                            early[i] = *reinterpret_cast<const f32x2 *>(
                                reinterpret_cast<const char *>(epi.ln.row_sums) + ((size_t)q * M + m) * sizeof(float2));
                        else
                            asm volatile("global_load_dwordx2 %0, %1, %2"
                                         : "=v"(early[i])
                                         : "v"((uint32_t)(((size_t)q * M + m) * sizeof(float2))), "s"(epi.ln.row_sums)
                                         : "memory");
                    }
                }
            }
        };
        // slab_loads_behind: slab loads requested after the sums that may still be outstanding when the sums are read
        auto finish_sums = [&](int slab_loads_behind) __attribute__((always_inline)) {
            if constexpr (TakesRowSums<Epi>::value) {
                if (SHARED || tid < BM) {
                    if constexpr (!kLateSums) {
                        if (slab_loads_behind >= 2)
                            TR_WAIT_VMCNT(2 * LPW);
                        else if (slab_loads_behind == 1)
                            TR_WAIT_VMCNT(LPW);
                        else
                            TR_WAIT_VMCNT(0);
                    }
                    // The other waves wait at a barrier while these do this, so it is kept short: the block sums (fp32)
                    // are added up in double in a fixed order (the sum of squares of a row that sits far from zero
                    // would lose the variance's digits in fp32), and the reciprocal root of the variance is taken in
                    // single precision with one Newton step.
                    double f1 = 0.0, f2 = 0.0;
#pragma unroll
                    for (int i = 0; i < NSUM; ++i) {
                        if constexpr (!kLateSums)
                            asm volatile("" : "+v"(early[i]));  // not to be read before the wait above
                        if (i * LANES_ROW + sum_part < epi.ln.sum_blocks) {
                            f1 += (double)early[i].x;
                            f2 += (double)early[i].y;
                        }
                    }
                    if constexpr (LANES_ROW >= 8)
                        f1 = add_lane_xor<8>(f1), f2 = add_lane_xor<8>(f2);
                    if constexpr (LANES_ROW >= 4)
                        f1 = add_lane_xor<16>(f1), f2 = add_lane_xor<16>(f2);
                    if constexpr (LANES_ROW >= 2)
                        f1 = add_lane_xor<32>(f1), f2 = add_lane_xor<32>(f2);
                    double mean;
                    const float ve = (float)row_moments(epi.ln, f1, f2, &mean);
                    const float e  = __builtin_amdgcn_rsqf(ve);
                    // an infinite variance has the root 0, and none at all without eps an infinite one
                    const float r  = e > 0.f && e < INFINITY ? e * (1.5f - 0.5f * ve * e * e) : e;
                    if (sum_part == 0)
                        reinterpret_cast<float2 *>(lds_dyn + CFG::lds_bytes)[sum_row] = make_float2(r, (float)mean);
                }
            }
        };
        // Large wave tiles with more than one step a slab: step s + 1's fragments are read between the MFMAs of step s, and so are
        // the first ones of the next slab, whose barrier stands in front of the last step.  Read behind the barrier, they are a
        // burst of all waves' reads that no MFMA covers (256 x 256: 48 KB, 380 of 2400 clocks a slab).  fp16, us, burst -> this:
        // 256 x 256 tiles 8192 x 4096 x 4096 239 -> 228.  Waves with one block of 32 x 32 have nothing to hide the reads behind: 64 x 64
        // tiles 256 x 3072 x 768 6.3 -> 6.6, four waves 985 x 2304 x 768 9.7 -> 10.1.
        constexpr bool PIPE = DT != TNN_ROCM_F32 && CFG::NW == 8 && KSTEPS >= 2 && (TM * TN > 4 || BLK == 16);
        static_assert(!PIPE || KSTEPS % 2 == 0, "two sets of fragments, every slab begins with the first");
        if constexpr (TakesRowSums<Epi>::value && !kLateSums)
            request_sums();
        int issued = 0;
#pragma unroll
        for (int p = 0; p < NS - 1; ++p)
            if (p < nk)
                issue(p, p), ++issued;
        TR_TL(5);  // first slabs requested
        if constexpr (TakesRowSums<Epi>::value && !kLateSums) {
            finish_sums(issued);
            TR_TL(6);  // handed-over row sums added up
        }
        request_ahead();
        int stage = 0, fill = NS - 1;  // stage of slab kt; stage that slab kt + NS - 1 goes to
        // one slab; with_sums (the last slab in the late form) also requests the row sums
        auto step = [&](int kt, auto with_sums) __attribute__((always_inline)) {
            // slab kt has landed once at most the loads of the slabs issued after it are outstanding
            const int behind = nk - 1 - kt;
            if (NS > 2 && behind >= 1)
                TR_WAIT_VMCNT(NS > 2 ? LPW : 0);
            else
                TR_WAIT_VMCNT(0);
            // everyone's part of slab kt is in LDS, and everyone is done reading slab kt - 1 (its fragments were
            // consumed by MFMAs already issued).  A bare barrier: __syncthreads() adds a fence that waits for
            // every outstanding load, the look-ahead ones included.
            __builtin_amdgcn_s_barrier();
            if (kt == 0)
                TR_TL(1);  // first slab landed
            asm volatile("" ::: "memory");  // no LDS access may be moved across the barrier by the compiler
            compute(stage, [&]() __attribute__((always_inline)) {
                if (kt + NS - 1 < nk)
                    issue(kt + NS - 1, fill);
                if constexpr (decltype(with_sums)::value)
                    request_sums();
            });
            stage = stage + 1 == NS ? 0 : stage + 1;
            fill  = fill + 1 == NS ? 0 : fill + 1;
        };
        if constexpr (PIPE) {
            constexpr int READS = TM + TN, MFMAS = TM * TN;
            uint4 fa[2][TM][1], fb[2][TN][1];
            int chunk[KSTEPS];
#pragma unroll
            for (int ks = 0; ks < KSTEPS; ++ks)
                chunk[ks] = frow + (((wk + ks * WGK) * (64 / BLK) + lane / BLK) ^ fswz) * 16;
            auto read_one = [&](int k, int ks, int from) __attribute__((always_inline)) {  // fragment k of step ks
                const unsigned char *at = lds_dyn + from * STAGE + chunk[ks];
                if (k < TM)
                    fa[ks & 1][k < TM ? k : 0][0] = *reinterpret_cast<const uint4 *>(at + (wm * TM + k) * BLK * SLAB);
                else
                    fb[ks & 1][k >= TM ? k - TM : 0][0] = *reinterpret_cast<const uint4 *>(at + BM * SLAB + (wn * TN + k - TM) * BLK * SLAB);
            };
            // slab kt, the first of whose fragments have been read; MORE: another one follows, LOADS: and one is requested; PAIR: the pair
            // of sets that its steps take turns on; FRESH: it begins their sums, with zeros that stand in the matrix instruction (zeroed
            // registers cost 0.35 us of the 8.7 of 3072 x 768 x 768, with four sets of nine blocks)
            // The sets but the first two are added up behind the last slab's matrix instructions, the two that are left where the epilogue
            // stages them.
            static_assert(SETS == 1 || KSTEPS == 2, "two steps a slab");
            constexpr bool FOLDS = CFG::FOLDS && SETS == 2;
            Acc total[FOLDS ? TM : 1][FOLDS ? TN : 1];
            auto slab = [&](int kt, auto more, auto loads, auto pair, auto fresh) __attribute__((always_inline)) {
                constexpr bool MORE = decltype(more)::value, LOADS = decltype(loads)::value;
                constexpr bool FRESH = decltype(fresh)::value;
                constexpr int PAIR   = SETS == 4 ? decltype(pair)::value : 0;
                const int here = stage, next = stage + 1 == NS ? 0 : stage + 1;
#pragma unroll
                for (int ks = 0; ks < KSTEPS; ++ks) {
                    const bool last = ks == KSTEPS - 1;
                    if (last && MORE) {
                        // this wave's fragments of slab kt are in registers; slab kt + 1 has landed once at most the loads of
                        // the slabs requested after it are outstanding
                        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                        if (NS > 2 && kt + 2 < nk)
                            TR_WAIT_VMCNT(NS > 2 ? LPW : 0);
                        else
                            TR_WAIT_VMCNT(0);
                        __builtin_amdgcn_s_barrier();
                        asm volatile("" ::: "memory");
                    }
                    if (last && !MORE && kLateSums)
                        request_sums();
                    if constexpr (Epi::kRowStats && !TakesRowSums<Epi>::value) {
#pragma unroll
                        for (int i = 0; i < TM; ++i)
                            if ((i + ks) % WGN == wn)
                                ln_take(fa[ks & 1][i][0], i);
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int q = 0; q < MFMAS; ++q) {
                        Acc &sum = parts[SETS > 1 ? 2 * PAIR + ks : 0][q / TN][q % TN];
                        if constexpr (FRESH)
                            sum = Acc{};
                        GemmTraits<DT>::mma(fb[ks & 1][q % TN][0], fa[ks & 1][q / TN][0], sum);
                        __builtin_amdgcn_sched_barrier(0);
                        if constexpr (!MORE && SETS == 4)
                            parts[2 - 2 * ks][q / TN][q % TN] += parts[3 - ks][q / TN][q % TN];
                        if (!last || MORE) {
#pragma unroll
                            for (int k = READS * q / MFMAS; k < READS * (q + 1) / MFMAS; ++k)
                                read_one(k, last ? 0 : ks + 1, last ? next : here);
                        }
                        if (last && LOADS) {
#pragma unroll
                            for (int k = LPW * q / MFMAS; k < LPW * (q + 1) / MFMAS; ++k)
                                issue_one(k, kt + NS, here);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                stage = next;
            };
            {
                static_assert(NS <= 3, "waits written for up to three stages");
                if (NS > 2 && nk > 1)
                    TR_WAIT_VMCNT(NS > 2 ? LPW : 0);
                else
                    TR_WAIT_VMCNT(0);
                __builtin_amdgcn_s_barrier();
                TR_TL(1);  // first slab landed
                asm volatile("" ::: "memory");
#pragma unroll
                for (int k = 0; k < READS; ++k)
                    read_one(k, 0, 0);
                // the last stage's slab only now: all workgroups start together, and what they request ahead stands in the way
                // of one another's first slabs
                if (NS - 1 < nk)
                    issue(NS - 1, NS - 1);
            }
            typedef std::integral_constant<int, 0> First;
            typedef std::integral_constant<int, 1> Second;
            typedef std::true_type Yes;
            typedef std::false_type No;
            int kt = 0;
            constexpr int PER_FOLD = 768 / KB;
            const bool folds = FOLDS && nk >= PER_FOLD + NS;  // the loop that requests others has slab PER_FOLD - 1
            if constexpr (SETS > 1) {
                constexpr int LEAD = SETS / 2;  // slabs that begin the sets
                if (LEAD - 1 + NS < nk) {
                    slab(0, Yes(), Yes(), First(), Yes());
                    if constexpr (SETS == 4)
                        slab(1, Yes(), Yes(), Second(), Yes());
                    kt = LEAD;
                } else {
#pragma unroll
                    for (int p = 0; p < SETS; ++p)
                        clear(parts[p]);
                }
                if constexpr (FOLDS)
                    if (folds)
                        clear(total);
            }
            if constexpr (SETS == 4)
                for (; kt + 1 + NS < nk; kt += 2) {
                    slab(kt, Yes(), Yes(), First(), No());
                    slab(kt + 1, Yes(), Yes(), Second(), No());
                }
            int to_fold = folds ? PER_FOLD - kt : nk;
            for (; kt + NS < nk; ++kt) {
                slab(kt, Yes(), Yes(), First(), No());
                if constexpr (FOLDS)
                    if (--to_fold == 0) {
                        to_fold = PER_FOLD;
                        add_to(total, parts[0]), add_to(total, parts[1]);
                        clear(parts[0]), clear(parts[1]);
                    }
            }
            for (; kt + 1 < nk; ++kt)
                slab(kt, Yes(), No(), Second(), No());
            slab(kt, No(), No(), First(), No());
            if constexpr (FOLDS)
                if (folds)
                    add_to(parts[0], total);
            if constexpr (kLateSums) {
                finish_sums(0);
                TR_TL(6);  // handed-over row sums added up
            }
        } else if constexpr (kLateSums) {
            // the last slab apart, so that the requested sums cross no loop edge on their way to the wait
            for (int kt = 0; kt + 1 < nk; ++kt)
                step(kt, std::false_type());
            step(nk - 1, std::true_type());
            finish_sums(0);
            TR_TL(6);  // handed-over row sums added up
        } else if constexpr (DT == TNN_ROCM_F32) {
            typedef SplitSlab<TM, TN, KSTEPS> Planes;
            Planes p, q;
            static_assert(DT != TNN_ROCM_F32 || NS == 2, "one slab is requested while the one before is multiplied");
            // slab kt in LDS, and every wave done with slab kt - 1; its fragments
            auto fetch = [&](int kt, typename Planes::Reads &rd) __attribute__((always_inline)) {
                // slab kt - 1 is in this wave's registers, see the barrier below
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                TR_WAIT_VMCNT(0);
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                const unsigned char *sa = lds_dyn + stage * STAGE, *sb = sa + BM * SLAB;
#pragma unroll
                for (int ks = 0; ks < KSTEPS; ++ks)
#pragma unroll
                    for (int h = 0; h < FRAGS; ++h) {
                        const int chunk = ((((wk + ks * WGK) * FRAGS + h) * 2 + (lane >> 5)) ^ fswz) * 16;
#pragma unroll
                        for (int i = 0; i < TM; ++i)
                            rd.f[ks][i][h] = *reinterpret_cast<const uint4 *>(sa + (wm * TM + i) * 32 * SLAB + frow + chunk);
#pragma unroll
                        for (int j = 0; j < TN; ++j)
                            rd.f[ks][TM + j][h] = *reinterpret_cast<const uint4 *>(sb + (wn * TN + j) * 32 * SLAB + frow + chunk);
                    }
            };
            auto advance = [&]() __attribute__((always_inline)) {
                stage = stage + 1 == NS ? 0 : stage + 1;
                fill  = fill + 1 == NS ? 0 : fill + 1;
            };
            auto half = [&](int kt, const Planes &now, Planes &next, auto loads) __attribute__((always_inline)) {
                typename Planes::Reads rd;
                fetch(kt, rd);
                const int there = fill;
                advance();
                now.template turn<decltype(loads)::value, false>(
                    rd, next, acc, split_const, [&](int k) __attribute__((always_inline)) { issue_one(k, kt + NS - 1, there); });
            };
            typedef std::integral_constant<int, LPW> WithLoads;
            typedef std::integral_constant<int, 0> NoLoads;
            {
                typename Planes::Reads rd;
                fetch(0, rd);
                if (NS - 1 < nk)
                    issue(NS - 1, fill);
                advance();
                p.convert(rd, split_const);
            }
            int kt = 1;
            for (; kt + NS < nk; kt += 2) {
                half(kt, p, q, WithLoads());
                half(kt + 1, q, p, WithLoads());
            }
            // the last slabs: one more to request at most
            if (kt + NS - 1 < nk) {
                half(kt, p, q, WithLoads());
                p = q;
                ++kt;
            }
            for (; kt + 1 < nk; kt += 2) {
                half(kt, p, q, NoLoads());
                half(kt + 1, q, p, NoLoads());
            }
            if (kt < nk) {
                half(kt, p, q, NoLoads());
                q.multiply(acc);
            } else {
                p.multiply(acc);
            }
        } else {
            for (int kt = 0; kt < nk; ++kt)
                step(kt, std::false_type());
        }
    } else {
    u32x4 ra0[A_VECS], rb0[B_VECS], ra1[A_VECS], rb1[B_VECS];

    // Loads carry no bounds branches: rows past the matrix edge are clamped to the last row (their products
    // land in accumulators that the epilogue never stores) and K is a whole number of slabs (checked by the
    // launcher), so every global load of a slab can be in flight at once.
    // vector v = tid + i*NT sits in slab row v / VPR at 16-byte column v % VPR; NT is a multiple of VPR, so
    // the column is the same for every i and the row advances by NT / VPR
    constexpr int ROW_STEP = NT / VPR;
    const int vrow = tid / VPR, vcol = tid % VPR;
    uint32_t a_off[A_VECS], b_off[B_VECS];  // element offsets (the launcher checks they fit 32 bits)
#pragma unroll
    for (int i = 0; i < A_VECS; ++i) {
        int row  = m0 + vrow + i * ROW_STEP;
        row      = row < M ? row : M - 1;
        a_off[i] = (uint32_t)row * (uint32_t)lda + (uint32_t)(vcol * VEC);
    }
#pragma unroll
    for (int i = 0; i < B_VECS; ++i) {
        int row  = n0 + vrow + i * ROW_STEP;
        row      = row < N ? row : N - 1;
        b_off[i] = (uint32_t)row * (uint32_t)ldb + (uint32_t)(vcol * VEC);
    }
// The three pipeline stages are macros on purpose: passing the register arrays through lambdas kept them in
// scratch memory (the compiler did not promote them), which costs more than the prefetch gains.
#define TR_LOAD_GLOBAL(RA, RB, K0)                                                                                    \
    {                                                                                                                 \
        _Pragma("unroll") for (int i = 0; i < A_VECS; ++i) RA[i] =                                                    \
            *reinterpret_cast<const u32x4 *>(A + a_off[i] + (K0));                                                    \
        _Pragma("unroll") for (int i = 0; i < B_VECS; ++i) RB[i] =                                                    \
            *reinterpret_cast<const u32x4 *>(B + b_off[i] + (K0));                                                    \
    }
#define TR_STORE_LDS(BUF, RA, RB)                                                                                     \
    {                                                                                                                 \
        _Pragma("unroll") for (int i = 0; i < A_VECS; ++i) *reinterpret_cast<u32x4 *>(                                \
            lds_a##BUF + (vrow + i * ROW_STEP) * STRIDE + vcol * 16) = RA[i];                                         \
        _Pragma("unroll") for (int i = 0; i < B_VECS; ++i) *reinterpret_cast<u32x4 *>(                                \
            lds_b##BUF + (vrow + i * ROW_STEP) * STRIDE + vcol * 16) = RB[i];                                         \
    }
#define TR_COMPUTE(BUF)                                                                                               \
    {                                                                                                                 \
        _Pragma("unroll") for (int kk = wk; kk < SLAB / 32; kk += WGK) {                                              \
            uint4 fa[TM], fb[TN];                                                                                     \
            _Pragma("unroll") for (int i = 0; i < TM; ++i) fa[i] = *reinterpret_cast<const uint4 *>(                  \
                lds_a##BUF + ((wm * TM + i) * 32 + frag_row) * STRIDE + kk * 32 + frag_off);                          \
            _Pragma("unroll") for (int j = 0; j < TN; ++j) fb[j] = *reinterpret_cast<const uint4 *>(                  \
                lds_b##BUF + ((wn * TN + j) * 32 + frag_row) * STRIDE + kk * 32 + frag_off);                          \
            _Pragma("unroll") for (int i = 0; i < TM; ++i) _Pragma("unroll") for (int j = 0; j < TN; ++j)             \
                GemmTraits<DT>::mma(fb[j], fa[i], acc[i][j]); /* rows of D = n, lanes of D = m */                     \
        }                                                                                                             \
    }

    unsigned char *const lds_a0 = lds_dyn, *const lds_b0 = lds_dyn + BM * STRIDE;
    unsigned char *const lds_a1 = lds_dyn + (BM + BN) * STRIDE, *const lds_b1 = lds_a1 + BM * STRIDE;

    // Slab schedule (two slabs in flight in registers, one in LDS being consumed).  The loop body is branch
    // free: look-ahead loads past the last slab are clamped to it and their LDS copy is never consumed.
    // (Forcing the look-ahead loads to the top of each phase with sched_barrier was measured slower: the
    // compiler's own interleaving of loads, LDS traffic and MFMAs is kept.)
    const int last = (nk - 1) * KB;
#define TR_CLAMPK(SLABIDX) (((SLABIDX)*KB) < last ? ((SLABIDX)*KB) : last)
    TR_LOAD_GLOBAL(ra0, rb0, 0);
    TR_LOAD_GLOBAL(ra1, rb1, TR_CLAMPK(1));
    request_ahead();
    TR_STORE_LDS(0, ra0, rb0);
    __syncthreads();
    for (int kt = 0; kt + 2 <= nk; kt += 2) {
        TR_LOAD_GLOBAL(ra0, rb0, TR_CLAMPK(kt + 2));
        TR_COMPUTE(0);
        TR_STORE_LDS(1, ra1, rb1);
        __syncthreads();
        TR_LOAD_GLOBAL(ra1, rb1, TR_CLAMPK(kt + 3));
        TR_COMPUTE(1);
        TR_STORE_LDS(0, ra0, rb0);
        __syncthreads();
    }
    if (nk & 1)
        TR_COMPUTE(0);
#undef TR_LOAD_GLOBAL
#undef TR_STORE_LDS
#undef TR_COMPUTE
#undef TR_CLAMPK
    }

    if constexpr (DT == TNN_ROCM_F32 && CFG::NSTAGE > 0) {
        constexpr int STEPS = SLAB / 64, REGS = BLK * BLK / 64;  // steps of 16 values of k per slab
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                float size = 0.f;
#pragma unroll
                for (int r = 0; r < REGS; ++r)
                    size += __builtin_fabsf(acc[i][j][r]);
#pragma unroll
                for (int r = 0; r < REGS; ++r)
                    acc[i][j][r] *= kSplitUnscale;
                if (__all(split_finite(size)))
                    continue;
                // clamped as the slabs' rows are
                const int ra = m0 + (wm * TM + i) * BLK + frag_row, rb = n0 + (wn * TN + j) * BLK + frag_row;
                const T *pa = A + (size_t)(ra < M ? ra : M - 1) * lda + BLK / 4 * (lane / BLK);
                const T *pb = B + (size_t)(rb < N ? rb : N - 1) * ldb + BLK / 4 * (lane / BLK);
                if constexpr (CFG::OWN)
                    multiply_again(pa, pb, nk * wk / WGK * STEPS, nk * (wk + 1) / WGK * STEPS, 1, acc[i][j]);
                else
                    multiply_again(pa, pb, wk, nk * STEPS, WGK, acc[i][j]);
            }
    }

    typedef typename std::remove_reference<decltype(acc[0][0][0])>::type AccT;
    // Row-contiguous epilogue.  In the accumulator layout one store instruction touches 32 rows with 16 bytes
    // each, i.e. 32 partial cache lines; the L2 then sees eight times as many write requests as there are lines.
    // For each 32-row group every wave writes its 32 x CW accumulator block to its own LDS region (the slab
    // buffers are free after the main loop); the workgroup then walks the staged rows with eight columns per
    // thread, adds the WGK partial sums and applies the epilogue, so a store instruction covers whole lines of C
    // and bias/residual are read in the same coalesced shape.
    constexpr int SSTR = CFG::SSTR;     // staged row stride in 32-bit words (16-byte pad spreads the b128 banks)
    typedef AccT acc4 __attribute__((ext_vector_type(4)));
    AccT *const stage_all = reinterpret_cast<AccT *>(lds_dyn);
    AccT *const stage_me  = stage_all + wave * (GROWS * SSTR);  // wave = (wm*WGN + wn)*WGK + wk
    const int tid_piece = tid % CPR, tid_rowpos = tid / CPR;
    __syncthreads();  // every wave is done reading the slabs
    TR_TL(2);         // main loop done
    // LayerNorm-folding epilogues: reduce the lanes' partial row sums over the two k-halves of a fragment and the WGK
    // k-waves (fixed order), giving {rstd, mean} per tile row; both arrays sit behind the staging area
    float2 *const row_st   = reinterpret_cast<float2 *>(lds_dyn + (TakesRowSums<Epi>::value ? CFG::lds_bytes : CFG::stage_bytes));  // [BM]
    double2 *const row_part = reinterpret_cast<double2 *>(row_st + BM);               // [WGK * WGN][BM]
    int8_t *const lut_lds = reinterpret_cast<int8_t *>(lds_dyn + CFG::stage_bytes);  // Int8Epilogue's table, 256 bytes
    if constexpr (std::is_same<Epi, Int8Epilogue>::value) {
        if (epi.lut && tid < 64)
            reinterpret_cast<uint32_t *>(lut_lds)[tid] = reinterpret_cast<const uint32_t *>(epi.lut)[tid];
        // read after the first staging barrier below
    }
    // the tile's columns of the epilogue's per-column arrays, and its rows' pairs: read after the first staging barrier
    float *const col_lds        = reinterpret_cast<float *>(lds_dyn + EpiLds<CFG, Epi>::col_offset);
    const float2 *const row_lds = reinterpret_cast<const float2 *>(lds_dyn + EpiLds<CFG, Epi>::row_offset);
    if constexpr (ColArrays<Epi>::value > 0) {
        if constexpr (!EARLY)
            request_columns();
#pragma unroll
        for (int q = 0; q < COLQ; ++q)
            if (q * NT + tid < ColArrays<Epi>::value * BN)
                col_lds[q * NT + tid] = early_col[q];
    }
    if constexpr (RowIn<Epi>::value) {
        if (tid < BM)
            reinterpret_cast<float2 *>(lds_dyn + EpiLds<CFG, Epi>::row_offset)[tid] = early_row;
    }
    if constexpr (Epi::kRowStats && TakesRowSums<Epi>::value) {
        // {rstd, mean} were parked in LDS before the main loop (the barrier above orders that write); hand them on
        if (epi.ln.stats && n0 == 0 && tid < BM && m0 + tid < M)
            store_out8(epi.through, &epi.ln.stats[m0 + tid], row_st[tid]);
    }
    if constexpr (Epi::kRowStats && !TakesRowSums<Epi>::value) {
        static_assert(CFG::NSTAGE > 0, "LayerNorm-folding epilogues run on the direct-to-LDS pipeline");
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            double s1 = add_lane_xor<32>(ln_s1[i]), s2 = add_lane_xor<32>(ln_s2[i]);
            if constexpr (BLK == 16)
                s1 = add_lane_xor<16>(s1), s2 = add_lane_xor<16>(s2);
            if (lane < BLK)
                row_part[(wk * WGN + wn) * BM + (wm * TM + i) * BLK + frag_row] = make_double2(s1, s2);
        }
        __syncthreads();
        if (tid < BM) {
            double s1 = 0.0, s2 = 0.0;
            for (int q = 0; q < WGK * WGN; ++q) {
                const double2 v = row_part[q * BM + tid];
                s1 += v.x;
                s2 += v.y;
            }
            double mean;
            const double var = row_moments(epi.ln, s1, s2, &mean);
            const float2 st  = make_float2((float)reciprocal_root(var), (float)mean);
            row_st[tid]      = st;
            if (epi.ln.stats && n0 == 0 && m0 + tid < M)  // every tile column holds them; the first one hands them on
                store_out8(epi.through, &epi.ln.stats[m0 + tid], st);
        }
        // row_st is read after the first staging barrier below
    }
    // The LayerNorm output y is written at the very end from this tile's own share of its rows of A; the vectors it
    // needs are requested here, once the last accumulators have been staged, so their latency hides under the
    // remaining epilogue instead of standing alone at the kernel's tail.
    constexpr int YPRE = 3;  // vectors a thread holds ahead (192 x 192 tiles: 12 rows x K/8 groups over 512 threads)
    u32x4 y_pre[Epi::kRowStats ? YPRE : 1];
    int y_r0 = 0, y_items = 0, y_groups = 1;
    if constexpr (Epi::kRowStats) {
        if (epi.ln.y) {
            const int tn = n0 / BN;
            y_groups     = K / 8;
            y_r0         = (int)((long)tn * BM / tiles_n);
            y_items      = ((int)((long)(tn + 1) * BM / tiles_n) - y_r0) * y_groups;
        }
    }
#pragma unroll
    for (int i = 0; i < GROUPS; ++i) {
        if constexpr (BLK == 32) {
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4)
                    *reinterpret_cast<acc4 *>(stage_me + (lane & 31) * SSTR + j * 32 + 8 * r4 + 4 * (lane >> 5)) =
                        acc4{acc[i][j][r4 * 4 + 0], acc[i][j][r4 * 4 + 1], acc[i][j][r4 * 4 + 2], acc[i][j][r4 * 4 + 3]};
        } else {
#pragma unroll
            for (int b = 0; b < TM / GROUPS; ++b)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    acc4 sums = acc[i * (TM / GROUPS) + b][j];
                    if constexpr (SETS > 1)
                        sums += parts[1][i * (TM / GROUPS) + b][j];
                    *reinterpret_cast<acc4 *>(stage_me + (b * 16 + (lane & 15)) * SSTR + j * 16 + 4 * (lane >> 4)) = sums;
                }
        }
        if constexpr (Epi::kRowStats) {
            if (i == GROUPS - 1) {
#pragma unroll
                for (int q = 0; q < YPRE; ++q) {
                    const int item = tid + q * NT;
                    if (epi.ln.y_ahead && item < y_items) {
                        const int m = m0 + y_r0 + item / y_groups;
                        if (m < M)
                            y_pre[q] = *reinterpret_cast<const u32x4 *>(A + (size_t)m * lda + (item % y_groups) * 8);
                    }
                }
            }
        }
        __syncthreads();
        // Waited for on every path: where a path passes their use by, the compiler waits where the paths meet, and there it waits for
        // the result's store too, 960 clocks in front of the row sums.
#pragma unroll
        for (int q = 0; q < MY_ITEMS * AHEAD; ++q)
            asm volatile("" : "+v"(ahead_vec[q / (AHEAD > 0 ? AHEAD : 1)][q % (AHEAD > 0 ? AHEAD : 1)]));
#pragma unroll
        for (int it = 0; it < MY_ITEMS; ++it) {
            const int item = it * NT + tid;
            if (ITEMS % NT != 0 && item >= ITEMS)
                break;
            // consecutive threads walk along a row of C, or down the rows where the epilogue writes a transposed
            // layout (consecutive rows are then consecutive in memory)
            // item % CPR and item / CPR: where CPR is not a power of two (96-column wave tiles) the thread index is
            // split once and every item adds its constant share, instead of a multiply-high sequence per item
            int piece, rowpos;
            if constexpr ((CPR & (CPR - 1)) != 0) {
                const int c     = tid_piece + (it * NT) % CPR;
                const int carry = c >= CPR ? 1 : 0;
                piece           = c - carry * CPR;
                rowpos          = tid_rowpos + (it * NT) / CPR + carry;
            } else {
                piece  = item % CPR;
                rowpos = item / CPR;
            }
            const int c8  = by_rows ? ((item / GROWS) % CPR) * 8 : piece * 8;
            const int row = by_rows ? (item % GROWS) : rowpos % GROWS;
            const int pos = rowpos / GROWS;  // = item / (CPR * GROWS) = pm * WGN + pn
            const AccT *src = stage_all + (pos * WGK) * (GROWS * SSTR) + row * SSTR + c8;
            acc4 lo = *reinterpret_cast<const acc4 *>(src);
            acc4 hi = *reinterpret_cast<const acc4 *>(src + 4);
#pragma unroll
            for (int q = 1; q < WGK; ++q) {
                lo += *reinterpret_cast<const acc4 *>(src + q * (GROWS * SSTR));
                hi += *reinterpret_cast<const acc4 *>(src + q * (GROWS * SSTR) + 4);
            }
            const int m = m0 + ((pos / WGN) * GROUPS + i) * GROWS + row;
            const int n = n0 + (pos % WGN) * CW + c8;
            const int nl = (pos % WGN) * CW + c8;  // column inside the tile
            const u32x4 *const ahead = AHEAD > 0 ? ahead_vec[it] : nullptr;
            if constexpr (Epi::kRowStats) {
                if (m < M && n + 7 < N) {  // N is a multiple of 8 for these epilogues (checked at launch)
                    AccT v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                    epi.store8(m, n, v, row_st[m - m0], col_lds + nl, BN, ahead);
                }
            } else if constexpr (EmitsRowSums<Epi>::value) {
                // N is a multiple of 8 for these epilogues (checked at launch); every item leaves its eight columns'
                // sums, zero where nothing is stored, so that the totals below see a fully written array
                float2 sm = make_float2(0.f, 0.f);
                if (m < M && n + 7 < N) {
                    AccT v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                    sm = epi.store8(m, n, v, col_lds + nl, BN, row_lds[m - m0], ahead);
                }
                if constexpr (CFG::sums_by_lanes) {
                    static_assert((CPR == 2 || CPR == 4 || CPR == 8) && (ITEMS % NT == 0 || ITEMS <= NT),
                                  "so many neighbouring lanes hold a row, and all of them have an item or none");
                    sm.x = add_neighbours<CPR>(sm.x);
                    sm.y = add_neighbours<CPR>(sm.y);
                    if (piece == 0 && m < M && n < N)
                        store_out8(epi.through, &epi.row_sums[(size_t)(n / CFG::sum_cols) * M + m], sm);
                } else {
                    *reinterpret_cast<float2 *>(const_cast<AccT *>(src)) = sm;
                }
            } else if (m < M) {
                AccT v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                if (n + 7 < N) {
                    if constexpr (std::is_same<Epi, Int8Epilogue>::value)
                        epi.store8(m, n, v, epi.lut ? lut_lds : nullptr, col_lds + nl, BN, ahead);
                    else if constexpr (RowIn<Epi>::value)
                        (void)epi.store8(m, n, v, col_lds + nl, BN, row_lds[m - m0], ahead);
                    else if constexpr (ColArrays<Epi>::value > 0)
                        epi.store8(m, n, v, col_lds + nl, BN, ahead);
                    else
                        epi.store8(m, n, v);
                } else {
                    // the last columns one at a time, from LDS again: eight copies of the epilogue were a third of the library
#pragma unroll 1
                    for (int t = 0; t < 8; ++t)
                        if (n + t < N) {
                            AccT x = src[t];
#pragma unroll
                            for (int q = 1; q < WGK; ++q)
                                x += src[q * (GROWS * SSTR) + t];
                            epi.store(m, n + t, x, epi.col_const(n + t));
                        }
                }
            }
        }
        if (i + 1 < GROUPS)
            __syncthreads();
    }
    TR_TL(3);  // C stored
    if constexpr (EmitsRowSums<Epi>::value && !CFG::sums_by_lanes) {
        // This tile's share of every row's sum and sum of squares, added up in a fixed order, for the folding GEMM that reads C next.
        // LANES neighbouring lanes share a row.  Tiles of 128 columns and more add in double, so that their pairs are rounded once and the
        // variance is as exact as from pairs of 64 columns (in fp32 rows far from zero had up to twice the error); narrower ones need not,
        // and it would cost 0.3 us of the 8 to 23 of theirs.
        typedef typename std::conditional<(BN > 96), double, float>::type Sum;
        constexpr int SPLIT = NT / BM, LANES = SPLIT >= 8 ? 8 : SPLIT >= 4 ? 4 : 2;
        static_assert(SPLIT >= 2 && BM * LANES % 64 == 0 && BN / 8 % LANES == 0, "whole waves, every lane with as many pairs");
        __syncthreads();
        if (tid < BM * LANES) {
            const int row   = tid / LANES;
            const AccT *src = stage_all + (row / GROWS * WGN * WGK) * (GROWS * SSTR) + row % GROWS * SSTR;
            Sum s1 = 0, s2 = 0;
#pragma unroll
            for (int q = 0; q < BN / 8; q += LANES) {
                const int piece   = q + tid % LANES;
                const float2 part = *reinterpret_cast<const float2 *>(src + (piece / CPR * WGK) * (GROWS * SSTR) + piece % CPR * 8);
                s1 += (Sum)part.x, s2 += (Sum)part.y;
            }
            s1 = add_neighbours<LANES>(s1), s2 = add_neighbours<LANES>(s2);
            if (tid % LANES == 0 && m0 + row < M)
                store_out8(epi.through, &epi.row_sums[(size_t)(n0 / BN) * M + m0 + row], make_float2((float)s1, (float)s2));
        }
    }
    if constexpr (Epi::kRowStats) {
        // y = LayerNorm(t) for this tile's share of its rows (the BM rows are dealt out evenly over the tile columns, so
        // every workgroup writes whole rows), in the LayerNorm kernel's half-precision form
        // x * rstd * gamma + (beta - mean * rstd * gamma)
        if (epi.ln.y) {
            typedef typename GemmTraits<DT>::elem TY;
            const int groups = y_groups, r0 = y_r0;
            int q = 0;
            for (int item = tid; item < y_items; item += NT, ++q) {
                const int row = r0 + item / groups, c = (item % groups) * 8, m = m0 + row;
                if (m >= M)
                    continue;
                const float2 st = row_st[row];
                const float mrs = st.y * st.x;
                float4 k0 = *reinterpret_cast<const float4 *>(epi.ln.gamma + c), k1 = *reinterpret_cast<const float4 *>(epi.ln.gamma + c + 4);
                float4 e0 = *reinterpret_cast<const float4 *>(epi.ln.beta + c), e1 = *reinterpret_cast<const float4 *>(epi.ln.beta + c + 4);
                const float kk[8] = {k0.x, k0.y, k0.z, k0.w, k1.x, k1.y, k1.z, k1.w};
                const float ee[8] = {e0.x, e0.y, e0.z, e0.w, e1.x, e1.y, e1.z, e1.w};
                u32x4 raw;
                if (epi.ln.y_ahead && q == 0)
                    raw = y_pre[0];
                else if (epi.ln.y_ahead && q == 1 && YPRE > 1)
                    raw = y_pre[YPRE > 1 ? 1 : 0];
                else if (epi.ln.y_ahead && q == 2 && YPRE > 2)
                    raw = y_pre[YPRE > 2 ? 2 : 0];
                else
                    raw = *reinterpret_cast<const u32x4 *>(A + (size_t)m * lda + c);
                TY *pe = reinterpret_cast<TY *>(&raw);
#pragma unroll
                for (int t = 0; t < 8; ++t)
                    Elem<DT>::st(&pe[t], Elem<DT>::ld(&pe[t]) * st.x * kk[t] + (ee[t] - mrs * kk[t]));
                *reinterpret_cast<u32x4 *>(reinterpret_cast<TY *>(epi.ln.y) + (size_t)m * K + c) = raw;
            }
        }
    }
    TR_TL(4);  // kernel end
}

// internal: the chosen tile shape does not leave row sums (256 x 256 tiles, staged in halves; more blocks of columns than a reader adds
// up) or does not take them; the caller launches the form without
constexpr int kNotWithRowSums = -12345;
thread_local int t_last_sum_blocks = 0;  // row-sum blocks of this thread's last tiled launch

template <int DT, typename CFG, typename Epi>
int launch_shape(hipStream_t s, const void *A, const void *B, int M, int N, int K, long lda, long ldb, const Epi &epi) {
    typedef typename GemmTraits<DT>::elem T;
    int tiles_m = (M + CFG::BM - 1) / CFG::BM, tiles_n = (N + CFG::BN - 1) / CFG::BN;
    typedef EpiLds<CFG, Epi> L;
    const size_t lds = L::total;
    const int sum_blocks = (N + CFG::sum_cols - 1) / CFG::sum_cols;
    if (EmitsRowSums<Epi>::value && sum_blocks > kMaxRowSumBlocks)
        return kNotWithRowSums;
    auto kern   = gemm_nk_tiled_kernel<DT, CFG, Epi>;
    if (lds > 64 * 1024) {
        // the attribute belongs to the (kernel, device) pair: one bit per device, per instantiation
        static std::atomic<unsigned long long> attr_set{0};
        int dev = 0;
        TR_CHECK_HIP(hipGetDevice(&dev));
        const unsigned long long bit = 1ull << (dev & 63);
        if (dev > 63 || !(attr_set.load(std::memory_order_acquire) & bit)) {
            TR_CHECK_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
            attr_set.fetch_or(bit, std::memory_order_release);
        }
    }
    // tiles resident together on one XCD (32 CUs): a square-ish group keeps their panels in that L2
    const long lds_per_cu = 160 * 1024;
    long per_cu   = lds_per_cu / (long)(lds + 1024);
    per_cu        = per_cu < 1 ? 1 : (per_cu > 4 ? 4 : per_cu);
    long resident = 32 * per_cu, per_xcd = ((long)tiles_m * tiles_n + 7) / 8;
    resident      = resident < per_xcd ? resident : per_xcd;
    int forced_group = g_gemm_group_m;
    if (forced_group <= 0)
        tune_override(N, K, &forced_group);
    int group_m   = forced_group > 0 ? forced_group : 1;
    if (forced_group <= 0)
        while ((long)(group_m + 1) * (group_m + 1) <= resident)
            ++group_m;
    group_m = group_m > tiles_m ? tiles_m : group_m;
    group_m = group_m > TileOrder::kMaxRows ? TileOrder::kMaxRows : group_m;
    const TileOrder order = TileOrder::of(tiles_m, tiles_n, group_m);
    unsigned grid = (unsigned)(((tiles_m * tiles_n + 7) / 8) * 8);
    t_last_sum_blocks = sum_blocks;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(CFG::NT), lds, s, (const T *)A, (const T *)B, M, N, K, (int)lda, (int)ldb,
                       order.group, order.rows, order.last_rows, order.packed, epi);
    TR_CHECK_LAUNCH();
    return 0;
}

template <int DT, typename CFG, typename Epi>
int launch_tiled(hipStream_t s, const void *A, const void *B, int M, int N, int K, long lda, long ldb, const Epi &epi) {
    if constexpr (EmitsRowSums<Epi>::value && !CFG::leaves_sums)
        return kNotWithRowSums;
    else
        return launch_shape<DT, CFG, Epi>(s, A, B, M, N, K, lda, ldb, epi);
}

// Configuration codes: [P] TM TN WGM WGN WGK S (one decimal digit each; slab bytes = 64 << S; P = number of
// direct-to-LDS stages, 9 = rings of the waves' own, absent = slabs staged through registers).
//   9111141   32 x  32, 4 k-waves with rings of their own     9121141   32 x  64, likewise
//   6111141   16 x  16, 6211141 32 x 16, 6121141 16 x 32: 16 x 16 blocks, 4 k-waves with rings of their own (three slabs)
//   3112221   64 x  64, 8 waves (two k-waves), 3 stages       2112211   64 x  64, 4 waves, 2 stages
//   7 and 8 (two and three stages): 16 x 16 blocks, 8 waves that share the slabs
//   8222222   64 x  64, 8322222 96 x 64, 8332222 96 x 96, 8422222 128 x 64: 2 x 2 positions and two k-waves, 256-byte slabs
//   7244211  128 x 128, 8244211 128 x 128, 8344211 192 x 128, 8364211 192 x 192: 4 x 2 positions; not int8: 8264211 128 x 192, 8444211 256 x 128
//   7484211  256 x 256: 4 x 2 positions
//   fp32 only: 6111181, 6211181 16 x 16 and 32 x 16, 8 k-waves; 9111181 32 x 32, 8 k-waves; 9221141 64 x 64, 4 k-waves with rings of their own;
//   2321142, 2231142, 2331142 96 x 64, 64 x 96 and 96 x 96, 4 k-waves; 2222121, 2332121 128 x 64 and 192 x 96, 4 waves (two k-waves);
//   2222221 128 x 128, 8 waves (two k-waves)
//   112210    64 x  64 and 222210 128 x 128, 4 waves: rows that are no multiple of 128 bytes
// Eight-wave workgroups put two waves on every SIMD inside one tile: while one waits for its LDS fragments the
// other issues MFMAs, and a larger tile per CU moves fewer bytes through LDS and L2 per flop.  Four-wave tiles
// larger than 128 x 128 (one wave per SIMD) were measured and never won with compiler-scheduled code.

// What a launch takes on this chip with each tile shape.  The busiest CU works through n = ceil(tiles / 256) tiles, up to
// `slots` of them side by side (what its LDS and registers hold): full sets of `slots`, then the rest.  A set costs its
// number of 128-byte k-slabs times slab[its tiles - 1], every set after the first also `round` (ramp and epilogue that
// nothing covers), and the launch `fixed`; microseconds.  The figures are a least-squares fit to some 800 launches (fp16 and
// int8: M from 16 to 8192, the four projections of hidden sizes 768 and 1024 with their fused epilogues; fp32: M from 16 to
// 3072), taken over twelve weight sets in turn so that weights come from the memory-side cache as they do inside a network:
// python -m tnn_amd.bench_ops --tile-sweep measures them and fits the rows.  A launch is 3 .. 20 % off its prediction on average,
// by shape (the large ones most), so picks closer than that are as good as drawn.  The half and int8 rows were then moved by hand as
// little as it took for few launches to be slower than with the tables and shapes before them; by hand altogether: 256 x 256 in both, and in
// the int8 table 128 x 128 (the second tile's slab of two stages, the round of three), 192 x 128 and 192 x 192.  The picks are 0.5 %
// (fp16, int8) and 0.9 .. 1.6 % (fp32, two sweeps) behind the best shape of each launch at hidden sizes 768 and 1024, at worst 5, 6 and 8 %; at 256
// to 2048 0.6 (fp16) and 0.8 % (int8), at worst 32 % (QKV of 12288 x 1536 x 512) and 13 %: profiles/gemm_tile_choice.txt, with the launches
// that are furthest behind, and inside the network.  Against the tables and shapes of 32 x 32 blocks, over 448 launches of each type
// (hidden sizes 256 to 2048, M from 16 to 12288), they take 0.939 (fp16) and 0.948 (int8) of the time
// in the mean, six and four of them 5 .. 10 % more.
// The rules this replaced, made for M >= 1024, were 51 %, 34 % and 77 % behind:
//   M=  32 N= 768 K=3072 fp16  23.1 -> 7.3 us   (64x64 tiles: 12 CUs, one two-stage slab after another)
//   M= 256 N= 768 K=3072 fp16  23.7 -> 7.2      M= 256 N=2304 K=768 fp16  8.7 -> 6.2
//   M=1000 N= 768 K=3072 fp16  24.3 -> 12.4     M=1000 N= 768 K=768 fp16  8.7 -> 5.5
struct TileCost {
    int code, bm, bn, slots;
    float fixed, round, slab[4];
};
constexpr TileCost kTilesHalf[] = {
    {6111141, 16, 16, 3, 3.45f, 1.51f, {0.027f, 0.067f, 0.092f}},
    {6211141, 32, 16, 2, 3.43f, 2.01f, {0.040f, 0.089f}},
    {6121141, 16, 32, 2, 3.37f, 1.74f, {0.046f, 0.095f}},
    {9111141, 32, 32, 2, 3.39f, 1.89f, {0.064f, 0.139f}},
    {9121141, 32, 64, 1, 3.54f, 2.58f, {0.113f}},
    {3112221, 64, 64, 3, 3.86f, 2.73f, {0.207f, 0.344f, 0.616f}},
    {2112211, 64, 64, 4, 3.04f, 1.86f, {0.411f, 0.480f, 0.573f, 0.855f}},
    {8222222, 64, 64, 1, 3.69f, 2.83f, {0.154f}},
    {8322222, 96, 64, 1, 4.38f, 3.65f, {0.192f}},
    {8332222, 96, 96, 1, 5.21f, 5.31f, {0.242f}},
    {8422222, 128, 64, 1, 4.48f, 4.16f, {0.239f}},
    {7244211, 128, 128, 2, 3.87f, 6.00f, {0.594f, 0.920f}},
    {8244211, 128, 128, 1, 4.81f, 6.73f, {0.358f}},
    {8264211, 128, 192, 1, 7.38f, 10.11f, {0.482f}},
    {8344211, 192, 128, 1, 6.59f, 8.74f, {0.465f}},
    {8364211, 192, 192, 1, 8.80f, 12.52f, {0.666f}},
    {8444211, 256, 128, 1, 7.77f, 11.65f, {0.596f}},
    {7484211, 256, 256, 1, 11.80f, 13.30f, {1.145f}},
};
// 256 x 256 tiles are for products that fill the chip with them: half the bytes a flop of 128 x 128 tiles.  A linear model knows
// neither that a round of 192 tiles is 13 % shorter than one of 256 nor what the epilogue leaves uncovered, so their row and the
// epilogues' wide_us() are fitted to the comparison with the other shapes' picks: 1155 launches of 185 products (1024 to 24576 rows,
// hidden sizes 256 to 4096).  With {10.0, 8.0, 1.6} for every epilogue 91 of the 839 that took 256 x 256 tiles were more than 3 %
// slower for it, by up to 21 %; now 15 of 888, by up to 9 %.  us, 128 x 128 -> 256 x 256, folded LayerNorm and GELU: 8192 x 4096 x 1024
// 89 -> 81, 4096 x 4096 x 1024 47 -> 42, 3072 x 4096 x 1024 37.3 -> 35.7 (with a bias only 34.8 -> 31.1); not picked 12288 x 3072 x 768
// 82 -> 92, 4096 x 3072 x 768 29.6 -> 31.1, 8192 x 1536 x 384 21.1 -> 22.7.  With twelve weight sets in turn, over 260 launches, the
// picks that are slower cost 25 % together (187 % with the old row), the shape where it is left out and faster 88 % (99 %).  The int8
// row is set by hand: of its picks three of 60 are slower, 24576 x 1920 x 640 into Q, K and V^T by 6 % and [16384, 1024] x 1024 and
// 24576 x 1280 x 1280 with a residual by 3 %.  That was with 32 x 32 blocks, whose row was {10.5, 12.0, 1.255} (int8 {10.5, 8.2, 2.049}).
// As 16 x 16 blocks a step's products are twice as many of half the length, between which the next step's reads spread finer, and
// the loop is 4 .. 11 % faster; the tile is staged in two halves instead of two blocks' rows.  us: 16384 x 4096 x 1024 with GELU
// 145.5 -> 138.6, 16384 x 1024 x 4096 115 -> 102, 8192 x 8192 x 8192 890 -> 838, bf16 839 -> 795, int8 16384 x 1024 x 4096 72.1 -> 66.6,
// 16384 x 4096 x 1024 103.0 -> 96.6, 8192 x 4096 x 4096 144.6 -> 136.6.  The half row's slab is smaller by that and its other two figures larger
// by twelve slabs of it, so that the line stays where it is at K = 768 (with 1.165 alone K = 512 lost 10 %) and moves with K.  The int8 row, and with it
// the second slab of two 128 x 128 tiles a CU (1.148, 10 % above what it measures at K of 3072 and up), are set to order the shapes
// from 128 x 128 on as they measure; us, the picks before and these, each with its own shapes: 8192 x 768 x 3072 31.0 -> 27.0,
// 4096 x 4096 x 4096 83.1 -> 65.8, 12288 x 1280 x 5120 96.9 -> 76.7.
// GELU adds 2.5 us a round of 256 x 256 tiles in this model, 1.75 before 128 x 128 tiles were of 16 x 16 blocks: with that,
// products moved to them whose sums the tiles before had in two parts (TileCfg), and that are no faster for it: 4096 x 3072 x 768
// 28.4 us, with 128 x 128 tiles 26.8, 6400 x 4096 x 1024 66.3 and 67.3.
// 16 x 16 blocks of a shared slab.  Up to 128 x 64: eight waves as 2 x 2 positions and two k-waves, so that a tile of any number of 32
// rows and columns is dealt out evenly.  96 x 96 as eight k-waves of 3 x 3 blocks of 32 x 32 passed 295 KB of partial sums through
// LDS behind its loop (half of the 11 us of 3072 x 768 x 768), now 74; 96 x 64 is one round of the chip where 64 x 64 are two.
// From 128 x 128 on: 4 x 2 positions and no k-waves.  The waves' blocks are longer than high, which costs half more LDS reads than square
// ones (12 KB a wave and slab of 128 x 128, not 8), but the sums pass through LDS once instead of twice and the fragments of a step are
// read under the products of the step before, across the slab's barrier too.  us, the picks before -> these:
//   fp16 3072 x 768 x 768 10.9 -> 8.8, 3072 x 768 x 3072 22.9 -> 20.1, 1536 x 768 x 3072 18.8 -> 14.5, 984 x 768 x 3072 13.0 -> 11.8,
//   700 x 3072 x 768 10.9 -> 8.3, 3072 x 3072 x 768 22.9 -> 21.1, 2048 x 2304 x 768 16.9 -> 14.4, 8192 x 3072 x 1024 77.2 -> 70.8,
//   8192 x 1024 x 4096 79.7 -> 70.7; int8 1536 x 768 x 3072 11.8 -> 9.3, 3072 x 768 x 3072 15.5 -> 13.2
// (Not taken: 64 x 96, 32 x 64, 64 x 32,
// 32 x 96, 64 x 128 with two k-waves, 0.1 % of the sweep together; 96 x 96 with two stages 8.9 -> 9.9 or four k-waves 9.1 -> 9.4;
// 128 x 64 and 192 x 96 with 4 x 2 positions, 0.1 % together; 128 x 256, the same as 256 x 128.)
// Tiles of 16 x 16 blocks with rings of the waves' own are for the products whose 32x32 tiles are too few for the chip: a CU's panels come through its L1 at
// 64 bytes a clock at best, so 24 tiles of (32 + 32) rows of K=3072 take 4 us for that alone, and 96 of (16 + 16) rows half.
// us a launch, best shape before -> now (fp32: 8 waves where K is long):
//   M= 32 N= 768 K=3072 fp16  7.4 -> 5.0   int8 5.0 -> 4.1   fp32 14.9 -> 8.8     M= 32 N=768 K=768 fp16 3.9 -> 3.2, fp32 6.4 -> 4.6
//   M=128 N= 768 K=3072 fp16  7.5 -> 6.0   int8 5.4 -> 4.7   fp32 14.9 -> 12.1    M=128 N=768 K=768 fp16 4.3 -> 3.5, fp32 6.7 -> 5.8
//   M= 32 N=2304 K=768  fp16  4.7 -> 4.5 (folded LayerNorm)  fp32  6.7 -> 5.9
// (Measured and not taken: eight waves for fp16 and int8, 0.1 .. 0.4 us behind; rings of four slabs, 0.1 behind.)
constexpr TileCost kTilesI8[] = {
    {6111141, 16, 16, 3, 3.21f, 1.59f, {0.031f, 0.071f, 0.084f}},
    {6211141, 32, 16, 2, 3.17f, 1.60f, {0.047f, 0.093f}},
    {6121141, 16, 32, 2, 3.13f, 1.58f, {0.051f, 0.092f}},
    {9111141, 32, 32, 2, 3.17f, 1.63f, {0.070f, 0.139f}},
    {9121141, 32, 64, 1, 3.29f, 2.09f, {0.123f}},
    {3112221, 64, 64, 3, 3.25f, 1.79f, {0.210f, 0.375f, 0.655f}},
    {2112211, 64, 64, 4, 2.68f, 1.77f, {0.426f, 0.565f, 0.562f, 0.874f}},
    {8222222, 64, 64, 1, 3.20f, 2.27f, {0.165f}},
    {8322222, 96, 64, 1, 3.92f, 3.17f, {0.206f}},
    {8332222, 96, 96, 1, 4.96f, 4.41f, {0.271f}},
    {8422222, 128, 64, 1, 3.66f, 3.60f, {0.271f}},
    {7244211, 128, 128, 2, 3.92f, 3.61f, {0.632f, 1.040f}},
    {8244211, 128, 128, 1, 4.99f, 12.00f, {0.418f}},
    {8344211, 192, 128, 1, 6.60f, 9.50f, {0.543f}},
    {8364211, 192, 192, 1, 8.95f, 12.02f, {0.850f}},
    {7484211, 256, 256, 1, 13.00f, 10.70f, {1.700f}},
};
// fp32 on three bf16 planes: six matrix instructions per operand pair and the conversion between them, so a step costs five
// times a half one.  Large wave tiles convert less per product, K is split over the waves of a CU wherever tiles are few, and
// two stages are enough where the next slab's loads are the first thing that follows a slab's barrier (turn() in SplitSlab).
// Fit and sweep as above (M from 16 to 3072, hidden size 768).
// us, v_mfma_f32 kernels -> planes, a whole plane of four values behind a matrix instruction -> a pair of values:
//   M=1536: N=768 K=768 27 -> 20.2 -> 17.3, N=3072 K=768 74 -> 61 -> 55, N=768 K=3072 83 -> 60 -> 51
//   M=128: N=768 K=768 7.6 -> 7.1 -> 6.8, N=3072 K=768 15.2 -> 11.4 -> 10.7, N=768 K=3072 17.6 -> 16.2 -> 15.3
// (the 16 x 16 blocks, which came after that, see above, not counted).  Since the dot products stand together (SplitSlab; six sets
// of weights in turn): M=1536 20.3 -> 19.2, 56.2 -> 52, 58.1 -> 54; M=128 6.8 -> 6.6, 12.1 -> 11.7, 13.5 -> 13.2.  The figures
// below are from before; with them the choice is 0.45 % from the best shape in the mean (192 launches, 16 to 3072 rows, hidden sizes
// 512 to 1024; fitted again 0.32 %).
// Error against float64 (2-norm over 2-norm; 300 x 760 x 768 / 129 x 264 x 3072): 1.5e-7 .. 3e-7 / 3e-7 .. 6e-7 by shape,
// v_mfma_f32_32x32x2_f32: 5.0e-7 / 9.9e-7.
constexpr TileCost kTilesF32[] = {
    {6111141, 16, 16, 3, 3.80f, 1.14f, {0.054f, 0.107f, 0.164f}},
    {6211141, 32, 16, 2, 3.83f, 1.35f, {0.089f, 0.184f}},
    {6121141, 16, 32, 2, 4.03f, 1.50f, {0.086f, 0.178f}},
    {6111181, 16, 16, 1, 3.71f, 2.33f, {0.053f}},
    {6211181, 32, 16, 1, 3.97f, 2.67f, {0.086f}},
    {9111141, 32, 32, 2, 3.92f, 1.81f, {0.115f, 0.253f}},
    {9121141, 32, 64, 1, 4.69f, 4.59f, {0.199f}},
    {9111181, 32, 32, 1, 4.27f, 3.31f, {0.120f}},
    {9221141, 64, 64, 1, 6.03f, 7.55f, {0.312f}},
    {2321142, 96, 64, 1, 5.69f, 9.55f, {0.445f}},
    {2231142, 64, 96, 1, 6.64f, 10.54f, {0.442f}},
    {2331142, 96, 96, 1, 8.12f, 15.53f, {0.619f}},
    {2222121, 128, 64, 2, 5.87f, 11.44f, {0.593f, 1.378f}},
    {2222221, 128, 128, 1, 7.53f, 20.38f, {1.065f}},
    {2332121, 192, 96, 1, 9.10f, 25.11f, {1.177f}},
};

// row_stats: the shape takes the rows' statistics from its own A fragments, which 32 rows of 16 x 16 blocks pay for with twice the
// sums a wave (32 rows, hidden sizes 768 and 1024: QKV 4.7 and 5.0 us, FFN1 4.9 and 5.3; with 16 x 32 tiles 4.4, 4.7, 4.6 and 4.9)
template <int COUNT>
inline int pick_tile_config(const TileCost (&shapes)[COUNT], long M, long N, size_t kbytes, bool row_stats, float wide_us) {
    int best        = 0;
    float best_cost = 0.f;
    const float slabs = (float)(kbytes / 128);
    for (const TileCost &t : shapes) {
        if (kbytes % (64u << (t.code % 10)) != 0)
            continue;
        const long tiles = ((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn), n = (tiles + kNumCU - 1) / kNumCU;
        const long sets = n / t.slots, rest = n % t.slots;
        float cost = t.fixed + slabs * ((float)sets * t.slab[t.slots - 1] + (rest ? t.slab[rest - 1] : 0.f)) +
                     t.round * (float)(sets + (rest ? 1 : 0) - 1) + (row_stats && t.code / 100000 == 62 ? 0.4f : 0.f) +
                     (t.bm == 256 && t.bn == 256 ? wide_us * (float)n : 0.f);
        if (best == 0 || cost < best_cost)
            best = t.code, best_cost = cost;
    }
    return best;
}

template <int DT, typename Epi>
int launch_gemm_fast(hipStream_t s, const void *A, const void *B, int M, int N, int K, long lda, long ldb,
                     const Epi &epi) {
    typedef typename GemmTraits<DT>::elem T;
    const int forced = g_gemm_force_cfg;
    int cfg       = forced > 0 ? forced : tune_override(N, K, nullptr);
    size_t kbytes = (size_t)K * sizeof(T);
    // direct-to-LDS loads address a panel with a 32-bit byte offset
    const bool wide = (size_t)M * lda * sizeof(T) >= (1ull << 32) || (size_t)N * ldb * sizeof(T) >= (1ull << 32);
    if (cfg == 0) {
        if (kbytes % 128 != 0 || wide)
            cfg = (((long)M + 127) / 128) * (((long)N + 127) / 128) > kNumCU ? 222210 : 112210;
        else if (DT == TNN_ROCM_F32)
            cfg = pick_tile_config(kTilesF32, M, N, kbytes, Epi::kRowStats, WideEpilogue<Epi>::us(epi));
        else if (DT == TNN_ROCM_I8)
            cfg = pick_tile_config(kTilesI8, M, N, kbytes, Epi::kRowStats, WideEpilogue<Epi>::us(epi));
        else
            cfg = pick_tile_config(kTilesHalf, M, N, kbytes, Epi::kRowStats, WideEpilogue<Epi>::us(epi));
    }
    switch (cfg) {  // a code of 128-byte or larger slabs without its stage digit
        case 112211: cfg = 2112211; break;
        case 222221:
        case 224211: cfg = 2222221; break;
        case 332221: cfg = 3332221; break;
        case 331182: cfg = 3331182; break;
        default: break;
    }
    if constexpr (DT != TNN_ROCM_F32) {
        switch (cfg) {  // codes of shapes that are no more: the same tile in slabs that every K of theirs is a whole number of
            case 2222221: cfg = 7244211; break;
            case 3332221: cfg = 8364211; break;
            case 2244211: cfg = 7484211; break;
            case 3331182: cfg = 8332222; break;
            case 3112222: cfg = 8222222; break;
            case 4221141: cfg = kbytes % 256 == 0 ? 8222222 : 3112221; break;
            case 3212221: cfg = kbytes % 256 == 0 ? 8422222 : 7244211; break;  // (128 x 64 has 256-byte slabs only)
            default: break;
        }
    }
    if (kbytes % (64u << (cfg % 10)) != 0) {
        set_error("gemm: K=%d is not a whole number of slabs for tuning configuration %d", K, cfg);
        return TNN_ROCM_ESHAPE;
    }
#define TR_FAST(TMv, TNv, WGMv, WGNv, WGKv, SLABv)                                                                    \
    return launch_tiled<DT, TileCfg<TMv, TNv, WGMv, WGNv, WGKv, SLABv>, Epi>(s, A, B, M, N, K, lda, ldb, epi)
#define TR_FAST_DL(TMv, TNv, WGMv, WGNv, WGKv, SLABv, NSv)                                                            \
    return launch_tiled<DT, TileCfg<TMv, TNv, WGMv, WGNv, WGKv, SLABv, NSv>, Epi>(s, A, B, M, N, K, lda, ldb, epi)
#define TR_FAST_DL16(TMv, TNv, WGMv, WGNv, WGKv, SLABv, NSv, ...)                                                     \
    return launch_tiled<DT, TileCfg<TMv, TNv, WGMv, WGNv, WGKv, SLABv, NSv, false, 16, __VA_ARGS__>, Epi>(s, A, B, M, N, K, lda, ldb, epi)
#define TR_FAST_SMALL(TMv, TNv, WGKv, SLABv, NSv)                                                                     \
    return launch_tiled<DT, TileCfg<TMv, TNv, 1, 1, WGKv, SLABv, NSv, true, 16>, Epi>(s, A, B, M, N, K, lda, ldb, epi)
#define TR_FAST_OWN(TMv, TNv, WGKv, SLABv, NSv)                                                                       \
    return launch_tiled<DT, TileCfg<TMv, TNv, 1, 1, WGKv, SLABv, NSv, true>, Epi>(s, A, B, M, N, K, lda, ldb, epi)
    if constexpr (TakesRowSums<Epi>::value) {
        if (cfg >= 9000000 || (cfg >= 6000000 && cfg < 7000000))
            return kNotWithRowSums;
    } else {
        switch (cfg) {
            case 9111141: TR_FAST_OWN(1, 1, 4, 128, 2);
            case 9121141: TR_FAST_OWN(1, 2, 4, 128, 2);
            default: break;
        }
        switch (cfg) {
            case 6111141: TR_FAST_SMALL(1, 1, 4, 128, 3);
            case 6211141: TR_FAST_SMALL(2, 1, 4, 128, 3);
            case 6121141: TR_FAST_SMALL(1, 2, 4, 128, 3);
            default: break;
        }
        if constexpr (DT == TNN_ROCM_F32) {
            switch (cfg) {
                case 6111181: TR_FAST_SMALL(1, 1, 8, 128, 3);
                case 6211181: TR_FAST_SMALL(2, 1, 8, 128, 3);
                default: break;
            }
        }
    }
    if constexpr (DT == TNN_ROCM_F32) {
        switch (cfg) {
            case 9111181: TR_FAST_OWN(1, 1, 8, 128, 2);
            case 9221141: TR_FAST_OWN(2, 2, 4, 128, 2);
            case 2321142: TR_FAST_DL(3, 2, 1, 1, 4, 256, 2);
            case 2231142: TR_FAST_DL(2, 3, 1, 1, 4, 256, 2);
            case 2331142: TR_FAST_DL(3, 3, 1, 1, 4, 256, 2);
            case 2222121: TR_FAST_DL(2, 2, 2, 1, 2, 128, 2);
            case 2332121: TR_FAST_DL(3, 3, 2, 1, 2, 128, 2);
            case 2222221: TR_FAST_DL(2, 2, 2, 2, 2, 128, 2);
            default: break;
        }
    } else {
        switch (cfg) {
            case 2112211: TR_FAST_DL(1, 1, 2, 2, 1, 128, 2);
            case 3112221: TR_FAST_DL(1, 1, 2, 2, 2, 128, 3);
            case 7244211: TR_FAST_DL16(2, 4, 4, 2, 1, 128, 2, 2);
            case 8244211: TR_FAST_DL16(2, 4, 4, 2, 1, 128, 3, 4);
            case 8344211:
                if (DT != TNN_ROCM_I8 && kbytes >= 4096)
                    TR_FAST_DL16(3, 4, 4, 2, 1, 128, 3, 2, DT != TNN_ROCM_I8);
                TR_FAST_DL16(3, 4, 4, 2, 1, 128, 3, 2);
            case 8364211: TR_FAST_DL16(3, 6, 4, 2, 1, 128, 3, 2);
            case 7484211: TR_FAST_DL16(4, 8, 4, 2, 1, 128, 2, 1);
            case 8222222: TR_FAST_DL16(2, 2, 2, 2, 2, 256, 3, 2);
            case 8322222: TR_FAST_DL16(3, 2, 2, 2, 2, 256, 3, 2);
            case 8332222: TR_FAST_DL16(3, 3, 2, 2, 2, 256, 3, 4);
            case 8422222: TR_FAST_DL16(4, 2, 2, 2, 2, 256, 3, 2);
            default: break;
        }
        if constexpr (DT != TNN_ROCM_I8) {
            switch (cfg) {
                case 8264211: TR_FAST_DL16(2, 6, 4, 2, 1, 128, 3, 2);
                case 8444211: TR_FAST_DL16(4, 4, 4, 2, 1, 128, 3, 2);
                default: break;
            }
        }
    }
    if constexpr (!Epi::kRowStats) {  // the LayerNorm-folding epilogues exist for the direct-to-LDS pipelines only
        switch (cfg) {
            case 112210: TR_FAST(1, 1, 2, 2, 1, 64);
            case 222210: TR_FAST(2, 2, 2, 2, 1, 64);
            default: break;
        }
    }
#undef TR_FAST_OWN
#undef TR_FAST_SMALL
#undef TR_FAST_DL16
#undef TR_FAST
#undef TR_FAST_DL
    set_error("gemm: unknown tuning configuration %d", cfg);
    return TNN_ROCM_EINVAL;
}

template <int DT, int BM, int BN, int WM, int WN, typename Epi>
int launch_gemm_cfg(hipStream_t s, bool b_nk, bool aligned, const void *A, const void *B, int M, int N, int K, long lda,
                    long ldb, int batch, int batch_a, int batch_b, long stride_a, long stride_b, const Epi &epi) {
    typedef typename GemmTraits<DT>::elem T;
    int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    dim3 grid((unsigned)(tiles_m * tiles_n), (unsigned)batch), block(WM * WN * 64);
#define TR_GEMM_LAUNCH(NK, AL)                                                                                        \
    hipLaunchKernelGGL((gemm_kernel<DT, BM, BN, WM, WN, NK, AL, Epi>), grid, block, 0, s, (const T *)A, (const T *)B, \
                       M, N, K, lda, ldb, batch_a, batch_b, stride_a, stride_b, tiles_m, tiles_n, epi)
    if (b_nk) {
        if (aligned)
            TR_GEMM_LAUNCH(true, true);
        else
            TR_GEMM_LAUNCH(true, false);
    } else {
        if (aligned)
            TR_GEMM_LAUNCH(false, true);
        else
            TR_GEMM_LAUNCH(false, false);
    }
#undef TR_GEMM_LAUNCH
    TR_CHECK_LAUNCH();
    return 0;
}

// Tile choice: 128x128 when that still yields at least ~1.5 waves of workgroups over the 256 CUs,
// otherwise 128x64 / 64x64 so small-N projections keep the chip busy.
template <int DT, typename Epi>
int launch_gemm(hipStream_t s, bool b_nk, bool aligned, const void *A, const void *B, int M, int N, int K, long lda,
                long ldb, int batch, int batch_a, int batch_b, long stride_a, long stride_b, const Epi &epi) {
    auto tiles = [&](int bm, int bn) { return (long)((M + bm - 1) / bm) * ((N + bn - 1) / bn) * batch; };
    if (tiles(128, 128) >= 384)
        return launch_gemm_cfg<DT, 128, 128, 2, 2, Epi>(s, b_nk, aligned, A, B, M, N, K, lda, ldb, batch, batch_a,
                                                        batch_b, stride_a, stride_b, epi);
    if (tiles(128, 64) >= 256)
        return launch_gemm_cfg<DT, 128, 64, 2, 2, Epi>(s, b_nk, aligned, A, B, M, N, K, lda, ldb, batch, batch_a,
                                                       batch_b, stride_a, stride_b, epi);
    return launch_gemm_cfg<DT, 64, 64, 2, 2, Epi>(s, b_nk, aligned, A, B, M, N, K, lda, ldb, batch, batch_a, batch_b,
                                                  stride_a, stride_b, epi);
}

}  // namespace

// ---- one launch per entry point and type: the argument checks are in gemm.hip ----------------------------------------------
template <int DT> int GemmTyped<DT>::plain(hipStream_t s, bool b_is_nk, const void *A, const void *B, void *C, int M, int N,
                                           int K, int lda, int ldb, int ldc, int batch, int batch_a, int batch_b,
                                           int epilogue, const float *bias, const void *residual, int ldr) {
    typedef typename Elem<DT>::type T;
    constexpr int VEC = 16 / sizeof(T);
    const long sa = (long)M * lda, sb = (long)(b_is_nk ? N : K) * ldb;
    const bool aligned = al16(A) && al16(B) && lda % VEC == 0 && ldb % VEC == 0 && K % VEC == 0 && (b_is_nk || N % VEC == 0) &&
                         (batch == 1 || (sa % VEC == 0 && sb % VEC == 0));
    FloatEpilogue<DT> epi;
    epi.flags          = epilogue;
    epi.bias           = bias;
    epi.residual       = (const T *)residual;
    epi.ldr            = ldr;
    epi.C              = (T *)C;
    epi.ldc            = ldc;
    epi.batch_stride_c = (long)M * ldc;
    epi.batch_stride_r = (long)M * ldr;
    const bool vec_out = N % 4 == 0 && ldc % VEC == 0 && al16(C) &&
                         (!(epilogue & TNN_ROCM_EPI_RESIDUAL) || (ldr % VEC == 0 && al16(residual))) &&
                         (!(epilogue & TNN_ROCM_EPI_BIAS) || al16(bias));
    if (b_is_nk && aligned && batch == 1 && vec_out && g_gemm_force_cfg >= 0 && (K * sizeof(T)) % 64 == 0)
        return launch_gemm_fast<DT, FloatEpilogue<DT>>(s, A, B, M, N, K, lda, ldb, epi);
    return launch_gemm<DT, FloatEpilogue<DT>>(s, b_is_nk, aligned, A, B, M, N, K, lda, ldb, batch, batch_a, batch_b, sa, sb, epi);
}

template <int DT> int GemmTyped<DT>::qkv_split(hipStream_t s, const void *x, const void *wqkv, const float *bqkv, void *qk,
                                               void *vt, int B, int S, int heads, int K, int vt_key_order) {
    const int H = heads * 64, T = B * S;
    QkvSplitEpilogue<DT> epi;
    epi.bias  = bqkv;
    epi.qk    = (typename Elem<DT>::type *)qk;
    epi.vt    = (typename Elem<DT>::type *)vt;
    epi.H     = H;
    epi.S     = S;
    epi.heads = heads;
    epi.vt_sh = vt_key_order;
    return launch_gemm_fast<DT, QkvSplitEpilogue<DT>>(s, x, wqkv, T, 3 * H, K, K, K, epi);
}

template <int DT, int SUMS>
int launch_ln(hipStream_t s, const void *t, const void *w_folded, const float *bias_folded, void *C, const LnFold &ln, int M,
              int N, int K, int flags, const void *residual) {
    LnFloatEpilogue<DT, SUMS> epi;
    epi.flags    = flags;
    epi.bias     = bias_folded;
    epi.residual = (const typename Elem<DT>::type *)residual;
    epi.C        = (typename Elem<DT>::type *)C;
    epi.ldc      = N;
    epi.ln       = ln;
    return launch_gemm_fast<DT, LnFloatEpilogue<DT, SUMS>>(s, t, w_folded, M, N, K, K, K, epi);
}

template <int DT>
int GemmTyped<DT>::ln(hipStream_t s, const void *t, const void *w_folded, const float *bias_folded, const float *colsum,
                      const float *gamma, const float *beta, float eps, void *C, void *y, float *row_stats,
                      const float *row_sums, int row_sum_blocks, int M, int N, int K, int flags, const void *residual) {
    const LnFold ln{(double)K, 1.0 / (double)K, eps, colsum, gamma, beta, y, g_ln_y_ahead.load(), (float2 *)row_stats,
                    (const float2 *)row_sums, row_sum_blocks};
    int rc = kNotWithRowSums;  // a tile shape that takes the statistics from its own tiles declines handed-over sums
    if (row_sums && row_sum_blocks <= 12)
        rc = launch_ln<DT, 12>(s, t, w_folded, bias_folded, C, ln, M, N, K, flags, residual);
    else if (row_sums)
        rc = launch_ln<DT, kMaxRowSumBlocks>(s, t, w_folded, bias_folded, C, ln, M, N, K, flags, residual);
    return rc == kNotWithRowSums ? launch_ln<DT, 0>(s, t, w_folded, bias_folded, C, ln, M, N, K, flags, residual) : rc;
}

template <int DT, int SUMS>
int launch_qkv_split_ln(hipStream_t s, const void *t, const void *wqkv_folded, const float *bqkv_folded, void *qk, void *vt,
                        const LnFold &ln, int B, int S, int heads, int K, int vt_key_order) {
    const int H = heads * 64, T = B * S;
    LnQkvSplitEpilogue<DT, SUMS> epi;
    epi.bias  = bqkv_folded;
    epi.qk    = (typename Elem<DT>::type *)qk;
    epi.vt    = (typename Elem<DT>::type *)vt;
    epi.H     = H;
    epi.S     = S;
    epi.heads = heads;
    epi.vt_sh = vt_key_order;
    epi.ln    = ln;
    return launch_gemm_fast<DT, LnQkvSplitEpilogue<DT, SUMS>>(s, t, wqkv_folded, T, 3 * H, K, K, K, epi);
}

template <int DT>
int GemmTyped<DT>::qkv_split_ln(hipStream_t s, const void *t, const void *wqkv_folded, const float *bqkv_folded,
                                const float *colsum, const float *gamma, const float *beta, float eps, void *qk, void *vt,
                                void *y, float *row_stats, const float *row_sums, int row_sum_blocks, int B, int S, int heads,
                                int K, int vt_key_order) {
    const LnFold ln{(double)K, 1.0 / (double)K, eps, colsum, gamma, beta, y, g_ln_y_ahead.load(), (float2 *)row_stats,
                    (const float2 *)row_sums, row_sum_blocks};
    int rc = kNotWithRowSums;
    if (row_sums && row_sum_blocks <= 12)
        rc = launch_qkv_split_ln<DT, 12>(s, t, wqkv_folded, bqkv_folded, qk, vt, ln, B, S, heads, K, vt_key_order);
    else if (row_sums)
        rc = launch_qkv_split_ln<DT, kMaxRowSumBlocks>(s, t, wqkv_folded, bqkv_folded, qk, vt, ln, B, S, heads, K, vt_key_order);
    if (rc != kNotWithRowSums)
        return rc;
    return launch_qkv_split_ln<DT, 0>(s, t, wqkv_folded, bqkv_folded, qk, vt, ln, B, S, heads, K, vt_key_order);
}

template <int DT, bool SUMS>
int launch_residual_ln(hipStream_t s, const void *x, const void *w, const float *bias, void *C, const void *t,
                       const float *row_stats, const float *gamma, const float *beta, int M, int N, int K, int flags,
                       float *row_sums) {
    LnResidualEpilogue<DT, SUMS> epi;
    epi.row_sums = (float2 *)row_sums;
    epi.flags    = flags;
    epi.bias     = bias;
    epi.t        = (const typename Elem<DT>::type *)t;
    epi.st       = (const float2 *)row_stats;
    epi.gamma    = gamma;
    epi.beta     = beta;
    epi.C        = (typename Elem<DT>::type *)C;
    epi.ldc      = N;
    return launch_gemm_fast<DT, LnResidualEpilogue<DT, SUMS>>(s, x, w, M, N, K, K, K, epi);
}

template <int DT>
int GemmTyped<DT>::residual_ln(hipStream_t s, const void *x, const void *w, const float *bias, void *C, const void *t,
                               const float *row_stats, const float *gamma, const float *beta, int M, int N, int K, int flags,
                               float *row_sums, int *row_sum_blocks) {
    // With the row sums first.  A tile shape whose blocks of columns are more than a reader adds up (and the caller's buffer of
    // kMaxRowSumBlocks * M pairs holds: 16 columns wide from N = 385 on, 32 columns wide from N = 769 on) declines in launch_shape, one
    // that leaves no sums (256 x 256) in launch_tiled; the plain form runs then and reports zero blocks.
    if (row_sums && N <= 64 * kMaxRowSumBlocks) {
        const int rc = launch_residual_ln<DT, true>(s, x, w, bias, C, t, row_stats, gamma, beta, M, N, K, flags, row_sums);
        if (rc == 0)
            *row_sum_blocks = t_last_sum_blocks;
        if (rc != kNotWithRowSums)
            return rc;
    }
    return launch_residual_ln<DT, false>(s, x, w, bias, C, t, row_stats, gamma, beta, M, N, K, flags, nullptr);
}

}  // namespace tnn_rocm
#endif
