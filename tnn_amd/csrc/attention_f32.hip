// Fused attention core in fp32: out = softmax(Q K^T * scale + mask) V, head_dim 64, so that the layers of the decomposed
// graph (head-splitting copies, two batched products, scaling, mask, softmax, head-merging copy: ten launches that write and
// read the [B*h, S, S] scores six times) become one kernel.  The replaced layers: cpu_mat_mul_layer_acc.cc,
// cpu_softmax_layer_acc.cc, cpu_permute_layer_acc.cc of the reference.
//
// Both products run on three bf16 planes per value (split_f32.h); scale, mask, exponentials, sums and the running rescale
// stay in fp32.  One workgroup = one (batch, head, block of 32 queries).  Its four waves take every fourth block of 32 keys
// each, with a running maximum and sum of their own, and are merged through LDS at the end: short sequences have few
// (batch, head, query block) triples (48 for one sequence of 128 tokens with 12 heads), and this way each of them keeps the
// four SIMDs of its CU busy.  Waves share no keys, so K and V go from memory (L2) straight into the fragment registers: K a
// row per lane, V two neighbouring columns per lane.
//
// Layout as in attention.hip: S^T = K Q^T, so a lane holds one query column and 16 of the 32 keys (register r of lane half g
// is key 8*(r/4) + 4*g + r%4), and the probabilities are in the register order that the second product O^T = V^T P^T wants,
// given V rows in that order.  Row i of block dt of O^T is column d = 2*i + dt of the head.
//
// An infinity, a NaN or a finite value from 2^104 on has no planes (split_f32.h) and makes every sum it enters something that is
// not finite, as a sum beyond 2^80 becomes by itself.  A workgroup that finds such a sum does its block again
// with the fp32 matrix instruction, operands straight from memory (`exact` below): the answer is then that of the layers in
// fp32 arithmetic.  The check is 33 instructions a wave.
//
// What bounds it: the vector ALU (4.5 instructions for each of the 80 values of K, P and V that a lane converts for a block, 10 for
// each of its 17 exponentials; 57 % of all clocks at 16 x 384 tokens, the matrix pipe 25 %, when it was 7) once a SIMD has three waves, and the
// latency of a block's chain below that.  So: three waves a SIMD (the planes of Q are made once per workgroup and lie in LDS, a
// block's rows are requested when the registers of the rows before are free), no work for the mask in blocks that are whole, and
// requests that every path to their waits makes alike, or the compiler waits for V where K is meant.
// us, 12 heads, in a row: the decomposed launches -> Q's planes in registers, two waves a SIMD -> this form
//   1 x 128 tokens 45 -> 6.9 -> 6.4, 4 x 384 136 -> 29.1 -> 26.2 (with an additive mask 38 -> 28), 16 x 384 79 -> 73, 1 x 16 6.1 -> 5.8
// and with exponentials as accurate as expf's (another machine) 1 x 128 6.68 -> 6.77, 4 x 384 27.1 -> 27.4, 16 x 384 73.9 -> 75.9,
// 1 x 16 6.07 -> 6.13; expf itself: see exp_not_positive
#include "common.h"
#include "split_f32.h"

using namespace tnn_rocm;

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kD             = 64;
constexpr int kBlockQ        = 32;
constexpr int kBlockK        = 32;
constexpr int kKvLenMaskZero = 1 << 30;  // flag bit of a kv_len entry, see tnn_rocm_mask_to_kv_len_flagged
constexpr int kStageRow      = kD + 4;   // floats; the pad spreads the rows over the banks

struct AttnF32Params : StoreThrough {
    const float *q, *k, *v;
    float *o;
    long q_sb, q_sh, q_ss, kv_sb, kv_sh, kv_ss, o_sb, o_sh, o_ss;
    int S, B, heads;
    FixedDivisor by_blocks, by_batch;
    float scale, split_scale;  // of a score, of a score made from planes
    int planes;                // 0: the scale is too small for split_scale, the block is done with the fp32 instruction
    const float *mask;  // [B,S] additive or null
    const int32_t *kv_len;
};

__device__ __forceinline__ float other_half(float v) {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return (threadIdx.x & 32) ? __uint_as_float(r[0]) : __uint_as_float(r[1]);
}

// exp(x) for x <= 0 as 2^n 2^f, n the whole number nearest to x log2 e.  The product with log2 e is formed in two parts and the
// second joins f behind the subtraction of n, which is exact, so that the argument of the exponential instruction is rounded once
// and its result never again.  Below -200 the result is zero without a product that overflows; a NaN stays one; results below the
// smallest normal value keep the bits there are.  Ten instructions where expf takes fourteen, for any sign.  Errors over every
// float of [-87.3, -2^-20]: at most 0.857 ulp, 2.63e-8 root mean square from -1 down, both as expf's (0.857, 2.63e-8).  The second part as
// a factor behind the exponential is seven instructions, but rounds the result again and loses what is not normal: 1.262 ulp,
// 3.63e-8.
__device__ __forceinline__ float exp_not_positive(float x) {
    x              = __builtin_elementwise_maximum(x, -200.f);
    const float y  = __fmul_rn(x, 1.44269502f);
    const float lo = fmaf(x, 1.92596299e-8f, fmaf(x, 1.44269502f, -y));
    const float n  = rintf(y);
    return __builtin_ldexpf(__builtin_amdgcn_exp2f(__fadd_rn(__fsub_rn(y, n), lo)), (int)n);
}

// At least three waves a SIMD (168 registers): 4 x 384 tokens are 576 workgroups, two and a quarter for each CU, and with two a CU
// the last 64 were a round of their own.  Four (128 registers) spill.
template <int NW> __global__ void __launch_bounds__(NW * 64, NW == 4 ? 3 : 1) attention_f32_kernel(AttnF32Params p) {
    // the planes of Q (a step's three, a lane's 16 bytes each), then every wave's sums
    constexpr int kQBytes = 4 * 3 * 64 * 16, kStageBytes = NW * kBlockQ * kStageRow * 4;
    __shared__ __attribute__((aligned(16))) unsigned char shared[kQBytes > kStageBytes ? kQBytes : kStageBytes];
    uint4 *const q_planes = reinterpret_cast<uint4 *>(shared);
    float(*const stage)[kBlockQ * kStageRow] = reinterpret_cast<float(*)[kBlockQ * kStageRow]>(shared);
    __shared__ float stat_m[NW][kBlockQ], stat_l[NW][kBlockQ];
    __shared__ int again[NW];

    touch_kernel_args<sizeof(AttnF32Params)>();
    const int tid  = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g    = lane >> 5;
    const int lq   = lane & 31;
    const int S    = p.S;
    // Every XCD takes a contiguous run of (batch, head) pairs, so a head's K and V are fetched into one L2 only.  The pairs go head
    // by head: each XCD then has heads of nearly all sequences, and none is left with the longest ones (12 heads, lengths S/2 .. S
    // / 16 .. S: 4 x 384 25.3 26.1 -> 24.2 21.5 us, 16 x 384 63.6 61.4 -> 60.0 56.4).
    const int n_q   = (S + kBlockQ - 1) / kBlockQ;
    const int total = n_q * p.heads * p.B;
    const int per   = (total + 7) >> 3;
    const int vid   = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if (vid >= total)
        return;  // the grid is padded to a multiple of 8; whole workgroups leave before any barrier
    const int bh   = p.by_blocks.quotient(vid);
    const int head = p.by_batch.quotient(bh);
    const int b    = bh - head * p.B;
    const int q0   = (vid - bh * n_q) * kBlockQ;

    int kv_end        = S;
    bool mask_is_zero = false;
    if (p.kv_len) {
        int l        = p.kv_len[b];
        mask_is_zero = l >= 0 && (l & kKvLenMaskZero) != 0;
        l            = l >= 0 ? (l & ~kKvLenMaskZero) : l;
        kv_end       = l < 0 ? 0 : (l < S ? l : S);
    }
    const float *qb = p.q + (size_t)b * p.q_sb + (size_t)head * p.q_sh;
    const float *kb = p.k + (size_t)b * p.kv_sb + (size_t)head * p.kv_sh;
    const float *vb = p.v + (size_t)b * p.kv_sb + (size_t)head * p.kv_sh;
    const float *mb = p.mask && !mask_is_zero ? p.mask + (size_t)b * S : nullptr;
    const uint32_t ss   = (uint32_t)p.kv_ss;
    const int n_tiles   = (kv_end + kBlockK - 1) / kBlockK;
    f32x16 oacc[2];
    float m_i, l_i, low;
    // Rows past the end are clamped to the last one: keys at or beyond kv_end get the score -inf, queries past S are never
    // stored.  Per-head extents fit 32 bits (checked by the launcher).
    // this lane's row of Q, or of K in block t: eight values of every 16-wide step
    auto load_row = [&](const float *src, f32x4 (&raw)[8]) __attribute__((always_inline)) {
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            raw[2 * kk]     = *reinterpret_cast<const f32x4 *>(src + kk * 16);
            raw[2 * kk + 1] = *reinterpret_cast<const f32x4 *>(src + kk * 16 + 4);
        }
    };
    // blocks inside the sequence have a uniform base and one offset per lane; the last one clamps its rows
    auto load_k = [&](int t, f32x4 (&raw)[8]) __attribute__((always_inline)) {
        const int row = t * kBlockK + lq < S ? lq : S - 1 - t * kBlockK;
        load_row(kb + (size_t)(uint32_t)(t * kBlockK) * ss + ((uint32_t)row * ss + 8u * g), raw);
    };
    auto begin = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int dt = 0; dt < 2; ++dt)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                oacc[dt][r] = 0.f;
        m_i = -INFINITY, l_i = 0.f, low = 0.f;
    };
    // V of block t: slot e of step st and lane half g is key 16*st + 4*g + e (e < 4), 16*st + 8 + 4*g + e-4
    auto load_v = [&](int t, f32x2 (&vraw)[16]) __attribute__((always_inline)) {
        const float *const block = vb + (size_t)(uint32_t)(t * kBlockK) * ss;
        uint32_t mine            = (uint32_t)(4 * g) * ss + 2u * lq;
        asm volatile("" : "+v"(mine));  // or every row's address is kept from block to block, in 32 registers
        if (t * kBlockK + kBlockK <= S) {
            typedef const __attribute__((address_space(1))) f32x2 *GlobalPair;
            uint64_t row = reinterpret_cast<uint64_t>(block + mine);
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                asm("" : "+v"(row));  // one addition a row, not a product and a sum in scalar registers
                vraw[i] = *reinterpret_cast<GlobalPair>(row);
                row += 4 * ((i & 3) == 3 ? 5 * (uint64_t)ss : ss);
            }
        } else {
            const uint32_t last_row = (uint32_t)(S - 1 - t * kBlockK);
#pragma unroll
            for (int i = 0; i < 16; ++i)
                vraw[i] = *reinterpret_cast<const f32x2 *>(block + (min(16u * (i >> 3) + (i & 3) + (i & 4) * 2 + 4u * g, last_row) * ss + 2u * lq));
        }
    };
    // softmax over block t's keys: scores * scale + mask, as the decomposed layers form them
    auto softmax = [&](int t, float scale, auto exp_of, f32x16 &s) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            low  = fminf(low, s[r]);
            s[r] = __fmul_rn(s[r], scale);
        }
        if (mb) {
            int first_key = t * kBlockK + 4 * g;
            asm volatile("" : "+v"(first_key));  // or the keys are counted outside, for every block
            float m[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int key = first_key + (r >> 2) * 8 + (r & 3);
                m[r]          = mb[key < S ? key : S - 1];
            }
#pragma unroll
            for (int r = 0; r < 16; ++r)
                s[r] = __fadd_rn(s[r], m[r]);
        }
        if (t * kBlockK + kBlockK > kv_end) {
            int left = kv_end - t * kBlockK - 4 * g;
            asm volatile("" : "+v"(left));
#pragma unroll
            for (int r = 0; r < 16; ++r)
                s[r] = (r >> 2) * 8 + (r & 3) < left ? s[r] : -INFINITY;
        }
        float mx = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; ++r)
            mx = fmaxf(mx, s[r]);
        mx                = fmaxf(mx, other_half(mx));
        const float m_new = fmaxf(m_i, mx);
        const float m_use = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = exp_of(m_i - m_use);
        float sum         = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            s[r] = exp_of(s[r] - m_use);
            sum += s[r];
        }
        l_i = fmaf(l_i, alpha, sum + other_half(sum));
        if (!__all(m_new == m_i)) {
#pragma unroll
            for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    oacc[dt][r] *= alpha;
        }
        m_i = m_new;
    };
    // every wave leaves its sums, scaled to its own maximum
    auto leave = [&]() __attribute__((always_inline)) {
        float *row = stage[wave] + lq * kStageRow;
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
            const int d0 = 2 * (8 * r4 + 4 * g);
            *reinterpret_cast<f32x4 *>(row + d0)     = f32x4{oacc[0][r4 * 4], oacc[1][r4 * 4], oacc[0][r4 * 4 + 1], oacc[1][r4 * 4 + 1]};
            *reinterpret_cast<f32x4 *>(row + d0 + 4) = f32x4{oacc[0][r4 * 4 + 2], oacc[1][r4 * 4 + 2], oacc[0][r4 * 4 + 3], oacc[1][r4 * 4 + 3]};
        }
        if (lane < 32) {
            stat_m[wave][lq] = m_i;
            stat_l[wave][lq] = l_i;
        }
    };

    {
        const SplitConst sc;
        f32x4 kraw[8];
        f32x2 vraw[16];
        begin();
        // the waves share the queries: each makes its share of the steps' planes for all
        const float *const q_row = qb + (size_t)(q0 + lq < S ? q0 + lq : S - 1) * p.q_ss + 8 * g;
        f32x4 qraw[8 / NW];
        Split3 own[4 / NW];  // read with one wave only: nothing to share
#pragma unroll
        for (int i = 0; i < 4 / NW; ++i) {
            qraw[2 * i]     = *reinterpret_cast<const f32x4 *>(q_row + (wave + i * NW) * 16);
            qraw[2 * i + 1] = *reinterpret_cast<const f32x4 *>(q_row + (wave + i * NW) * 16 + 4);
        }
        const int first = wave < n_tiles ? wave : 0;  // a wave without a block requests the first one all the same
        load_k(first, kraw);
        if (NW == 1)
            load_v(0, vraw);
#pragma unroll
        for (int i = 0; i < 4 / NW; ++i) {
            const f32x4 lo = qraw[2 * i], hi = qraw[2 * i + 1];
            const float x[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            const Split3 qf  = split3(x, sc);
            if (NW == 1) {
                own[i] = qf;
                continue;
            }
#pragma unroll
            for (int w = 0; w < 3; ++w)
                q_planes[((wave + i * NW) * 3 + w) * 64 + lane] = make_uint4(qf.p[w][0], qf.p[w][1], qf.p[w][2], qf.p[w][3]);
        }
        if (NW > 1)
            __syncthreads();
        // scores of block t, from the rows in kraw
        auto scores = [&](f32x16 &s) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < 16; ++r)
                s[r] = 0.f;
            int mine = lane;
            asm volatile("" : "+v"(mine));  // or the compiler reads Q's planes once, into 48 registers
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                const f32x4 lo = kraw[2 * kk], hi = kraw[2 * kk + 1];
                const float x[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                Split3 qf = own[kk % (4 / NW)];
#pragma unroll
                for (int w = 0; NW > 1 && w < 3; ++w)
                    *reinterpret_cast<uint4 *>(qf.p[w]) = q_planes[(kk * 3 + w) * 64 + mine];
                const Split3 kf = split3(x, sc);
#pragma unroll
                for (int pr = 0; pr < kSplitProducts; ++pr)
                    split_mma(kf, qf, pr, s);
            }
        };
        // O^T += V^T P^T over half st of the block
        auto weigh = [&](int st, const f32x16 &s, const f32x2 (&vraw)[16]) __attribute__((always_inline)) {
            const float x[8] = {s[8 * st + 0], s[8 * st + 1], s[8 * st + 2], s[8 * st + 3],
                                s[8 * st + 4], s[8 * st + 5], s[8 * st + 6], s[8 * st + 7]};
            const Split3 pf  = split3(x, sc);
#pragma unroll
            for (int dt = 0; dt < 2; ++dt) {
                const f32x2 *vr  = vraw + st * 8;
                const float y[8] = {vr[0][dt], vr[1][dt], vr[2][dt], vr[3][dt], vr[4][dt], vr[5][dt], vr[6][dt], vr[7][dt]};
                const Split3 vf  = split3(y, sc);
#pragma unroll
                for (int pr = 0; pr < kSplitProducts; ++pr)
                    split_mma(vf, pf, pr, oacc[dt]);
            }
        };
        // V is requested with the block's begin, the next block's K when half of V is done with
        for (int t = wave; t < n_tiles; t += NW) {
            f32x16 s;
            if (NW > 1)
                load_v(t, vraw);
            asm volatile("" ::: "memory");
            scores(s);
            softmax(t, p.split_scale, [](float x) __attribute__((always_inline)) { return exp_not_positive(x); }, s);
            weigh(0, s, vraw);
#pragma unroll
            for (int i = 8; i < 16; ++i)
                asm volatile("" : "+v"(vraw[i]));  // all of V is here: weigh(1) does not wait for K
            asm volatile("" ::: "memory");
            if (t + NW < n_tiles)
                load_k(t + NW, kraw);
            else
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    asm volatile("" : "=v"(kraw[i]));  // no registers for the values of before
            asm volatile("" ::: "memory");
            weigh(1, s, vraw);
        }
    }
    __syncthreads();  // every wave is done with Q's planes
    leave();
    {
        // a score of -inf may be one that has no planes, or one that is; anything else that is not finite is in the sums
        float size = l_i;
#pragma unroll
        for (int dt = 0; dt < 2; ++dt)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                size += __builtin_fabsf(oacc[dt][r]);
        // the sums of up to four waves are added up below
        const int bad = !p.planes || __any(!split_finite(size * 4.f) || !split_finite(low));
        if (lane == 0)
            again[wave] = bad;
    }
    __syncthreads();
    int any_bad = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w)
        any_bad |= again[w];
    const bool exact = __builtin_amdgcn_readfirstlane(any_bad) != 0;
    // probabilities are taken down by a power of two of at least S, so that no partial sum runs over before the division
    const int down = 32 - __builtin_clz((unsigned)S);
    if (exact) {
        __syncthreads();  // everyone has read the flags
        const float pscale = __uint_as_float((uint32_t)(127 - down) << 23);
        begin();
#pragma unroll 1
        for (int t = wave; t < n_tiles; t += NW) {
            f32x16 s;
#pragma unroll
            for (int r = 0; r < 16; ++r)
                s[r] = 0.f;
            const float *k_row = kb + (size_t)(uint32_t)(t * kBlockK) * ss +
                                 ((uint32_t)(t * kBlockK + lq < S ? lq : S - 1 - t * kBlockK) * ss + 8u * g);
            const float *q_row = qb + (size_t)(q0 + lq < S ? q0 + lq : S - 1) * p.q_ss + 8 * g;
#pragma unroll 1
            for (int kk = 0; kk < 4; ++kk)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const f32x4 kr = *reinterpret_cast<const f32x4 *>(k_row + kk * 16 + h * 4);
                    const f32x4 qr = *reinterpret_cast<const f32x4 *>(q_row + kk * 16 + h * 4);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        s = __builtin_amdgcn_mfma_f32_32x32x2f32(kr[e], qr[e], s, 0, 0, 0);
                }
            softmax(t, p.scale, [](float x) __attribute__((always_inline)) { return expf(x); }, s);
            f32x2 vraw[16];
            load_v(t, vraw);
#pragma unroll
            for (int r = 0; r < 16; ++r)
#pragma unroll
                for (int dt = 0; dt < 2; ++dt)
                    oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(vraw[r][dt], s[r] * pscale, oacc[dt], 0, 0, 0);
        }
        leave();
        __syncthreads();
    }
    const float up = exact ? __uint_as_float((uint32_t)(127 + down) << 23) : kSplitUnscale;

    // ---- merge the waves
#pragma unroll
    for (int it = 0; it < kBlockQ * kD / 4 / (NW * 64); ++it) {
        const int item = it * NW * 64 + tid, row = item / (kD / 4), c = item % (kD / 4) * 4;
        if (q0 + row >= S)
            continue;
        float top = stat_m[0][row];
#pragma unroll
        for (int w = 1; w < NW; ++w)
            top = fmaxf(top, stat_m[w][row]);
        top = top == -INFINITY ? 0.f : top;
        f32x4 acc   = {0.f, 0.f, 0.f, 0.f};
        float total_l = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const float f = expf(stat_m[w][row] - top);
            total_l       = fmaf(stat_l[w][row], f, total_l);
            const f32x4 x = *reinterpret_cast<const f32x4 *>(stage[w] + row * kStageRow + c);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                acc[e] = fmaf(x[e], f, acc[e]);
        }
        // no key at all: zeros; a row whose every score is -inf: no number, as the softmax layer makes of it
        const float inv = total_l > 0.f ? 1.0f / total_l : kv_end > 0 ? NAN : 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            acc[e] = acc[e] * inv * up;
        store_out16(p.through, p.o + (size_t)b * p.o_sb + (size_t)head * p.o_sh + (size_t)(q0 + row) * p.o_ss + c,
                    __builtin_bit_cast(store_u32x4, acc));
    }
}

}  // namespace

namespace tnn_rocm {

// the argument checks are tnn_rocm_attention's; strides in elements
int launch_attention_f32(hipStream_t s, const float *q, const float *k, const float *v, float *out, int B, int heads, int S,
                         long q_sb, long q_sh, long q_ss, long kv_sb, long kv_sh, long kv_ss, long o_sb, long o_sh, long o_ss,
                         float scale, const float *mask, const int32_t *kv_len) {
    AttnF32Params p;
    p.q = q, p.k = k, p.v = v, p.o = out;
    p.q_sb = q_sb, p.q_sh = q_sh, p.q_ss = q_ss;
    p.kv_sb = kv_sb, p.kv_sh = kv_sh, p.kv_ss = kv_ss;
    p.o_sb = o_sb, p.o_sh = o_sh, p.o_ss = o_ss;
    p.S = S, p.B = B, p.heads = heads;
    p.by_blocks = FixedDivisor::of((uint32_t)((S + kBlockQ - 1) / kBlockQ));
    p.by_batch  = FixedDivisor::of((uint32_t)B);
    p.scale       = scale;
    p.split_scale = scale * kSplitUnscale;
    p.planes      = !(scale > -1e-20f && scale < 1e-20f);  // no bit of split_scale is lost from 2^-78 on
    p.mask   = mask;
    p.kv_len = kv_len;
    const long total = (long)((S + kBlockQ - 1) / kBlockQ) * heads * B;
    TR_REQUIRE(total < (1l << 30), TNN_ROCM_ESHAPE, "attention: too many query blocks");
    const dim3 grid((unsigned)((total + 7) / 8 * 8));
    // one block of keys: nothing to share among waves
    if (S <= kBlockK)
        hipLaunchKernelGGL(attention_f32_kernel<1>, grid, dim3(64), 0, s, p);
    else
        hipLaunchKernelGGL(attention_f32_kernel<4>, grid, dim3(256), 0, s, p);
    TR_CHECK_LAUNCH();
    return 0;
}

}  // namespace tnn_rocm
