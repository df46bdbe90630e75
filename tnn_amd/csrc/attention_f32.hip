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
// What bounds it: the vector ALU (conversion of K, V and P: 36 instructions per operand and 16-wide step, and the
// exponentials) and the matrix pipe, about equal.  us, the decomposed launches -> this kernel, 12 heads:
//   1 x 128 tokens 45 -> 7.6, 4 x 384 136 -> 29 (K and V read once per block of 32 queries: 113 MB from L2), 8 x 128 11, 1 x 512 16
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
    FixedDivisor by_blocks, by_heads;
    float scale, split_scale;  // of a score, of a score made from planes
    int planes;                // 0: the scale is too small for split_scale, the block is done with the fp32 instruction
    const float *mask;  // [B,S] additive or null
    const int32_t *kv_len;
};

__device__ __forceinline__ float other_half(float v) {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return (threadIdx.x & 32) ? __uint_as_float(r[0]) : __uint_as_float(r[1]);
}

template <int NW> __global__ void __launch_bounds__(NW * 64, NW == 4 ? 2 : 1) attention_f32_kernel(AttnF32Params p) {
    __shared__ __attribute__((aligned(16))) float stage[NW][kBlockQ * kStageRow];
    __shared__ float stat_m[NW][kBlockQ], stat_l[NW][kBlockQ];
    __shared__ int again[NW];

    touch_kernel_args<sizeof(AttnF32Params)>();
    const int tid  = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g    = lane >> 5;
    const int lq   = lane & 31;
    const int S    = p.S;
    // every XCD takes a contiguous run of (batch, head) pairs, so a head's K and V are fetched into one L2 only
    const int n_q   = (S + kBlockQ - 1) / kBlockQ;
    const int total = n_q * p.heads * p.B;
    const int per   = (total + 7) >> 3;
    const int vid   = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if (vid >= total)
        return;  // the grid is padded to a multiple of 8; whole workgroups leave before any barrier
    const int bh   = p.by_blocks.quotient(vid);
    const int b    = p.by_heads.quotient(bh);
    const int head = bh - b * p.heads;
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
    auto load_q = [&](f32x4 (&raw)[8]) __attribute__((always_inline)) {
        const int row = q0 + lq < S ? q0 + lq : S - 1;
        load_row(qb + (size_t)row * p.q_ss + 8 * g, raw);
    };
    auto load_k = [&](int t, f32x4 (&raw)[8]) __attribute__((always_inline)) {
        const int row = t * kBlockK + lq < S ? t * kBlockK + lq : S - 1;
        load_row(kb + ((uint32_t)row * ss + 8u * g), raw);
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
#pragma unroll
        for (int st = 0; st < 2; ++st)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                int row = t * kBlockK + 16 * st + 4 * g + (e & 3) + (e & 4) * 2;
                row     = row < S ? row : S - 1;
                vraw[st * 8 + e] = *reinterpret_cast<const f32x2 *>(vb + ((uint32_t)row * ss + 2u * lq));
            }
    };
    // softmax over block t's keys: scores * scale + mask, as the decomposed layers form them
    auto softmax = [&](int t, float scale, f32x16 &s) __attribute__((always_inline)) {
        float mx = -INFINITY;
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
            const int key0 = t * kBlockK + 8 * r4 + 4 * g;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                low     = fminf(low, s[r4 * 4 + e]);
                float v = __fmul_rn(s[r4 * 4 + e], scale);
                if (mb)
                    v = __fadd_rn(v, mb[key0 + e < S ? key0 + e : S - 1]);
                v             = key0 + e < kv_end ? v : -INFINITY;
                s[r4 * 4 + e] = v;
                mx            = fmaxf(mx, v);
            }
        }
        mx                = fmaxf(mx, other_half(mx));
        const float m_new = fmaxf(m_i, mx);
        const float m_use = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = expf(m_i - m_use);
        float sum         = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            s[r] = expf(s[r] - m_use);
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
        Split3 qf[4];
        f32x4 kraw[8];
        load_q(kraw);
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            const f32x4 lo = kraw[2 * kk], hi = kraw[2 * kk + 1];
            const float x[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            qf[kk]           = split3(x, sc);
        }
        begin();
        if (wave < n_tiles)
            load_k(wave, kraw);
        for (int t = wave; t < n_tiles; t += NW) {
            f32x2 vraw[16];
            load_v(t, vraw);
            // ---- S^T = K Q^T
            f32x16 s;
#pragma unroll
            for (int r = 0; r < 16; ++r)
                s[r] = 0.f;
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                const f32x4 lo = kraw[2 * kk], hi = kraw[2 * kk + 1];
                const float x[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                const Split3 kf  = split3(x, sc);
#pragma unroll
                for (int pr = 0; pr < kSplitProducts; ++pr)
                    split_mma(kf, qf[kk], pr, s);
            }
            if (t + NW < n_tiles)
                load_k(t + NW, kraw);
            softmax(t, p.split_scale, s);
            // ---- O^T += V^T P^T
#pragma unroll
            for (int st = 0; st < 2; ++st) {
                const float x[8] = {s[8 * st + 0], s[8 * st + 1], s[8 * st + 2], s[8 * st + 3],
                                    s[8 * st + 4], s[8 * st + 5], s[8 * st + 6], s[8 * st + 7]};
                const Split3 pf  = split3(x, sc);
                Split3 vf[2];
#pragma unroll
                for (int dt = 0; dt < 2; ++dt) {
                    const f32x2 *vr  = vraw + st * 8;
                    const float y[8] = {vr[0][dt], vr[1][dt], vr[2][dt], vr[3][dt], vr[4][dt], vr[5][dt], vr[6][dt], vr[7][dt]};
                    vf[dt]           = split3(y, sc);
                }
#pragma unroll
                for (int pr = 0; pr < kSplitProducts; ++pr)
#pragma unroll
                    for (int dt = 0; dt < 2; ++dt)
                        split_mma(vf[dt], pf, pr, oacc[dt]);
            }
        }
    }
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
            f32x4 kraw[8], qraw[8];
            load_k(t, kraw);
            load_q(qraw);
#pragma unroll
            for (int kk = 0; kk < 8; ++kk)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    s = __builtin_amdgcn_mfma_f32_32x32x2f32(kraw[kk][e], qraw[kk][e], s, 0, 0, 0);
            softmax(t, p.scale, s);
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
    p.by_heads  = FixedDivisor::of((uint32_t)heads);
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
