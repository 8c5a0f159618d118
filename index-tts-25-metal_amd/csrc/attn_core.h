// Causal attention of prompt rows on the matrix cores, shared by the GPT and Qwen prefills.
//
// A workgroup of four waves takes 16 query rows of one head.  Each wave takes every fourth
// chunk of 32 keys with a running maximum, sum and weighted V sum of its own (the online
// recurrence of mit2_gpt_causal_attention_sgq_f32, kernels.metal:2249-2292), and the four are
// merged through LDS at the end: a 155-row prefix has at most five chunks, so its longest
// tile is two chunks deep instead of three 64-key passes.
//
// Both products are formed transposed, so a lane keeps one query (lane & 15) throughout and
// nothing passes through LDS between them:
//   S^T = K Q^T: lane (g, q) ends with the scores of query q and keys 4 g + r (+ 16);
//   O^T = V^T P^T: those same eight weights, in that order, are the lane's operand of the
//   second product (any order of the keys serves, V is read in the same one), and its
//   result, dimensions 4 g + r of query q, is rescaled by the lane's own factor.
// FP32 inputs and weights are split into three BF16 numbers and multiplied with six
// instructions, the five small products in accumulators of their own (gemm_core.h).  An infinite
// or NaN value, and one past the largest BF16, makes every sum that it is in NaN or infinite:
// attn_refine forms such outputs again with FP32 products.
#pragma once
#include "gemm_core.h"

namespace itts {

struct SplitFrag {
    bf16x8 h, m, l;
};
__device__ __forceinline__ SplitFrag split_frag(const float (&x)[8]) {
    u32x4 h, m, l;
    split_piece(x, h, m, l);
    return {__builtin_bit_cast(bf16x8, h), __builtin_bit_cast(bf16x8, m), __builtin_bit_cast(bf16x8, l)};
}
__device__ __forceinline__ void split_mfma(const SplitFrag& a, const SplitFrag& b, f32x4& hi, f32x4& lo) {
    lo = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.l, b.h, lo, 0, 0, 0);
    hi = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.h, b.h, hi, 0, 0, 0);
    lo = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.h, b.l, lo, 0, 0, 0);
    lo = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.m, b.m, lo, 0, 0, 0);
    lo = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.m, b.h, lo, 0, 0, 0);
    lo = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.h, b.m, lo, 0, 0, 0);
}

constexpr int kAttnWaves = 4, kAttnTile = 16, kAttnKeys = 32;

template <int HD>
struct alignas(16) AttnLds {  // rows of o are written 16 bytes at a time
    float o[kAttnWaves][kAttnTile][HD + 4];
    float m[kAttnWaves][kAttnTile], l[kAttnWaves][kAttnTile];
    static_assert((HD + 4) % 4 == 0, "16-byte rows");
};

// One wave's state over the chunks it has seen.
template <int HD>
struct AttnState {
    float m = -INFINITY, l = 0.0f;  // l: this lane's keys only
    f32x4 hi[HD / 16], lo[HD / 16];
    __device__ AttnState() {
#pragma unroll
        for (int t = 0; t < HD / 16; ++t) hi[t] = lo[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
};

// Keys c0 .. c0 + 31 (those past kn - 1 reread it and are masked) of rows kb / vb, HD floats
// apart.  pos: the last key this lane's query sees, -1 if it sees none of these rows.
template <int HD>
__device__ __forceinline__ void attn_chunk(AttnState<HD>& st, const SplitFrag (&q)[HD / 32], const float* kb, const float* vb, int c0, int kn,
                                           int pos, float scale, int lane) {
    const int g = lane >> 4, c = lane & 15;
    f32x4 kr[2][HD / 32][2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const float* p = kb + static_cast<size_t>(min(c0 + 16 * t + c, kn - 1)) * HD + 8 * g;
#pragma unroll
        for (int d = 0; d < HD / 32; ++d) {
            kr[t][d][0] = *reinterpret_cast<const f32x4*>(p + 32 * d);
            kr[t][d][1] = *reinterpret_cast<const f32x4*>(p + 32 * d + 4);
        }
    }
    float v[HD / 16][8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float* p = vb + static_cast<size_t>(min(c0 + (j < 4 ? 4 * g + j : 12 + 4 * g + j), kn - 1)) * HD + c;
#pragma unroll
        for (int t = 0; t < HD / 16; ++t) v[t][j] = p[16 * t];
    }
    __builtin_amdgcn_sched_barrier(0);  // every load of the chunk is in flight before the first product
    float s[8];
    bool ok[8];
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        f32x4 hi = {0.f, 0.f, 0.f, 0.f}, lo = hi;
#pragma unroll
        for (int d = 0; d < HD / 32; ++d) {
            float x[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] = kr[t][d][i >> 2][i & 3];
            split_mfma(split_frag(x), q[d], hi, lo);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            ok[4 * t + r] = c0 + 16 * t + 4 * g + r <= pos;
            s[4 * t + r] = ok[4 * t + r] ? (hi[r] + lo[r]) * scale : -INFINITY;
            mx = fmaxf(mx, s[4 * t + r]);
        }
    }
    mx = xmax16(xmax32(mx));
    const float mnew = fmaxf(st.m, mx);
    const float corr = st.m == -INFINITY ? 0.0f : expf(st.m - mnew);
    float p[8], sum = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        p[i] = ok[i] ? expf(s[i] - mnew) : 0.0f;
        sum += p[i];
    }
    st.l = st.l * corr + sum;
    st.m = mnew;
    const SplitFrag pf = split_frag(p);
#pragma unroll
    for (int t = 0; t < HD / 16; ++t) {
        st.hi[t] *= corr;
        st.lo[t] *= corr;
        split_mfma(split_frag(v[t]), pf, st.hi[t], st.lo[t]);
    }
}

// Merges the four waves' states; thread t of 256 ends with the outputs of query t / 16 at the
// HD / 16 dimensions from HD / 16 (t % 16) on.
template <int HD>
__device__ __forceinline__ void attn_merge(AttnLds<HD>& lds, const AttnState<HD>& st, int wave, int lane, float (&out)[HD / 16]) {
    const int g = lane >> 4, c = lane & 15;
    const float l = xsum16(xsum32(st.l, st.l), xsum32(st.l, st.l));
    if (g == 0) {
        lds.m[wave][c] = st.m;
        lds.l[wave][c] = l;
    }
#pragma unroll
    for (int t = 0; t < HD / 16; ++t) *reinterpret_cast<f32x4*>(&lds.o[wave][c][16 * t + 4 * g]) = st.hi[t] + st.lo[t];
    __syncthreads();
    const int r = threadIdx.x >> 4, d0 = (threadIdx.x & 15) * (HD / 16);
    float m = lds.m[0][r];
#pragma unroll
    for (int w = 1; w < kAttnWaves; ++w) m = fmaxf(m, lds.m[w][r]);
    float den = 0.0f;
#pragma unroll
    for (int i = 0; i < HD / 16; ++i) out[i] = 0.0f;
#pragma unroll
    for (int w = 0; w < kAttnWaves; ++w) {
        const float f = lds.m[w][r] == -INFINITY ? 0.0f : expf(lds.m[w][r] - m);
        den = __builtin_fmaf(lds.l[w][r], f, den);
#pragma unroll
        for (int i = 0; i < HD / 16; ++i) out[i] = __builtin_fmaf(lds.o[w][r][d0 + i], f, out[i]);
    }
#pragma unroll
    for (int i = 0; i < HD / 16; ++i) out[i] /= den;
}

// Outputs of attn_merge that are not finite, formed again from the FP32 rows: thread t's query
// (its row: p) and the keys 0 .. pos() of rows kb / vb, all the same for the 16 threads of a query.
// The whole wave calls it; `valid` outputs only.
template <int HD, class Pos>
__device__ __forceinline__ void attn_refine(const float* p, const float* kb, const float* vb, Pos pos, float scale, bool valid, int lane,
                                            float (&out)[HD / 16]) {
    constexpr int D = HD / 16;
    float t = out[0];
#pragma unroll
    for (int i = 1; i < D; ++i) t += out[i];
    const uint64_t bad = __ballot(valid && !(fabsf(t) <= 3.402823466e38f));
    if (__builtin_expect(bad == 0, 1)) return;
    if (((bad >> (lane & 48)) & 0xffff) == 0) return;
    const int d0 = (lane & 15) * D, keys = pos() + 1;
    float q[D], m = -INFINITY, l = 0.0f;
#pragma unroll
    for (int i = 0; i < D; ++i) q[i] = p[d0 + i];
    auto score = [&](int k) {
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < D; ++i) s = __builtin_fmaf(q[i], kb[static_cast<size_t>(k) * HD + d0 + i], s);
        return row16_sum(s) * scale;
    };
#pragma clang loop unroll(disable)
    for (int k = 0; k < keys; ++k) m = fmaxf(m, score(k));
#pragma unroll
    for (int i = 0; i < D; ++i) out[i] = 0.0f;
#pragma clang loop unroll(disable)
    for (int k = 0; k < keys && l == l; ++k) {  // (NaN stays)
        const float w = expf(score(k) - m);
        l += w;
#pragma unroll
        for (int i = 0; i < D; ++i) out[i] = __builtin_fmaf(w, vb[static_cast<size_t>(k) * HD + d0 + i], out[i]);
    }
#pragma unroll
    for (int i = 0; i < D; ++i) out[i] /= l;
}

// This lane's operand of query row p (HD floats).
template <int HD>
__device__ __forceinline__ void attn_query(const float* p, int lane, SplitFrag (&q)[HD / 32]) {
#pragma unroll
    for (int d = 0; d < HD / 32; ++d) {
        float x[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = p[32 * d + 8 * (lane >> 4) + i];
        q[d] = split_frag(x);
    }
}

}  // namespace itts
