// Prefill kernels (the P-row prefix forward of gpt.cpp:88-125 with initial=true).
//
// * ln_rows: LayerNorm of each 1280-wide row (kernels.metal:618-669), one workgroup per row.
// * gemm: C[M][N] = A[M][K] * W[N][K]^T + bias on the matrix cores, replacing the
//   broadcast-bias + MPS GEMM pair of metal_context.mm:368-410.  The operands are FP32 values
//   split into three BF16 numbers and multiplied by BF16 instructions (gemm_core.h); A comes
//   split from the kernel that produced it (LayerNorm, attention, GELU), weights are split on
//   the way to LDS.  Epilogues: q rows + K/V cache store (kernels.metal:1250-1266), residual
//   add in place, GELU, plain store, SiLU-gated pairs.
//   When the tiles alone would leave CUs idle, K is split over gridDim.z: each split writes
//   its partial tile to a workspace and gemm_reduce adds the splits in order, then the bias
//   and the epilogue.
// * causal_attention: 16 query rows of a head per workgroup, both products on the matrix
//   cores (attn_core.h).
// Rows of several sequences may be stacked (ragged batch prefill): row m belongs to
// cache slot row_slot[m] at position row_pos[m] and attends to that slot's rows
// 0..row_pos[m].
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "attn_core.h"
#include "kernels.h"

namespace itts {
namespace {

__global__ __launch_bounds__(256) void ln_rows_kernel(LnRowsArgs a) {
    __shared__ float red[4];
    const int row = blockIdx.x, tid = threadIdx.x;
    float v[1][5];
#pragma unroll
    for (int i = 0; i < 5; ++i) v[0][i] = a.x[static_cast<size_t>(row) * kWidth + tid + 256 * i];
    ln_block<1, 5>(v, a.w, a.b, red);
#pragma unroll
    for (int i = 0; i < 5; ++i) split_store(a.y, split_off(row, tid + 256 * i, kWidth), v[0][i]);
}

// SiLU-gated product of one (gate, up) column pair (kernels.metal:363-374).
__device__ __forceinline__ float swiglu_f(float g, float u) { return (g / (1.0f + expf(-g))) * u; }

// Cache element of K/V column rr (of 2 x 1280) at position pos of a slot.
__device__ __forceinline__ size_t kv_off(const GemmArgs& a, int rr, uint32_t slot, uint32_t pos) {
    const bool is_v = rr >= kWidth;
    const int c = is_v ? rr - kWidth : rr;
    return static_cast<size_t>(slot) * a.kv_slot_stride + a.kv_layer_off + (is_v ? a.kv_v_off : 0) +
           (static_cast<size_t>(c >> 6) * a.kv_cap + pos) * kHeadDim + (c & 63);
}

// One result of a GEMM: the sum of row `row` and column `col` (of split z).  Every lane of a wave calls
// it, lanes l and l ^ 1 with columns col and col ^ 1 of a row; rows past the last are not stored.
template <int EPI, bool SPLIT>
__device__ __forceinline__ void gemm_store_one(const GemmArgs& a, int z, int row, int col, float sum) {
    const bool live = row < a.M;
    const float v = sum + (SPLIT ? 0.0f : a.bias[col]);
    if constexpr (SPLIT) {
        if (live) a.ws[(static_cast<size_t>(z) * a.M + row) * a.N + col] = sum;
    } else if constexpr (EPI == kGemmGelu) {
        if (live) split_store(a.c_split, split_off(row, col, a.N), gelu_f(v));
    } else if constexpr (EPI == kGemmSwiglu) {
        const float u = __shfl_xor(v, 1, 64);
        if (live && !(col & 1)) split_store(a.c_split, split_off(row, col / 2, a.N / 2), swiglu_f(v, u));
    } else if constexpr (EPI == kGemmQkv) {
        if (!live) return;
        if (col < kWidth) a.c[static_cast<size_t>(row) * kWidth + col] = v;
        else a.kv[kv_off(a, col - kWidth, a.row_slot[row], a.row_pos[row])] = v;
    } else {
        if (!live) return;
        float* p = a.c + static_cast<size_t>(row) * a.N + col;
        *p = EPI == kGemmResid ? *p + v : v;
    }
}

// Row block y covers row tiles [y RT, (y + 1) RT) of A; split z covers K range
// [z kchunk, min(K, (z + 1) kchunk)) and, with SPLIT, writes its raw partial tile to
// a.ws[z][M][N] for gemm_reduce_kernel.  Row tiles past the last are clamped to it (their
// results are not stored), so the main loop (gemm_core.h) has no branches.
template <class T, int EPI, bool SPLIT>
__global__ __launch_bounds__(kGemmThreads) void gemm_kernel(GemmArgs a, int kchunk) {
    __shared__ __align__(16) uint8_t lds[T::kLdsBytes];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const auto [bx, by, bz] = gemm_place();
    const int kb = SPLIT ? bz * kchunk : 0;
    const int nst = ((SPLIT ? min(a.K, kb + kchunk) : a.K) - kb) / 32;
    uint16_t* ring = reinterpret_cast<uint16_t*>(lds);
    const __amdgpu_buffer_rsrc_t ars = gemm_rsrc(a.a, static_cast<uint32_t>(split_elems(a.M, a.K) * 2));
    const int tiles = (a.M + 15) / 16;
    if (wave >= 4) {
        gemm_loader<T>(ring, static_cast<const typename T::W*>(a.w) + static_cast<size_t>(bx) * T::BN * a.K + kb, a.K, nst, tid - 256);
        return;
    }
    constexpr int TR = T::TR, TC = T::TC;
    const int wr = wave / T::WC, wc = wave % T::WC;
    const int tile0 = by * T::RT + wr * TR;
    uint32_t off[TR];
#pragma unroll
    for (int i = 0; i < TR; ++i) off[i] = (static_cast<uint32_t>(min(tile0 + i, tiles - 1)) * (a.K / 32) + kb / 32) * (kTileElems * 2) + lane * 16;
    GemmAcc<T> sums;
    gemm_compute<T>(
        ring, ars, [&](int i, int s) { return GemmOff{off[i], static_cast<uint32_t>(s) * (kTileElems * 2)}; }, nst, wc, lane, sums);
    const int n0 = bx * T::BN + wc * TC * 16;  // the wave's first column
    const auto dot = [&](int m, int n) {
        return gemm_dot(static_cast<const typename T::W*>(a.w) + static_cast<size_t>(n0 + n) * a.K + kb, nst * 32,
                        [&](int k) { return split_value(a.a + split_off(m, kb + k, a.K)); });
    };
    const bool suspect = sums.suspect();
    if constexpr (SPLIT || (EPI != kGemmGelu && EPI != kGemmSwiglu)) {
        if (__builtin_expect(suspect, 0)) {
            gemm_refine<T>(lds, a.M, tile0, wave, lane, sums, dot, [&](int m, int n, float v) { gemm_store_one<EPI, SPLIT>(a, bz, m, n0 + n, v); });
            return;
        }
    }
    f32x4 acc[TR][TC];
    sums.sum(acc);

    // acc[i][c][r]: row 16 (tile0 + i) + rq + r, column col0 + 16 c
    const int col0 = n0 + (lane & 15);
    const int rq = 4 * (lane >> 4);
    if constexpr (SPLIT) {
        gemm_store_partial<T>(a.ws + static_cast<size_t>(bz) * a.M * a.N, a.M, a.N, tile0, col0, lane, acc);
    } else if constexpr (EPI == kGemmGelu || EPI == kGemmSwiglu) {
        float bias[TC];
#pragma unroll
        for (int c = 0; c < TC; ++c) bias[c] = a.bias[col0 + 16 * c];
        if constexpr (EPI == kGemmGelu) {
            gemm_store_split<T, false>(
                lds, wave, lane, a.c_split, a.M, a.N, 0, tile0, n0, [&](int i, int c, int r) { return gelu_f(acc[i][c][r] + bias[c]); }, suspect,
                [&](int m, int n) { return gelu_f(dot(m, n) + a.bias[n0 + n]); });
        } else {  // columns col and col ^ 1 sit in lanes l and l ^ 1, on the same rows
            gemm_store_split<T, true>(
                lds, wave, lane, a.c_split, a.M, a.N / 2, 0, tile0, n0 / 2,
                [&](int i, int c, int r) {
                    const float v = acc[i][c][r] + bias[c];
                    return swiglu_f(v, __shfl_xor(v, 1, 64));
                },
                suspect, [&](int m, int n) { return swiglu_f(dot(m, 2 * n) + a.bias[n0 + 2 * n], dot(m, 2 * n + 1) + a.bias[n0 + 2 * n + 1]); });
        }
    } else {
        float bias[TC];
#pragma unroll
        for (int c = 0; c < TC; ++c) bias[c] = a.bias[col0 + 16 * c];
        // K/V columns (a workgroup's columns are all q or all K/V: 1280 is a multiple of BN)
        const bool kv_cols = EPI == kGemmQkv && bx * T::BN >= kWidth;
        const int ldc = EPI == kGemmQkv ? kWidth : a.N;
#pragma unroll
        for (int i = 0; i < TR; ++i) {
            // Every row's residual, or cache slot and position, requested before the first
            // store (rows past M read row 0): a load under the per-row branch was waited
            // for before the next.
            float out[TC][4];
            uint32_t rs[4] = {}, rp[4] = {};
            const int row0 = (tile0 + i) * 16 + rq;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int rc = row0 + r < a.M ? row0 + r : 0;
                if (kv_cols) {
                    rs[r] = a.row_slot[rc];
                    rp[r] = a.row_pos[rc];
                }
#pragma unroll
                for (int c = 0; c < TC; ++c) {
                    out[c][r] = acc[i][c][r] + bias[c];
                    if constexpr (EPI == kGemmResid) out[c][r] += a.c[static_cast<size_t>(rc) * a.N + col0 + 16 * c];
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                pin_value(rs[r]);
                pin_value(rp[r]);
#pragma unroll
                for (int c = 0; c < TC; ++c) pin_value(out[c][r]);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (row0 + r < a.M) {
#pragma unroll
                    for (int c = 0; c < TC; ++c) {
                        if (kv_cols) a.kv[kv_off(a, col0 + 16 * c - kWidth, rs[r], rp[r])] = out[c][r];
                        else a.c[static_cast<size_t>(row0 + r) * ldc + col0 + 16 * c] = out[c][r];
                    }
                }
        }
    }
}

// The same for up to 16 RT rows (gemm_core.h, gemm_small).
template <typename WT, int RT, int EPI, bool SPLIT>
__global__ __launch_bounds__(64 * kSmallWaves) void gemm_small_kernel(GemmArgs a, int kchunk) {
    __shared__ GemmSmallLds<RT> lds;
    const int kb = SPLIT ? blockIdx.y * kchunk : 0, nst = ((SPLIT ? min(a.K, kb + kchunk) : a.K) - kb) / 32;
    const uint32_t row_bytes = a.K / 32 * (kTileElems * 2);
    float sum[2];
    gemm_small<WT, RT>(lds, static_cast<const WT*>(a.w) + static_cast<size_t>(blockIdx.x) * 16 * a.K + kb, a.K, nst,
                       gemm_rsrc(a.a, static_cast<uint32_t>(split_elems(a.M, a.K) * 2)), kb / 32 * (kTileElems * 2), row_bytes, a.M,
                       [&](int m, int k) { return split_value(a.a + split_off(m, kb + k, a.K)); }, sum);
#pragma unroll
    for (int q = 0; q < (RT > 2 ? 2 : 1); ++q)
        gemm_store_one<EPI, SPLIT>(a, blockIdx.y, (threadIdx.x >> 4) + 32 * q, blockIdx.x * 16 + (threadIdx.x & 15), sum[q]);
}

// Partial 0 + partial 1 + ... of four consecutive elements from e on, in split order.  Every
// split's load is issued before the first add (SM, a power of two >= the split count, loads;
// indices past the split count reread the last split and their adds are skipped), so the
// loads overlap instead of forming a chain of round trips.
template <int SM>
__device__ __forceinline__ f32x4 split_sum_n(const GemmArgs& a, size_t e, size_t plane) {
    f32x4 w[SM];
#pragma unroll
    for (int z = 0; z < SM; ++z) w[z] = *reinterpret_cast<const f32x4*>(a.ws + static_cast<size_t>(min(z, a.splits - 1)) * plane + e);
    f32x4 d = w[0];
#pragma unroll
    for (int z = 1; z < SM; ++z)
        if (z < a.splits) d += w[z];
    return d;
}
__device__ __forceinline__ f32x4 split_sum(const GemmArgs& a, size_t e, size_t plane) {
    if (a.splits <= 2) return split_sum_n<2>(a, e, plane);
    if (a.splits <= 4) return split_sum_n<4>(a, e, plane);
    if (a.splits <= 8) return split_sum_n<8>(a, e, plane);
    return split_sum_n<kGemmMaxSplits>(a, e, plane);
}

// Finishes a split-K GEMM: dot = partial 0 + partial 1 + ... in split order, then + bias and
// the epilogue; a thread takes 4 columns (kGemmSwiglu: 4 pairs) of one row.  (Eight
// per thread, one 16-byte store per plane, left a 48-row c_fc 96 workgroups of long GELU chains.)
template <int EPI>
__global__ __launch_bounds__(256) void gemm_reduce_kernel(GemmArgs a) {
    constexpr int W = EPI == kGemmSwiglu ? 8 : 4;
    const size_t plane = static_cast<size_t>(a.M) * a.N, total = plane / W;
    for (size_t t = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; t < total; t += static_cast<size_t>(gridDim.x) * blockDim.x) {
        const size_t e = t * W;
        const int row = static_cast<int>(e / a.N), col = static_cast<int>(e % a.N);
        float v[W];
        uint32_t rs = 0, rp = 0;
        if (EPI == kGemmQkv && col >= kWidth) {  // requested with the partials, not after them
            rs = a.row_slot[row];
            rp = a.row_pos[row];
        }
#pragma unroll
        for (int q = 0; q < W / 4; ++q) {
            const f32x4 d = split_sum(a, e + 4 * q, plane) + *reinterpret_cast<const f32x4*>(a.bias + col + 4 * q);
#pragma unroll
            for (int i = 0; i < 4; ++i) v[4 * q + i] = d[i];
        }
        if constexpr (EPI == kGemmGelu) {
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = gelu_f(v[i]);
            split_store4(a.c_split, split_off(row, col, a.N), v);
        } else if constexpr (EPI == kGemmSwiglu) {
            float o[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = swiglu_f(v[2 * i], v[2 * i + 1]);
            split_store4(a.c_split, split_off(row, col / 2, a.N / 2), o);
        } else {
            f32x4 o = {v[0], v[1], v[2], v[3]};
            if (EPI == kGemmQkv && col >= kWidth) {
                *reinterpret_cast<f32x4*>(a.kv + kv_off(a, col - kWidth, rs, rp)) = o;
            } else {
                f32x4* p = reinterpret_cast<f32x4*>(a.c + static_cast<size_t>(row) * (EPI == kGemmQkv ? kWidth : a.N) + col);
                if constexpr (EPI == kGemmResid) o = *p + o;
                *p = o;
            }
        }
    }
}

// Finishes a split-K kGemmResid GEMM of 1280-wide rows and the LayerNorm after it, one
// workgroup per row: c[m] += (partials in split order + bias), then ln_out[m] =
// LayerNorm(c[m]).  Thread t holds columns t + 256 i as ln_rows_kernel does, so both
// results are bitwise those of gemm_reduce_kernel<kGemmResid> followed by ln_rows_kernel.
__global__ __launch_bounds__(256) void gemm_reduce_ln_kernel(GemmArgs a) {
    __shared__ float red[4];
    const int row = blockIdx.x, tid = threadIdx.x;
    const size_t plane = static_cast<size_t>(a.M) * a.N;
    // Every load of the five columns before the first add and store, within one split-count
    // case: per column, the split sums behind a branch and the store to c before the next
    // column's loads made each column a memory round trip of its own.
    float v[1][5];
    auto body = [&](auto sm) {
        constexpr int SM = decltype(sm)::value;
        float cv[5], bv[5], w[5][SM];
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            const int col = tid + 256 * i;
            const size_t e = static_cast<size_t>(row) * a.N + col;
            cv[i] = a.c[e];
            bv[i] = a.bias[col];
#pragma unroll
            for (int z = 0; z < SM; ++z) w[i][z] = a.ws[static_cast<size_t>(min(z, a.splits - 1)) * plane + e];
        }
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            float s = w[i][0];  // split_sum_n's order
#pragma unroll
            for (int z = 1; z < SM; ++z)
                if (z < a.splits) s += w[i][z];
            v[0][i] = cv[i] + (s + bv[i]);
            a.c[static_cast<size_t>(row) * a.N + tid + 256 * i] = v[0][i];
        }
    };
    if (a.splits <= 2)
        body(std::integral_constant<int, 2>{});
    else if (a.splits <= 4)
        body(std::integral_constant<int, 4>{});
    else if (a.splits <= 8)
        body(std::integral_constant<int, 8>{});
    else
        body(std::integral_constant<int, kGemmMaxSplits>{});
    ln_block<1, 5>(v, a.ln_w, a.ln_b, red);
#pragma unroll
    for (int i = 0; i < 5; ++i) split_store(a.ln_out, split_off(row, tid + 256 * i, kWidth), v[0][i]);
}

// Causal attention over one head for 16 consecutive rows (attn_core.h).  The rows are taken in
// runs that share a cache slot (stacked sequences: positions restart at 0 in each slot): for
// each run the slot's keys 0 .. max position, in a state of its own (a row of another slot has
// weight 0 there, and 0 times a NaN or an infinite V is NaN), of which the run's rows are
// stored.  Later rows have more keys: they start first.  Three waves per SIMD: left to the
// compiler, the state in a loop takes registers for two (571 rows 30.1 us, with three 27.0; 155
// rows 8.2 and 8.8; one state over all runs 28.1 and 8.2).
__global__ __launch_bounds__(64 * kAttnWaves, 3) void causal_attention_kernel(CausalArgs a) {
    __shared__ AttnLds<kHeadDim> lds;
    const int m0 = (gridDim.x - 1 - blockIdx.x) * kAttnTile, h = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nq = min(kAttnTile, a.M - m0);
    const int qr = min(lane & 15, nq - 1);
    const int slot_q = static_cast<int>(a.row_slot[m0 + qr]), pos_q = static_cast<int>(a.row_pos[m0 + qr]);
    SplitFrag q[kHeadDim / 32];
    attn_query<kHeadDim>(a.q + static_cast<size_t>(m0 + qr) * kWidth + h * kHeadDim, lane, q);
    AttnState<kHeadDim> st;
    int r0 = 0;
    const float* kb = nullptr;  // the run's keys
    auto finish = [&](int r1) {  // the state's rows, r0 .. r1 - 1
        float out[4];
        attn_merge<kHeadDim>(lds, st, wave, lane, out);
        const int r = tid >> 4, rc = min(r, nq - 1);
        const bool own = r >= r0 && r < r1;
        attn_refine<kHeadDim>(a.q + static_cast<size_t>(m0 + rc) * kWidth + h * kHeadDim, kb, kb + a.kv_v_off,
                              [&] { return static_cast<int>(a.row_pos[m0 + rc]); }, 0.125f, own, lane, out);
        if (own) split_store4(a.out, split_off(m0 + r, h * kHeadDim + 4 * (tid & 15), kWidth), out);
    };
    while (true) {
        const int slot = __builtin_amdgcn_readlane(slot_q, r0);
        const uint32_t same = static_cast<uint32_t>(__ballot(slot_q == slot)) & ((1u << nq) - 1u) & ~((1u << r0) - 1u);
        const int r1 = r0 + __popc(same);                                // a slot's rows are consecutive
        const int kn = __builtin_amdgcn_readlane(pos_q, r1 - 1) + 1;     // and in order
        kb = a.kv + static_cast<size_t>(slot) * a.kv_slot_stride + a.kv_layer_off + static_cast<size_t>(h) * a.kv_cap * kHeadDim;
        const int pos = qr >= r0 && qr < r1 ? pos_q : -1;
        for (int c0 = wave * kAttnKeys; c0 < kn; c0 += kAttnWaves * kAttnKeys)
            attn_chunk<kHeadDim>(st, q, kb, kb + a.kv_v_off, c0, kn, pos, 0.125f, lane);
        if (__builtin_expect(r1 == nq, 1)) break;
        finish(r1);
        __syncthreads();  // the merge has read its LDS
        st = AttnState<kHeadDim>();
        r0 = r1;
    }
    finish(nq);
}

}  // namespace

hipError_t launch_ln_rows(const LnRowsArgs& a, hipStream_t s) {
    hipLaunchKernelGGL(ln_rows_kernel, dim3(a.rows), dim3(256), 0, s, a);
    return hipGetLastError();
}

namespace {

int ceil_div(int a, int b) { return (a + b - 1) / b; }

int device_cus() {
    static int cus = [] {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return 256;
        return n > 0 ? n : 256;
    }();
    return cus;
}

// The plan with the least estimated time, over every tile shape and split count.  The estimate
// is a least-squares fit to timings of these kernels on MI355X (every tile shape, 1..16 splits,
// 8 to 1200 rows of the 1280/5120-wide and the 1024..6144-wide shapes, weights from HBM; the
// plan it picks takes 2.6% longer than the best one on average), in microseconds:
//   launch + rounds tile + (k steps) (rounds^(2 per CU ? grow : 1) step + crowd max(0, r - free))
//       + (split: reduce + 1e-6 per_split splits M N)
// where r = workgroups / CUs and rounds = ceil(r).  `step` is a workgroup's time per 32 k when
// the chip is mostly idle; `crowd` is what it grows by when every CU is busy (weights and
// operands then share the L2s, and at 150 rows and more the matrix cores' own rate: 12-tile
// workgroups on 240 CUs reach 1.0 PFLOP/s of BF16 products, a large BF16 library product 1.13).
struct GemmCost {
    double launch, tile, step, crowd, reduce, per_split, grow, free;
};
constexpr GemmCost kGemmCost[2][kTiles] = {
    {   // FP32 weights
        {2.00, 1.44, 0.260, 0.0455, 2.94, 0.50, 0.555, 0.743},
        {2.65, 1.46, 0.239, 0.0621, 2.48, 0.68, 0.736, 0.0},
        {3.61, 1.02, 0.314, 0.111, 2.00, 1.37, 1.0, 0.497},
        {4.78, 1.29, 0.472, 0.237, 1.00, 1.43, 1.0, 0.5},
        {4.11, 2.11, 0.585, 0.406, 1.00, 1.06, 1.0, 0.411},
    },
    {   // BF16 weights
        {2.32, 0.935, 0.111, 0.0223, 2.47, 0.50, 0.874, 0.469},
        {2.39, 0.711, 0.136, 0.0260, 2.22, 1.73, 0.888, 0.494},
        {3.72, 0.0, 0.162, 0.0603, 1.60, 2.12, 1.0, 0.319},
        {4.30, 0.608, 0.291, 0.170, 1.00, 1.53, 1.0, 0.534},
        {3.79, 0.907, 0.358, 0.296, 1.00, 1.46, 1.0, 0.414},
    }};
}  // namespace

GemmSmallPlan gemm_small_plan(int M, int N, int K, int max_splits, bool bf16) {
    const int rt = ceil_div(M, 16), tiles = N / 16, cus = device_cus();
    if (rt > (bf16 ? 2 : 4)) return {0, 0};
    const int want = std::max(1, std::min(max_splits, cus / tiles));
    const int units = ceil_div(K, kSmallK), per = ceil_div(units, want);
    const GemmSmallPlan p{ceil_div(units, per), per * kSmallK};
    if (p.kchunk > 1280 || tiles * p.splits > (rt == 1 ? cus + cus * 9 / 16 : cus)) return {0, 0};  // (one row tile: 400 of 256 CUs)
    return p;
}

GemmPlan gemm_plan(int M, int N, int K, int max_splits, bool bf16, bool reduce) {
    const int rtot = ceil_div(M, 16), cus = device_cus();
    const double mn = static_cast<double>(M) * N;
    GemmPlan best{kTiles - 1, ceil_div(rtot, kTileRt[kTiles - 1]), 1, K};
    double best_t = 1e30;
    for (int i = 0; i < kTiles; ++i) {
        const GemmCost& c = kGemmCost[bf16][i];
        const int mb = ceil_div(rtot, kTileRt[i]);
        for (int s = 1; s <= max_splits; ++s) {
            const int kc = ceil_div(ceil_div(K, s), kGemmK) * kGemmK;
            if (ceil_div(K, kc) != s) continue;
            const double r = static_cast<double>(N / kGemmBn) * mb * s / cus, rounds = std::ceil(r);
            double t = c.launch + rounds * c.tile + kc / 32.0 * (std::pow(rounds, c.grow) * c.step + c.crowd * std::max(0.0, r - c.free));
            if (s > 1) t += (reduce ? c.reduce : 0.0) + c.per_split * s * mn / 1e6;
            if (t < best_t) {
                best_t = t;
                best = GemmPlan{i, mb, s, kc};
            }
        }
    }
    return best;
}

namespace {

template <typename WT, int EPI, bool SPLIT>
void launch_gemm_tile(const GemmArgs& a, const GemmPlan& p, hipStream_t s) {
    const dim3 grid(a.N / kGemmBn, p.mblocks, p.splits);
    gemm_tile<WT>(p.tile, [&](auto t) { hipLaunchKernelGGL((gemm_kernel<decltype(t), EPI, SPLIT>), grid, dim3(kGemmThreads), 0, s, a, p.kchunk); });
}

}  // namespace

namespace {

// Row tiles that gemm_small_kernel is built for: gemm_small_plan's four (BF16 weights two), and one for
// the GELU and SiLU epilogues, whose 5120 and 6144 columns are more than a workgroup per CU.
template <int EPI>
constexpr int gemm_small_tiles(bool bf16) {
    return EPI == kGemmGelu || EPI == kGemmSwiglu ? 1 : bf16 ? 2 : 4;
}
template <typename WT, int EPI, bool SPLIT>
void launch_gemm_small(const GemmArgs& a, const GemmSmallPlan& p, hipStream_t s) {
    const dim3 grid(a.N / 16, p.splits), block(64 * kSmallWaves);
    constexpr int RTS = gemm_small_tiles<EPI>(sizeof(WT) == 2);
    switch (ceil_div(a.M, 16)) {
        case 1: hipLaunchKernelGGL((gemm_small_kernel<WT, 1, EPI, SPLIT>), grid, block, 0, s, a, p.kchunk); break;
        case 2:
            if constexpr (RTS >= 2) hipLaunchKernelGGL((gemm_small_kernel<WT, 2, EPI, SPLIT>), grid, block, 0, s, a, p.kchunk);
            break;
        case 3:
            if constexpr (RTS >= 3) hipLaunchKernelGGL((gemm_small_kernel<WT, 3, EPI, SPLIT>), grid, block, 0, s, a, p.kchunk);
            break;
        default:
            if constexpr (RTS >= 4) hipLaunchKernelGGL((gemm_small_kernel<WT, 4, EPI, SPLIT>), grid, block, 0, s, a, p.kchunk);
            break;
    }
}

// Launches f<weight type, epilogue>() for the epilogue (kGemmStore and kGemmSwiglu: FP32 weights).
template <class F>
void with_epilogue(int epi, bool bf16, F f) {
    switch (epi) {
        case kGemmQkv: bf16 ? f(uint16_t{}, std::integral_constant<int, kGemmQkv>{}) : f(float{}, std::integral_constant<int, kGemmQkv>{}); break;
        case kGemmResid: bf16 ? f(uint16_t{}, std::integral_constant<int, kGemmResid>{}) : f(float{}, std::integral_constant<int, kGemmResid>{}); break;
        case kGemmGelu: bf16 ? f(uint16_t{}, std::integral_constant<int, kGemmGelu>{}) : f(float{}, std::integral_constant<int, kGemmGelu>{}); break;
        case kGemmStore: f(float{}, std::integral_constant<int, kGemmStore>{}); break;
        default: f(float{}, std::integral_constant<int, kGemmSwiglu>{}); break;
    }
}

// After the partial sums (splits > 1) or the results: the split reduce with the epilogue, the LayerNorm.
hipError_t finish_gemm(const GemmArgs& a, int epi, hipStream_t s) {
    if (a.splits == 1) {
        if (a.ln_out) hipLaunchKernelGGL(ln_rows_kernel, dim3(a.M), dim3(256), 0, s, LnRowsArgs{a.c, a.ln_out, a.ln_w, a.ln_b, a.M});
    } else if (a.ln_out) {
        hipLaunchKernelGGL(gemm_reduce_ln_kernel, dim3(a.M), dim3(256), 0, s, a);
    } else {
        const int w = epi == kGemmSwiglu ? 8 : 4;  // columns of a reduce thread
        const int rblocks = static_cast<int>(std::min<size_t>((static_cast<size_t>(a.M) * a.N / w + 255) / 256, 2048));
        with_epilogue(epi, false, [&](auto, auto e) { hipLaunchKernelGGL((gemm_reduce_kernel<decltype(e)::value>), dim3(rblocks), dim3(256), 0, s, a); });
    }
    return hipGetLastError();
}

hipError_t launch_gemm_plan(GemmArgs a, int epi, bool bf16, const GemmPlan& p, hipStream_t s) {
    a.splits = p.splits;
    if (p.splits > 1) {  // the partial tiles do not depend on the epilogue
        if (bf16) launch_gemm_tile<uint16_t, kGemmStore, true>(a, p, s);
        else launch_gemm_tile<float, kGemmStore, true>(a, p, s);
    } else {
        with_epilogue(epi, bf16, [&](auto w, auto e) { launch_gemm_tile<decltype(w), decltype(e)::value, false>(a, p, s); });
    }
    return finish_gemm(a, epi, s);
}

hipError_t launch_gemm_small_plan(GemmArgs a, int epi, bool bf16, const GemmSmallPlan& p, hipStream_t s) {
    a.splits = p.splits;
    if (p.splits > 1) {
        if (bf16) launch_gemm_small<uint16_t, kGemmStore, true>(a, p, s);
        else launch_gemm_small<float, kGemmStore, true>(a, p, s);
    } else {
        with_epilogue(epi, bf16, [&](auto w, auto e) { launch_gemm_small<decltype(w), decltype(e)::value, false>(a, p, s); });
    }
    return finish_gemm(a, epi, s);
}

}  // namespace

hipError_t launch_gemm(const GemmArgs& a, int epi, bool bf16, hipStream_t s) {
    if (a.N % kGemmBn || a.K % kGemmK || a.M < 1 || !a.ws) return hipErrorInvalidValue;
    if ((epi == kGemmStore || epi == kGemmSwiglu) && bf16) return hipErrorInvalidValue;  // FP32 weights only (the Qwen decoder)
    if (a.ln_out && (epi != kGemmResid || a.N != kWidth)) return hipErrorInvalidValue;
    if (split_elems(a.M, a.K) * 2 >= 0x40000000u) return hipErrorInvalidValue;  // 32-bit operand offsets
    const int splits = std::max(1, static_cast<int>(std::min<size_t>(kGemmMaxSplits, kGemmWsFloats / (static_cast<size_t>(a.M) * a.N))));
    const GemmSmallPlan small = gemm_small_plan(a.M, a.N, a.K, splits, bf16);
    const bool one_tile = (epi == kGemmGelu || epi == kGemmSwiglu) && small.splits == 1;
    if (small.splits && !(one_tile && a.M > 16)) return launch_gemm_small_plan(a, epi, bf16, small, s);
    return launch_gemm_plan(a, epi, bf16, gemm_plan(a.M, a.N, a.K, splits, bf16, true), s);
}

hipError_t launch_causal_attention(const CausalArgs& a, hipStream_t s) {
    hipLaunchKernelGGL(causal_attention_kernel, dim3(ceil_div(a.M, kAttnTile), kHeads), dim3(64 * kAttnWaves), 0, s, a);
    return hipGetLastError();
}

}  // namespace itts
