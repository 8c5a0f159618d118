// EnhancedCodec::decode (src/codec.cpp:57-72), the consumer of the GPT's semantic codes, on
// the MI355X: codes [T] -> features [2T][1024], time-major.
//
//   x      = out_project(codebook[codes])                       (codec.cpp:57-63; 8 -> 1024)
//   x      = LN(conv7(x))                                       (vocos_pass, codec.cpp:36-40; 1024 -> 384)
//   12 x:  x += gamma * pwconv2(GELU(pwconv1(LN(dwconv7(x))))) (codec.cpp:41-47; 384 -> 2048 -> 384)
//   y      = decoder.1(LN(x))                                   (codec.cpp:48; 384 -> 1024)
//   out    = conv3(nearest_x2(y))                               (codec.cpp:68-70; 1024 -> 1024 over 2T)
// LayerNorm eps 1e-6, biased variance (kernels.metal:618-669 with codec.cpp:28); GELU is the
// codec's erf form, erf from the Abramowitz-Stegun 7.1.26 polynomial (kernels.metal:3133-3137);
// "same" convolutions pad kernel/2 zeros on each side (kernels.metal:1397-1426, 1516-1541).
//
// Kernels (41 launches per decode, 42 when the up conv's K is split):
//   * codec_lookup: one workgroup per code, the 8-wide codebook row times out_project.
//   * codec_gemm<EPI>: C = A W^T + bias on the matrix cores with split operands (gemm_core.h); every
//     A is written split by the kernel before.  A "same" convolution of kernel k over time-major
//     rows is this GEMM with K = k * Cin: row t of A is the k consecutive input rows t .. t + k - 1
//     of the zero-padded input, so a lane's operand row moves down one row per tap, and the
//     weights are stored [Cout][k][Cin].
//   * The conv3 over the doubled rows reads row t twice: out[2t] = w0 y[t-1] + (w1 + w2) y[t] and
//     out[2t+1] = (w0 + w1) y[t] + w2 y[t+1].  It is one two-tap GEMM over y with 2048 columns
//     (even, then odd output rows, the odd ones a row further down): two thirds of the
//     products, and no doubled input.
//   * codec_rows: everything between two GEMMs of the ConvNeXt stack in one launch: the split sums,
//     bias, gamma and residual (or the first LayerNorm) of a row and its neighbours, then the
//     depthwise conv7 and LayerNorm (or the final LayerNorm).  Each row is formed by the
//     workgroups of four row pairs instead of a launch of its own.
// A decode of a given length is captured once as a HIP graph and replayed (the launches bound
// short decodes); the padding rows are written by kernels, not memsets.
#include <type_traits>
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <stdexcept>
#include <string>
#include <unordered_map>
#include <vector>

#include "gemm_core.h"
#include "itts_gpt.h"

namespace itts {
namespace {

constexpr int kCW = 1024;        // codec feature width
constexpr int kCH = 384;         // ConvNeXt width
constexpr int kCF = 2048;        // ConvNeXt hidden width
constexpr int kCBlocks = 12;
constexpr int kCK = 7;           // embed / depthwise kernel
constexpr int kUpK = 3;          // up conv kernel
constexpr int kUpN = 2 * kCW;    // up conv as a GEMM: even and odd output rows
constexpr int kUpTaps = 2;
constexpr int kCodebook = 8192;
constexpr int kCodeDim = 8;
constexpr int kMaxCodes = 5000;  // codec.cpp:58
constexpr float kCodecEps = 1e-6f;

// 0.5 x (1 + erf(x / sqrt 2)), erf by Abramowitz & Stegun 7.1.26 (|error| <= 1.5e-7), the form
// the reference's codec GELU evaluates.
__device__ __forceinline__ float codec_gelu(float x) {
    const float v = x * 0.7071067811865475f, a = fabsf(v), t = 1.0f / (1.0f + 0.3275911f * a);
    const float p = (((((1.061405429f * t - 1.453152027f) * t) + 1.421413741f) * t - 0.284496736f) * t + 0.254829592f) * t;
    float erf = 1.0f - p * expf(-a * a);
    if (v < 0) erf = -erf;
    return 0.5f * x * (1.0f + erf);
}

// Row r of the embed conv's zero-padded input (T + 2 pad rows), split: rows pad .. pad + T - 1 are
// the projected codebook rows of the codes, the others zero.  The two padding rows of the up
// conv's input (0 and T + 1 of ypad) are cleared here too.
__global__ __launch_bounds__(256) void codec_lookup_kernel(const uint32_t* codes, const float* cb, const float* w, const float* b,
                                                           uint16_t* out, uint16_t* ypad, int T, int pad) {
    const int r = blockIdx.x, tid = threadIdx.x;
    const float zero[4] = {0.f, 0.f, 0.f, 0.f};
    if (r < 2) split_store4(ypad, split_off(r * (T + 1), 4 * tid, kCW), zero);
    if (r < pad || r >= T + pad) {
        split_store4(out, split_off(r, 4 * tid, kCW), zero);
        return;
    }
    const float* e = cb + static_cast<size_t>(codes[r - pad]) * kCodeDim;
    const f32x4 e0 = *reinterpret_cast<const f32x4*>(e), e1 = *reinterpret_cast<const f32x4*>(e + 4);
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int o = 4 * tid + i;
        const f32x4 w0 = *reinterpret_cast<const f32x4*>(w + static_cast<size_t>(o) * kCodeDim);
        const f32x4 w1 = *reinterpret_cast<const f32x4*>(w + static_cast<size_t>(o) * kCodeDim + 4);
        float acc = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; ++j) acc = __builtin_fmaf(w0[j], e0[j], acc);
#pragma unroll
        for (int j = 0; j < 4; ++j) acc = __builtin_fmaf(w1[j], e1[j], acc);
        v[i] = acc + b[o];
    }
    split_store4(out, split_off(r, 4 * tid, kCW), v);
}

// kEpiPartial: raw sums of K range z to ws[z].  kEpiGelu: GELU, split.  kEpiShift: + bias, split,
// one row down (the up conv's padded input).  kEpiUp: + bias, columns n >= 1024 to the odd rows.
enum CodecEpi : int { kEpiPartial = 0, kEpiGelu = 1, kEpiShift = 2, kEpiUp = 3 };

struct CodecGemm {
    const uint16_t* a;   // split operand (of a convolution: the padded rows, kCW wide)
    int a_rows;          // rows of it
    const float* w;      // [N][K]
    const float* bias;   // [N]
    float* c;            // kEpiUp output
    uint16_t* cs;        // kEpiGelu, kEpiShift output
    int M, N, K;
    float* ws;           // partial sums [splits][M][N]
    int kchunk;          // K per split
};

// One result of a GEMM: the sum of row `row` and column `col` (of K range z).
template <int EPI>
__device__ __forceinline__ void codec_store_one(const CodecGemm& g, int z, int row, int col, float sum) {
    if (row >= g.M) return;
    if constexpr (EPI == kEpiPartial) g.ws[(static_cast<size_t>(z) * g.M + row) * g.N + col] = sum;
    else if constexpr (EPI == kEpiGelu) split_store(g.cs, split_off(row, col, g.N), codec_gelu(sum + g.bias[col]));
    else if constexpr (EPI == kEpiShift) split_store(g.cs, split_off(row + 1, col, g.N), sum + g.bias[col]);
    else g.c[(2 * static_cast<size_t>(row) + (col >= kCW ? 1 : 0)) * kCW + (col & (kCW - 1))] = sum + g.bias[col];
}

template <class T, int EPI, bool CONV>
__global__ __launch_bounds__(kGemmThreads) void codec_gemm_kernel(CodecGemm g) {
    __shared__ __align__(16) uint8_t lds[T::kLdsBytes];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const auto [bx, by, bz] = gemm_place();
    const int kb = bz * g.kchunk, nst = (min(g.K, kb + g.kchunk) - kb) / 32;
    uint16_t* ring = reinterpret_cast<uint16_t*>(lds);
    if (wave >= 4) {
        gemm_loader<T>(ring, g.w + static_cast<size_t>(bx) * T::BN * g.K + kb, g.K, nst, tid - 256);
        return;
    }
    constexpr int TR = T::TR, TC = T::TC;
    const int wr = wave / T::WC, wc = wave % T::WC;
    const int tile0 = by * T::RT + wr * TR;
    const int akt = CONV ? kCW / 32 : g.K / 32;  // k steps of an operand row
    const __amdgpu_buffer_rsrc_t ars = gemm_rsrc(g.a, static_cast<uint32_t>(split_elems(g.a_rows, akt * 32) * 2));
    GemmAcc<T> sums;
    if constexpr (CONV) {
        // k step s is step s % 32 of tap s / 32, which reads a row further down; rows past the
        // operand's buffer read as zero (result rows past M only)
        const int row0 = tile0 * 16 + (lane & 15) + (bx * T::BN >= kCW ? 1 : 0);  // (the up conv's odd rows)
        gemm_compute<T>(
            ring, ars,
            [&](int i, int s) {
                const int sg = kb / 32 + s, row = row0 + 16 * i + (sg >> 5);
                return GemmOff{static_cast<uint32_t>(row >> 4) * (kCW / 32 * kTileElems * 2) + ((row & 15) + (lane & 48)) * 16,
                               static_cast<uint32_t>(sg & 31) * (kTileElems * 2)};
            },
            nst, wc, lane, sums);
    } else {
        const int tiles = (g.M + 15) / 16;
        uint32_t off[TR];
#pragma unroll
        for (int i = 0; i < TR; ++i) off[i] = (static_cast<uint32_t>(min(tile0 + i, tiles - 1)) * akt + kb / 32) * (kTileElems * 2) + lane * 16;
        gemm_compute<T>(
            ring, ars, [&](int i, int s) { return GemmOff{off[i], static_cast<uint32_t>(s) * (kTileElems * 2)}; }, nst, wc, lane, sums);
    }
    const int n0 = bx * T::BN + wc * TC * 16;  // the wave's first column
    const auto dot = [&](int m, int n) {
        return gemm_dot(g.w + static_cast<size_t>(n0 + n) * g.K + kb, nst * 32, [&](int k) {
            const int kk = kb + k;  // of a convolution: tap kk / kCW, a row further down each
            return split_value(g.a + (CONV ? split_off(m + (n0 >= kCW ? 1 : 0) + kk / kCW, kk % kCW, kCW) : split_off(m, kk, g.K)));
        });
    };
    const bool suspect = sums.suspect();
    if constexpr (EPI == kEpiPartial || EPI == kEpiUp) {
        if (__builtin_expect(suspect, 0)) {
            gemm_refine<T>(lds, g.M, tile0, wave, lane, sums, dot, [&](int m, int n, float v) { codec_store_one<EPI>(g, bz, m, n0 + n, v); });
            return;
        }
    }
    f32x4 acc[TR][TC];
    sums.sum(acc);
    const int col0 = n0 + (lane & 15);
    if constexpr (EPI == kEpiPartial) {
        gemm_store_partial<T>(g.ws + static_cast<size_t>(bz) * g.M * g.N, g.M, g.N, tile0, col0, lane, acc);
    } else {
        float bias[TC];
#pragma unroll
        for (int c = 0; c < TC; ++c) bias[c] = g.bias[col0 + 16 * c];
        if constexpr (EPI == kEpiGelu) {
            gemm_store_split<T, false>(
                lds, wave, lane, g.cs, g.M, g.N, 0, tile0, n0, [&](int i, int c, int r) { return codec_gelu(acc[i][c][r] + bias[c]); }, suspect,
                [&](int m, int n) { return codec_gelu(dot(m, n) + g.bias[n0 + n]); });
        } else if constexpr (EPI == kEpiShift) {
            gemm_store_split<T, false>(
                lds, wave, lane, g.cs, g.M, g.N, 1, tile0, n0, [&](int i, int c, int r) { return acc[i][c][r] + bias[c]; }, suspect,
                [&](int m, int n) { return dot(m, n) + g.bias[n0 + n]; });
        } else {
#pragma unroll
            for (int i = 0; i < TR; ++i) {
                const int row = (tile0 + i) * 16 + 4 * (lane >> 4);
#pragma unroll
                for (int c = 0; c < TC; ++c)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        acc[i][c][r] += bias[c];
                        pin_value(acc[i][c][r]);
                    }
                const int odd = n0 >= kCW ? 1 : 0;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (row + r < g.M) {
                        float* p = g.c + (2 * static_cast<size_t>(row + r) + odd) * kCW + (col0 & (kCW - 1));
#pragma unroll
                        for (int c = 0; c < TC; ++c) p[16 * c] = acc[i][c][r];
                    }
            }
        }
    }
}

// The same for up to 16 RT rows of an operand that is not a convolution's (gemm_core.h, gemm_small).
template <int RT, int EPI>
__global__ __launch_bounds__(64 * kSmallWaves) void codec_gemm_small_kernel(CodecGemm g) {
    __shared__ GemmSmallLds<RT> lds;
    const int kb = blockIdx.y * g.kchunk, nst = (min(g.K, kb + g.kchunk) - kb) / 32;
    float sum[2];
    gemm_small<float, RT>(lds, g.w + static_cast<size_t>(blockIdx.x) * 16 * g.K + kb, g.K, nst,
                          gemm_rsrc(g.a, static_cast<uint32_t>(split_elems(g.M, g.K) * 2)), kb / 32 * (kTileElems * 2),
                          g.K / 32 * (kTileElems * 2), g.M, [&](int m, int k) { return split_value(g.a + split_off(m, kb + k, g.K)); }, sum);
#pragma unroll
    for (int q = 0; q < (RT > 2 ? 2 : 1); ++q)
        codec_store_one<EPI>(g, blockIdx.y, (threadIdx.x >> 4) + 32 * q, blockIdx.x * 16 + (threadIdx.x & 15), sum[q]);
}

// The up conv's splits, added in split order, + bias; a thread takes four columns.
template <int SM>
__global__ __launch_bounds__(256) void codec_up_reduce_kernel(CodecGemm g, int splits) {
    const size_t e = (static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x) * 4, plane = static_cast<size_t>(g.M) * kUpN;
    if (e >= plane) return;
    const size_t row = e / kUpN;
    const int n = static_cast<int>(e % kUpN);
    f32x4 w[SM];
#pragma unroll
    for (int z = 0; z < SM; ++z) w[z] = *reinterpret_cast<const f32x4*>(g.ws + static_cast<size_t>(min(z, splits - 1)) * plane + e);
    f32x4 d = w[0];
#pragma unroll
    for (int z = 1; z < SM; ++z)
        if (z < splits) d += w[z];
    *reinterpret_cast<f32x4*>(g.c + (2 * row + (n >= kCW ? 1 : 0)) * kCW + (n & (kCW - 1))) = d + *reinterpret_cast<const f32x4*>(g.bias + n);
}

// LayerNorm of a 384-wide row held as 6 values per lane (columns lane + 64 i): mean, then
// the biased variance of the centred values, eps 1e-6.
__device__ __forceinline__ void ln384(float (&v)[6], const float* gw, const float* gb, int lane) {
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < 6; ++i) s += v[i];
    const float mean = wave_sum(s) / float(kCH);
    float q = 0.0f;
#pragma unroll
    for (int i = 0; i < 6; ++i) {
        const float d = v[i] - mean;
        q += d * d;
    }
    const float inv = 1.0f / sqrtf(wave_sum(q) / float(kCH) + kCodecEps);
#pragma unroll
    for (int i = 0; i < 6; ++i) {
        const int c = lane + 64 * i;
        v[i] = (v[i] - mean) * inv * gw[c] + gb[c];
    }
}

// Rows between the GEMMs.  x row = LayerNorm(split sum + bias) (FIRST: after the embed conv) or
// x_in + gamma * (split sum + bias) (after pwconv2); then, with DW, the depthwise conv7 of x (same
// padding) and LayerNorm, else LayerNorm alone; split.  A workgroup of eight waves owns two rows:
// with DW each wave forms one of the eight rows they read (three before, three after, zeros
// outside [0, T)), so the neighbours' split sums are read again (from L2) instead of a launch
// between them; the owned rows go to x_out, which is not x_in (the neighbours read that).
struct CodecRows {
    const float* ws;
    int splits, T;
    const float *bias, *gamma, *x_in;
    float* x_out;
    const float *fw, *fb;    // FIRST: its LayerNorm
    const float *dw, *db;    // depthwise conv
    const float *lw, *lb;    // the LayerNorm at the end
    uint16_t* out;
};
constexpr int kRowsOwn = 2, kRowsWaves = 8;

template <bool FIRST, bool DW>
__global__ __launch_bounds__(64 * kRowsWaves) void codec_rows_kernel(CodecRows a) {
    __shared__ float xs[kRowsWaves][kCH];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int halo = DW ? kCK / 2 : 0;
    const int t0 = blockIdx.x * kRowsOwn, t = t0 + wave - halo;
    const bool live = t >= 0 && t < a.T && wave < kRowsOwn + 2 * halo;
    // the depthwise weights of the owned rows' waves, requested with the split sums
    float dw[6][kCK], db[6];
    if (DW && wave < kRowsOwn) {
#pragma unroll
        for (int i = 0; i < 6; ++i) {
            db[i] = a.db[lane + 64 * i];
#pragma unroll
            for (int k = 0; k < kCK; ++k) dw[i][k] = a.dw[(lane + 64 * i) * kCK + k];
        }
    }
    float v[6];
#pragma unroll
    for (int i = 0; i < 6; ++i) v[i] = 0.0f;
    if (live) {
        const size_t row = static_cast<size_t>(t) * kCH + lane, plane = static_cast<size_t>(a.T) * kCH;
        float res[6], bias[6], gamma[6];
#pragma unroll
        for (int i = 0; i < 6; ++i) {
            bias[i] = a.bias[lane + 64 * i];
            res[i] = FIRST ? 0.0f : a.x_in[row + 64 * i];
            gamma[i] = FIRST ? 1.0f : a.gamma[lane + 64 * i];
        }
        // every split's partial of a group requested before its first add; in split order
        auto sum = [&](auto sm) {
            constexpr int SM = decltype(sm)::value;
            for (int z0 = 0; z0 < a.splits; z0 += SM) {
                float w[SM][6];
#pragma unroll
                for (int z = 0; z < SM; ++z)
#pragma unroll
                    for (int i = 0; i < 6; ++i) w[z][i] = a.ws[static_cast<size_t>(min(z0 + z, a.splits - 1)) * plane + row + 64 * i];
#pragma unroll
                for (int z = 0; z < SM; ++z)
                    if (z0 + z < a.splits) {
#pragma unroll
                        for (int i = 0; i < 6; ++i) v[i] += w[z][i];
                    }
            }
        };
        if (a.splits <= 2) sum(std::integral_constant<int, 2>{});
        else if (a.splits <= 4) sum(std::integral_constant<int, 4>{});
        else sum(std::integral_constant<int, 8>{});
#pragma unroll
        for (int i = 0; i < 6; ++i) v[i] = FIRST ? v[i] + bias[i] : res[i] + (v[i] + bias[i]) * gamma[i];  // codec.cpp:46: x + scale(h, gamma)
        if constexpr (FIRST) ln384(v, a.fw, a.fb, lane);
        if (DW && wave >= halo && wave < halo + kRowsOwn) {
#pragma unroll
            for (int i = 0; i < 6; ++i) a.x_out[row + 64 * i] = v[i];
        }
    }
    int ot = t;
    if constexpr (DW) {
#pragma unroll
        for (int i = 0; i < 6; ++i) xs[wave][lane + 64 * i] = v[i];
        __syncthreads();
        ot = t0 + wave;
        if (wave >= kRowsOwn || ot >= a.T) return;
#pragma unroll
        for (int i = 0; i < 6; ++i) {
            const int c = lane + 64 * i;
            float acc = db[i];
#pragma unroll
            for (int k = 0; k < kCK; ++k) acc += xs[wave + k][c] * dw[i][k];
            v[i] = acc;
        }
    } else if (!live) {
        return;
    }
    ln384(v, a.lw, a.lb, lane);
#pragma unroll
    for (int i = 0; i < 6; ++i) split_store(a.out, split_off(ot, lane + 64 * i, kCH), v[i]);
}

#define CODEC_CHECK(x)                                                                                                  \
    do {                                                                                                                \
        const hipError_t e_ = (x);                                                                                      \
        if (e_ != hipSuccess) throw std::runtime_error(std::string("HIP error ") + hipGetErrorString(e_) + " in " #x); \
    } while (0)

template <typename T>
struct Buf {
    T* p = nullptr;
    size_t n = 0;
    Buf() = default;
    Buf(const Buf&) = delete;
    Buf& operator=(const Buf&) = delete;
    ~Buf() {
        if (p) (void)hipFree(p);
    }
    bool ensure(size_t count) {  // true when the buffer moved
        if (count <= n) return false;
        if (p) CODEC_CHECK(hipFree(p));
        p = nullptr;
        n = 0;
        CODEC_CHECK(hipMalloc(&p, count * sizeof(T)));
        n = count;
        return true;
    }
    void upload(const std::vector<T>& v) {
        ensure(v.size());
        CODEC_CHECK(hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
    }
};

// At most this many K splits of a GEMM whose partial sums the next kernel adds anyway.
constexpr int kCodecSplits = 32;
constexpr size_t kCodecWsFloats = size_t(16) << 20;  // and at most this many partial sums, except of one split

}  // namespace

// A named host tensor as the constructor takes it.
struct CodecTensor {
    const float* data;
    std::vector<int64_t> shape;
};

struct CodecEngine {
    hipStream_t stream = nullptr;
    hipEvent_t ev[2] = {};
    Buf<float> cb, op_w, op_b, emb_w, emb_b, n0_w, n0_b, fin_w, fin_b, dec_w, dec_b, up_w, up_b;
    struct Block {
        Buf<float> dw, db, lw, lb, w1, b1, w2, b2, gamma;
    } blk[kCBlocks];
    Buf<uint16_t> xpad, hn, f, ypad;  // split GEMM operands (gemm_core.h)
    Buf<float> x[2], out, ws;
    Buf<uint32_t> dcodes;
    // Decodes of one length replay a captured graph (ITTS_CODEC_GRAPHS=0: eager launches).  A
    // buffer that moves bumps `generation`, and graphs captured before are dropped.
    bool use_graphs = true;
    uint64_t generation = 0, graph_generation = 0;
    std::unordered_map<int, hipGraphExec_t> graphs;

    static GemmPlan plan(int M, int N, int K, int max_splits, bool reduce) {
        const size_t mn = static_cast<size_t>(M) * N;
        return gemm_plan(M, N, K, std::max(1, std::min<int>(max_splits, static_cast<int>(kCodecWsFloats / mn))), false, reduce);
    }
    static GemmPlan embed_plan(int T) { return plan(T, kCH, kCK * kCW, kCodecSplits, false); }
    static GemmPlan up_plan(int T) { return plan(T, kUpN, kUpTaps * kCW, 8, true); }
    template <class T>
    void grow(Buf<T>& b, size_t n) {
        if (!b.ensure(n)) return;
        ++generation;
        if (std::is_same_v<T, uint16_t>)  // padding rows of operands: finite, whatever the memory held
            CODEC_CHECK(hipMemsetAsync(b.p, 0, b.n * sizeof(T), stream));
    }
    // Every buffer a decode of T codes touches, sized before anything is queued (and captured).
    void reserve(int T) {
        const size_t pad = kCK / 2;
        grow(dcodes, T);
        grow(xpad, split_elems(T + 2 * pad, kCW));
        for (auto& b : x) grow(b, static_cast<size_t>(T) * kCH);
        grow(hn, split_elems(T, kCH));
        grow(f, split_elems(T, kCF));
        grow(ypad, split_elems(T + 2, kCW));
        grow(out, static_cast<size_t>(2 * T) * kCW);
        grow(ws, static_cast<size_t>(T) * std::max({embed_plan(T).splits * kCH, cut(T, kCH, kCF, kCodecSplits).splits() * kCH, up_plan(T).splits * kUpN}));
    }

    template <int EPI>
    void gemm_few(CodecGemm g, const GemmSmallPlan& p) {
        if (EPI == kEpiPartial && ws.n < static_cast<size_t>(p.splits) * g.M * g.N) throw std::logic_error("codec split-K workspace not reserved");
        g.ws = ws.p;
        g.kchunk = p.kchunk;
        const dim3 grid(g.N / 16, p.splits), block(64 * kSmallWaves);
        switch ((g.M + 15) / 16) {
            case 1: hipLaunchKernelGGL((codec_gemm_small_kernel<1, EPI>), grid, block, 0, stream, g); break;
            case 2: hipLaunchKernelGGL((codec_gemm_small_kernel<2, EPI>), grid, block, 0, stream, g); break;
            case 3: hipLaunchKernelGGL((codec_gemm_small_kernel<3, EPI>), grid, block, 0, stream, g); break;
            default: hipLaunchKernelGGL((codec_gemm_small_kernel<4, EPI>), grid, block, 0, stream, g); break;
        }
        CODEC_CHECK(hipGetLastError());
    }

    // A plan's cut with what launches it: few rows of a plain operand take the small kernel.
    struct Cut {
        GemmSmallPlan few;
        GemmPlan tiles;
        int splits() const { return few.splits ? few.splits : tiles.splits; }
    };
    static Cut cut(int M, int N, int K, int max_splits) {
        return {gemm_small_plan(M, N, K, max_splits, false), plan(M, N, K, max_splits, false)};
    }
    template <int EPI>
    void gemm(const CodecGemm& g, const Cut& c) {
        if (c.few.splits) gemm_few<EPI>(g, c.few);
        else gemm<EPI, false>(g, c.tiles);
    }
    template <int EPI, bool CONV>
    void gemm(CodecGemm g, const GemmPlan& p) {
        if (g.N % kGemmBn || g.K % kGemmK || g.M < 1) throw std::logic_error("codec GEMM shape");
        if (EPI == kEpiPartial && ws.n < static_cast<size_t>(p.splits) * g.M * g.N) throw std::logic_error("codec split-K workspace not reserved");
        if (EPI != kEpiPartial && p.splits != 1) throw std::logic_error("codec GEMM splits");
        g.ws = ws.p;
        g.kchunk = p.kchunk;
        gemm_tile<float>(p.tile, [&](auto t) {
            hipLaunchKernelGGL((codec_gemm_kernel<decltype(t), EPI, CONV>), dim3(g.N / kGemmBn, p.mblocks, p.splits), dim3(kGemmThreads), 0, stream, g);
        });
        CODEC_CHECK(hipGetLastError());
    }
    std::string last_error;

    ~CodecEngine() {
        drop_graphs();
        for (auto& e : ev)
            if (e) (void)hipEventDestroy(e);
        if (stream) (void)hipStreamDestroy(stream);
    }

    // EnhancedCodec::EnhancedCodec (codec.cpp:5-20): the shapes the decode path reads, with the
    // reference's message.
    void create(const std::unordered_map<std::string, CodecTensor>& t) {
        auto get = [&](const std::string& name, std::vector<int64_t> shape) -> const float* {
            auto it = t.find(name);
            if (it == t.end()) throw std::runtime_error("Missing tensor: " + name);
            if (it->second.shape != shape) throw std::runtime_error("Unsupported 2.5 codec shape: " + name);
            return it->second.data;
        };
        auto vec = [](const float* p, size_t n) { return std::vector<float>(p, p + n); };
        // [Cout][Cin][k] -> [Cout][k][Cin]: a conv becomes a GEMM over k consecutive input rows
        auto conv_w = [](const float* p, int cout, int cin, int k) {
            std::vector<float> r(static_cast<size_t>(cout) * cin * k);
            for (int o = 0; o < cout; ++o)
                for (int i = 0; i < cin; ++i)
                    for (int j = 0; j < k; ++j)
                        r[(static_cast<size_t>(o) * k + j) * cin + i] = p[(static_cast<size_t>(o) * cin + i) * k + j];
            return r;
        };
        const std::string q = "codec.quantizer.quantizers.0", d = "codec.decoder.0";
        cb.upload(vec(get(q + ".codebook.weight", {kCodebook, kCodeDim}), static_cast<size_t>(kCodebook) * kCodeDim));
        op_w.upload(vec(get(q + ".out_project.weight", {kCW, kCodeDim}), static_cast<size_t>(kCW) * kCodeDim));
        op_b.upload(vec(get(q + ".out_project.bias", {kCW}), kCW));
        emb_w.upload(conv_w(get(d + ".embed.weight", {kCH, kCW, kCK}), kCH, kCW, kCK));
        emb_b.upload(vec(get(d + ".embed.bias", {kCH}), kCH));
        n0_w.upload(vec(get(d + ".norm.weight", {kCH}), kCH));
        n0_b.upload(vec(get(d + ".norm.bias", {kCH}), kCH));
        for (int i = 0; i < kCBlocks; ++i) {
            const std::string l = d + ".convnext." + std::to_string(i);
            Block& b = blk[i];
            b.dw.upload(vec(get(l + ".dwconv.weight", {kCH, 1, kCK}), static_cast<size_t>(kCH) * kCK));
            b.db.upload(vec(get(l + ".dwconv.bias", {kCH}), kCH));
            b.lw.upload(vec(get(l + ".norm.weight", {kCH}), kCH));
            b.lb.upload(vec(get(l + ".norm.bias", {kCH}), kCH));
            b.w1.upload(vec(get(l + ".pwconv1.weight", {kCF, kCH}), static_cast<size_t>(kCF) * kCH));
            b.b1.upload(vec(get(l + ".pwconv1.bias", {kCF}), kCF));
            b.w2.upload(vec(get(l + ".pwconv2.weight", {kCH, kCF}), static_cast<size_t>(kCH) * kCF));
            b.b2.upload(vec(get(l + ".pwconv2.bias", {kCH}), kCH));
            b.gamma.upload(vec(get(l + ".gamma", {kCH}), kCH));
        }
        fin_w.upload(vec(get(d + ".final_layer_norm.weight", {kCH}), kCH));
        fin_b.upload(vec(get(d + ".final_layer_norm.bias", {kCH}), kCH));
        dec_w.upload(vec(get("codec.decoder.1.weight", {kCW, kCH}), static_cast<size_t>(kCW) * kCH));
        dec_b.upload(vec(get("codec.decoder.1.bias", {kCW}), kCW));
        // even rows: taps w0 | w1 + w2 (rows t - 1, t); odd rows: w0 + w1 | w2 (rows t, t + 1)
        const float* uw = get("codec.up.weight", {kCW, kCW, kUpK});
        const float* ub = get("codec.up.bias", {kCW});
        std::vector<float> up(static_cast<size_t>(kUpN) * kUpTaps * kCW), upb(kUpN);
        for (int o = 0; o < kCW; ++o) {
            float *ev = &up[static_cast<size_t>(o) * kUpTaps * kCW], *od = &up[static_cast<size_t>(kCW + o) * kUpTaps * kCW];
            for (int i = 0; i < kCW; ++i) {
                const float* w = uw + (static_cast<size_t>(o) * kCW + i) * kUpK;
                ev[i] = w[0];
                ev[kCW + i] = w[1] + w[2];
                od[i] = w[0] + w[1];
                od[kCW + i] = w[2];
            }
            upb[o] = upb[kCW + o] = ub[o];
        }
        up_w.upload(up);
        up_b.upload(upb);
        const char* env = std::getenv("ITTS_CODEC_GRAPHS");
        use_graphs = !(env && std::strcmp(env, "0") == 0);
        CODEC_CHECK(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
        for (auto& e : ev) CODEC_CHECK(hipEventCreate(&e));
    }

    void check_codes(const uint32_t* codes, uint32_t n) const {
        bool ok = n >= 1 && n <= static_cast<uint32_t>(kMaxCodes) && codes;
        for (uint32_t i = 0; ok && i < n; ++i) ok = codes[i] < static_cast<uint32_t>(kCodebook);
        if (!ok) throw std::invalid_argument("Codec expects 1..5000 code IDs in [0,8192)");
    }

    // The whole decode of T codes already in dcodes, queued on the stream (kernels only, into
    // buffers reserve(T) sized); result in out.
    void enqueue(int T) {
        const int pad = kCK / 2;
        hipStream_t s = stream;
        hipLaunchKernelGGL(codec_lookup_kernel, dim3(T + 2 * pad), dim3(256), 0, s, dcodes.p, cb.p, op_w.p, op_b.p, xpad.p, ypad.p, T, pad);
        CODEC_CHECK(hipGetLastError());
        const dim3 rows((T + kRowsOwn - 1) / kRowsOwn), threads(64 * kRowsWaves);
        const GemmPlan pe = embed_plan(T), pu = up_plan(T);
        const Cut p1 = cut(T, kCF, kCH, 1), p2 = cut(T, kCH, kCF, kCodecSplits), pd = cut(T, kCW, kCH, 1);
        gemm<kEpiPartial, true>({xpad.p, T + 2 * pad, emb_w.p, nullptr, nullptr, nullptr, T, kCH, kCK * kCW, nullptr, 0}, pe);
        hipLaunchKernelGGL((codec_rows_kernel<true, true>), rows, threads, 0, s,
                           CodecRows{ws.p, pe.splits, T, emb_b.p, nullptr, nullptr, x[0].p, n0_w.p, n0_b.p, blk[0].dw.p, blk[0].db.p, blk[0].lw.p,
                                     blk[0].lb.p, hn.p});
        CODEC_CHECK(hipGetLastError());
        for (int i = 0; i < kCBlocks; ++i) {
            const Block& b = blk[i];
            gemm<kEpiGelu>({hn.p, T, b.w1.p, b.b1.p, nullptr, f.p, T, kCF, kCH, nullptr, 0}, p1);
            gemm<kEpiPartial>({f.p, T, b.w2.p, nullptr, nullptr, nullptr, T, kCH, kCF, nullptr, 0}, p2);
            CodecRows r{ws.p, p2.splits(), T, b.b2.p, b.gamma.p, x[i & 1].p, x[1 - (i & 1)].p, nullptr, nullptr, nullptr, nullptr, fin_w.p, fin_b.p, hn.p};
            if (i + 1 < kCBlocks) {
                const Block& n = blk[i + 1];
                r.dw = n.dw.p;
                r.db = n.db.p;
                r.lw = n.lw.p;
                r.lb = n.lb.p;
                hipLaunchKernelGGL((codec_rows_kernel<false, true>), rows, threads, 0, s, r);
            } else {
                hipLaunchKernelGGL((codec_rows_kernel<false, false>), rows, threads, 0, s, r);
            }
            CODEC_CHECK(hipGetLastError());
        }
        gemm<kEpiShift>({hn.p, T, dec_w.p, dec_b.p, nullptr, ypad.p, T, kCW, kCH, nullptr, 0}, pd);
        const CodecGemm u{ypad.p, T + 2, up_w.p, up_b.p, out.p, nullptr, T, kUpN, kUpTaps * kCW, ws.p, 0};
        if (pu.splits == 1) {
            gemm<kEpiUp, true>(u, pu);
            return;
        }
        gemm<kEpiPartial, true>(u, pu);
        const dim3 ug(static_cast<unsigned>((static_cast<size_t>(T) * kUpN / 4 + 255) / 256));
        if (pu.splits <= 2) hipLaunchKernelGGL(codec_up_reduce_kernel<2>, ug, dim3(256), 0, s, u, pu.splits);
        else if (pu.splits <= 4) hipLaunchKernelGGL(codec_up_reduce_kernel<4>, ug, dim3(256), 0, s, u, pu.splits);
        else hipLaunchKernelGGL(codec_up_reduce_kernel<8>, ug, dim3(256), 0, s, u, pu.splits);
        CODEC_CHECK(hipGetLastError());
    }

    void drop_graphs() {
        for (auto& kv : graphs) (void)hipGraphExecDestroy(kv.second);
        graphs.clear();
    }
    // One decode of T codes: a replay of its captured graph, or eager launches.
    void run(int T) {
        if (!use_graphs) {
            enqueue(T);
            return;
        }
        if (graph_generation != generation || graphs.size() >= 64) {
            drop_graphs();
            graph_generation = generation;
        }
        auto it = graphs.find(T);
        if (it == graphs.end()) {
            hipGraph_t g = nullptr;
            CODEC_CHECK(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
            try {
                enqueue(T);
            } catch (...) {
                (void)hipStreamEndCapture(stream, &g);
                if (g) (void)hipGraphDestroy(g);
                throw;
            }
            CODEC_CHECK(hipStreamEndCapture(stream, &g));
            hipGraphExec_t exec = nullptr;
            const hipError_t e = hipGraphInstantiate(&exec, g, nullptr, nullptr, 0);
            (void)hipGraphDestroy(g);
            CODEC_CHECK(e);
            it = graphs.emplace(T, exec).first;
        }
        CODEC_CHECK(hipGraphLaunch(it->second, stream));
    }

    void decode(const uint32_t* codes, uint32_t n, float* host_out) {
        check_codes(codes, n);
        reserve(static_cast<int>(n));
        CODEC_CHECK(hipMemcpyAsync(dcodes.p, codes, n * 4, hipMemcpyHostToDevice, stream));
        run(static_cast<int>(n));
        CODEC_CHECK(hipMemcpyAsync(host_out, out.p, static_cast<size_t>(2) * n * kCW * 4, hipMemcpyDeviceToHost, stream));
        CODEC_CHECK(hipStreamSynchronize(stream));
    }

    // Mean duration of the device work of decode(n codes) over iters back-to-back runs, and its
    // FLOPs (the GEMMs as they are run, the up conv with two taps; lookup, norms, depthwise convs
    // and copies are < 0.5% of them).
    void bench(uint32_t n, uint32_t iters, float* avg_ms, double* flops) {
        if (!iters || n < 1 || n > static_cast<uint32_t>(kMaxCodes)) throw std::invalid_argument("Invalid codec benchmark request");
        std::vector<uint32_t> codes(n);
        for (uint32_t i = 0; i < n; ++i) codes[i] = (i * 2654435761u) % kCodebook;
        reserve(static_cast<int>(n));
        CODEC_CHECK(hipMemcpyAsync(dcodes.p, codes.data(), n * 4, hipMemcpyHostToDevice, stream));
        run(static_cast<int>(n));  // warm-up (and the graph's capture)
        CODEC_CHECK(hipEventRecord(ev[0], stream));
        for (uint32_t i = 0; i < iters; ++i) run(static_cast<int>(n));
        CODEC_CHECK(hipEventRecord(ev[1], stream));
        CODEC_CHECK(hipEventSynchronize(ev[1]));
        float ms = 0;
        CODEC_CHECK(hipEventElapsedTime(&ms, ev[0], ev[1]));
        *avg_ms = ms / iters;
        const double T = n;
        *flops = 2.0 * T * kCH * kCK * kCW + kCBlocks * 2.0 * (2.0 * T * kCH * kCF) + 2.0 * T * kCW * kCH + 2.0 * T * kUpN * kUpTaps * kCW;
    }
};

}  // namespace itts

struct itts_codec {
    itts::CodecEngine e;
};

namespace {
thread_local std::string g_codec_create_error;

template <class F>
int codec_guarded(itts_codec* c, F&& f) {
    try {
        f();
        return ITTS_OK;
    } catch (const std::invalid_argument& e) {
        (c ? c->e.last_error : g_codec_create_error) = e.what();
        return ITTS_EINVAL;
    } catch (const std::runtime_error& e) {
        (c ? c->e.last_error : g_codec_create_error) = e.what();
        return ITTS_ERUNTIME;
    } catch (const std::exception& e) {
        (c ? c->e.last_error : g_codec_create_error) = e.what();
        return ITTS_ELOGIC;
    }
}

int codec_create(const std::unordered_map<std::string, itts::CodecTensor>& t, itts_codec** out) {
    if (!out) return ITTS_EINVAL;
    *out = nullptr;
    auto c = std::make_unique<itts_codec>();
    const int st = codec_guarded(nullptr, [&] { c->e.create(t); });
    if (st == ITTS_OK) *out = c.release();
    return st;
}
}  // namespace

extern "C" {

int itts_codec_create(const itts_tensor* tensors, int32_t count, itts_codec** out) {
    std::unordered_map<std::string, itts::CodecTensor> t;
    for (int32_t i = 0; tensors && i < count; ++i) {
        const itts_tensor& x = tensors[i];
        if (!x.name || !x.data || x.ndim < 0 || x.ndim > 4) {
            g_codec_create_error = "Invalid tensor table";
            return ITTS_EINVAL;
        }
        t[x.name] = {x.data, std::vector<int64_t>(x.shape, x.shape + x.ndim)};
    }
    return codec_create(t, out);
}

int itts_codec_create_from_bundle(const itts_bundle* b, itts_codec** out) {
    if (!b) {
        g_codec_create_error = "Invalid bundle";
        return ITTS_EINVAL;
    }
    std::unordered_map<std::string, itts::CodecTensor> t;
    const int32_t n = itts_bundle_count(b);
    for (int32_t i = 0; i < n; ++i) {
        itts_bundle_tensor bt{};
        if (itts_bundle_tensor_at(b, i, &bt) != ITTS_OK) continue;
        const std::string name = bt.name;
        if (name.rfind("codec.", 0) != 0 || bt.dtype != ITTS_DTYPE_F32) continue;
        t[name] = {static_cast<const float*>(bt.data), std::vector<int64_t>(bt.shape, bt.shape + bt.ndim)};
    }
    return codec_create(t, out);
}

void itts_codec_destroy(itts_codec* c) { delete c; }

const char* itts_codec_last_error(const itts_codec* c) { return c ? c->e.last_error.c_str() : g_codec_create_error.c_str(); }

int itts_codec_decode(itts_codec* c, const uint32_t* codes, uint32_t n, float* out) {
    if (!c) return ITTS_EINVAL;
    return codec_guarded(c, [&] {
        if (!out) throw std::invalid_argument("Codec expects 1..5000 code IDs in [0,8192)");
        c->e.decode(codes, n, out);
    });
}

int itts_codec_bench(itts_codec* c, uint32_t n, uint32_t iters, float* avg_ms, double* flops) {
    if (!c || !avg_ms || !flops) return ITTS_EINVAL;
    return codec_guarded(c, [&] { c->e.bench(n, iters, avg_ms, flops); });
}

}  // extern "C"
