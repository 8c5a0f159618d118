// The matrix-core main loop shared by the prefill GEMMs: C = A W^T with FP32 (or BF16)
// weights and FP32 results, on the BF16 matrix instructions.
//
// Every FP32 operand x is held as three BF16 numbers, x = hi + mid + lo, each the nearest BF16
// to what the ones before it leave (8 + 8 + 8 significant bits: nothing is left over), and a
// product is the sum of the six partial products whose size can reach an FP32 rounding:
//   hi hi + (hi mid + mid hi) + (mid mid + hi lo + lo hi),
// each exact in the matrix cores and added in FP32.  Of the three dropped products, mid lo and
// lo mid are at most 2^-25 of |hi hi| each and 2^-24 together, half a unit in the last place of
// one product, and lo lo is 2^-34 of it.  A BF16 weight is its own hi:
// three products.  The hi hi products have an accumulator of their own and the others, 2^-8
// of it and less, a second one added at the end, so the running sum is rounded by one
// instruction in six (all six into one accumulator: twice the error, and above the FP32
// instruction's).  Against that instruction (v_mfma_f32_16x16x4f32: 2048 FLOP in 32 cycles) six
// v_mfma_f32_16x16x32_bf16 (16384 FLOP in 16 cycles each) take 96 cycles where it takes 256.
//
// Infinities, NaN and weights past the largest BF16 do not survive the split: they make every sum
// of the small products that they are in NaN or infinite.  Such a tile's results are formed again
// with FP32 products where they are not finite (gemm_refine): an activation's value is in its
// three numbers all the same, a weight's is in memory.
#pragma once
#include <algorithm>

#include "common.h"

namespace itts {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------------ split operands
// Layout of a split [rows][K] operand in memory: tiles of 16 rows x 32 k, and per tile the hi,
// mid and lo planes of 64 pieces of eight consecutive k, piece 16 (k / 8 % 4) + row % 16.  A
// plane of a tile is what the 64 lanes of one matrix instruction hold (lane l: row l & 15,
// k 8 (l >> 4) .. + 7), 1 KB in lane order, so a wave reads its operand with one 16-byte load
// per lane and no LDS.  Rows are padded to a multiple of 16.  The padding is zeroed when the
// buffer is made and then holds what longer operands left: a result row depends on its own
// operand row only, but NaN in the padding sends its tile through the slower epilogue.
constexpr int kPlaneElems = 512;              // one plane of a tile
constexpr int kTileElems = 3 * kPlaneElems;   // hi, mid, lo
__host__ __device__ inline size_t split_elems(size_t rows, size_t k) { return (rows + 15) / 16 * 16 * k * 3; }
__device__ __forceinline__ size_t split_off(int row, int col, int k) {
    return (static_cast<size_t>(row >> 4) * (k >> 5) + (col >> 5)) * kTileElems + ((col >> 3) & 3) * 128 + (row & 15) * 8 + (col & 7);
}

// Two floats to BF16, nearest even, the first in the low half (v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint32_t bf16_pair(float a, float b) {
    const bf16x2 v = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
    return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ float bf16_lo(uint32_t v) { return __uint_as_float(v << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t v) { return __uint_as_float(v & 0xffff0000u); }

// hi, mid and lo of a pair; x - hi and (x - hi) - mid are exact.  STORED: hi is at most the largest
// BF16, so a finite x is hi + (mid + lo) whatever its size, and mid is infinite if x is (split_value).
constexpr float kBf16Max = 3.3895314e38f;
template <bool STORED = false>
__device__ __forceinline__ void split_pair(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
    h = STORED ? bf16_pair(__builtin_amdgcn_fmed3f(a, -kBf16Max, kBf16Max), __builtin_amdgcn_fmed3f(b, -kBf16Max, kBf16Max)) : bf16_pair(a, b);
    a -= bf16_lo(h);
    b -= bf16_hi(h);
    m = bf16_pair(a, b);
    l = bf16_pair(a - bf16_lo(m), b - bf16_hi(m));
}
template <bool STORED = false>
__device__ __forceinline__ void split_piece(const float (&x)[8], u32x4& h, u32x4& m, u32x4& l) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t a, b, c;
        split_pair<STORED>(x[2 * i], x[2 * i + 1], a, b, c);
        h[i] = a;
        m[i] = b;
        l[i] = c;
    }
}
// Stores one element / four / one eight-element piece of a split operand.
__device__ __forceinline__ void split_store(uint16_t* p, size_t off, float x) {
    uint32_t h, m, l;
    split_pair<true>(x, 0.0f, h, m, l);
    p[off] = static_cast<uint16_t>(h);
    p[off + kPlaneElems] = static_cast<uint16_t>(m);
    p[off + 2 * kPlaneElems] = static_cast<uint16_t>(l);
}
// Four consecutive elements, from a column that is a multiple of four.
__device__ __forceinline__ void split_store4(uint16_t* p, size_t off, const float (&x)[4]) {
    u32x2 h, m, l;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        uint32_t a, b, c;
        split_pair<true>(x[2 * i], x[2 * i + 1], a, b, c);
        h[i] = a;
        m[i] = b;
        l[i] = c;
    }
    *reinterpret_cast<u32x2*>(p + off) = h;
    *reinterpret_cast<u32x2*>(p + off + kPlaneElems) = m;
    *reinterpret_cast<u32x2*>(p + off + 2 * kPlaneElems) = l;
}
__device__ __forceinline__ void split_store_piece(uint16_t* p, size_t off, const float (&x)[8]) {
    u32x4 h, m, l;
    split_piece<true>(x, h, m, l);
    *reinterpret_cast<u32x4*>(p + off) = h;
    *reinterpret_cast<u32x4*>(p + off + kPlaneElems) = m;
    *reinterpret_cast<u32x4*>(p + off + 2 * kPlaneElems) = l;
}

// The value stored at p (its hi).
__device__ __forceinline__ float split_value(const uint16_t* p) {
    const float h = bf16_to_f32(p[0]), m = bf16_to_f32(p[kPlaneElems]), l = bf16_to_f32(p[2 * kPlaneElems]);
    return fabsf(m) == INFINITY ? m : h + (m + l);
}

// One sum in FP32, in k order: a(k) is the operand's value, w the weight row at its first k.
// NaN stays NaN, and ends it.
__device__ __forceinline__ bool not_finite(float v) { return !(fabsf(v) <= 3.402823466e38f); }
__device__ __forceinline__ float gemm_weight(float w) { return w; }
__device__ __forceinline__ float gemm_weight(uint16_t w) { return bf16_to_f32(w); }
template <typename WT, class A>
__device__ __forceinline__ float gemm_dot(const WT* w, int len, A a) {
    float s = 0.0f;
#pragma clang loop unroll(disable)
    for (int k = 0; k < len && s == s; ++k) s = __builtin_fmaf(a(k), gemm_weight(w[k]), s);
    return s;
}

// ------------------------------------------------------------------ tile shapes
// A workgroup of eight waves computes RT x 16 rows by BN columns: four waves load and split
// weights, four multiply.  The multiplying waves stand WR x WC (WR WC = 4) over TR row tiles
// and TC column strips of 16 each.  One loading and one multiplying wave share a SIMD, so the
// splitting (vector ALU) runs beside the matrix instructions, and the weight loads have a
// vmcnt of their own: the operand loads of a multiplying wave never wait behind HBM.
constexpr int kGemmThreads = 512;
constexpr int kGemmUnroll = 4;  // k steps per turn of the multiplying waves' loop
constexpr int kGemmK = 32 * kGemmUnroll;  // K ranges are multiples of this
constexpr int kGemmRing = 3;  // k steps of split weights in LDS: read, read ahead, being written
template <typename WT, int WR_, int TR_, int TC_>
struct GemmTile {
    using W = WT;
    static constexpr int WR = WR_, WC = 4 / WR_, TR = TR_, TC = TC_;
    static constexpr int RT = WR * TR, BM = RT * 16, NS = WC * TC, BN = NS * 16;
    static constexpr int PB = sizeof(WT) == 4 ? 3 : 1;       // planes of a weight
    static constexpr int PD = 2 * kGemmUnroll;               // k steps of weights requested ahead
    static constexpr int NLOW = TR == 1 ? 2 : 1;             // accumulators of the small products per tile
    static constexpr int NA = TR <= 2 ? 4 : 3;               // operand register sets (NA - 1 k steps ahead)
    static constexpr int kStepElems = NS * PB * kPlaneElems;
    // the epilogues that write split rows pass each wave's 16 x 16 TC values through LDS
    static constexpr int kEpiFloats = 16 * (16 * TC + 4);
    static constexpr int kLdsBytes =
        kGemmRing * kStepElems * 2 > 4 * kEpiFloats * 4 ? kGemmRing * kStepElems * 2 : 4 * kEpiFloats * 4;
    static_assert(BN == 64, "the loading threads cover 64 columns");
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t gemm_rsrc(const void* p, uint32_t bytes) {
    const uint64_t u = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<uint32_t>(u))));
    const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<uint32_t>(u >> 32))));
    // descriptor word 3: raw 32-bit buffer; reads past `bytes` return zero and touch no memory
    return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>((static_cast<uint64_t>(hi) << 32) | lo), 0,
                                             __builtin_amdgcn_readfirstlane(static_cast<int>(bytes)), 0x00020000);
}
__device__ __forceinline__ u32x4 gemm_load16(__amdgpu_buffer_rsrc_t rs, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, static_cast<int>(voff), static_cast<int>(soff), 0));
}

// ------------------------------------------------------------------ loading waves
// Thread t of 256 owns, of each 32-wide k step, the piece (column t / 4, eight k at
// 8 (t % 4)): four threads read 128 consecutive bytes of a weight row.  In LDS a piece goes to
// slot 16 g + (c ^ 2 g) of its strip (g = k / 8 % 4, c = column % 16): eight neighbouring
// threads (two columns, four g) write, and eight neighbouring lanes (one g, eight c) read,
// eight different 16-byte banks.  k step s + 2 is written while the multiplying waves use step s,
// one barrier per step; PD steps are in flight from memory.  `w`: the tile's first row, at its
// first k.
template <class T>
__device__ __forceinline__ void gemm_loader(uint16_t* ring, const typename T::W* w, int K, int nst, int t) {
    using WT = typename T::W;
    constexpr int NL = sizeof(WT) == 4 ? 2 : 1;  // 16-byte loads per thread and step
    constexpr int PD = T::PD;
    const __amdgpu_buffer_rsrc_t rs = gemm_rsrc(w, static_cast<uint32_t>((static_cast<size_t>(T::BN - 1) * K + nst * 32) * sizeof(WT)));
    constexpr int kAhead = T::PB == 3 ? 3 : 2;  // steps split (FP32) or written ahead of the first barrier
    const int g = t & 3, c = t >> 2;
    const uint32_t voff = static_cast<uint32_t>((static_cast<size_t>(c) * K + 8 * g) * sizeof(WT));
    uint16_t* dst = ring + (c >> 4) * T::PB * kPlaneElems + (16 * g + ((c & 15) ^ (2 * g))) * 8;
    u32x4 raw[PD][NL];
    auto load = [&](int slot, int s) {  // steps past the last: out of the buffer's range, no memory access
        const uint32_t o = s < nst ? voff + static_cast<uint32_t>(s) * 32 * sizeof(WT) : 0x40000000u;
#pragma unroll
        for (int q = 0; q < NL; ++q) raw[slot][q] = gemm_load16(rs, o + 16 * q, 0);
    };
    u32x4 plane[3];
    auto split = [&](int slot) {
        float x[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = __uint_as_float(raw[slot][i / 4 % NL][i & 3]);
        split_piece(x, plane[0], plane[1], plane[2]);
    };
    int buf = 0;
    auto put = [&](const u32x4* v) {
#pragma unroll
        for (int q = 0; q < T::PB; ++q) *reinterpret_cast<u32x4*>(dst + buf * T::kStepElems + q * kPlaneElems) = v[q];
        buf = buf + 1 == kGemmRing ? 0 : buf + 1;
    };
#pragma unroll
    for (int s = 0; s < PD; ++s) load(s, s);
#pragma unroll
    for (int s = 0; s < kAhead; ++s) {
        if constexpr (T::PB == 3) split(s);
        if (s < 2) put(T::PB == 3 ? plane : raw[s]);
        load(s, PD + s);
    }
    __syncthreads();
    // A step's FP32 pieces were split the step before, so its LDS writes are on their way while the
    // next pieces are split (about 350 cycles): one after the other, they held up the barrier (155
    // rows: 3840 x 1280 17.9 -> 16.5 us, 5120 x 1280 20.3 -> 19.7).  Eight loading waves of half a
    // piece each, or two k steps per barrier, measured the same as this.
    // sched_barrier: the split stays behind the barrier and its loads are issued at once; moved
    // across, they made a step wait for loads of the steps after it.
    auto step = [&](int s, int u) {
        const int n = (u + kAhead) % PD;
        __builtin_amdgcn_sched_barrier(0);
        put(T::PB == 3 ? plane : raw[n]);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (T::PB == 3) split(n);
        load(n, s + u + kAhead + PD);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
    };
    int s = 0;
    for (; s + PD <= nst; s += PD) {
#pragma unroll
        for (int u = 0; u < PD; ++u) step(s, u);
    }
    if (s < nst) {  // nst is a multiple of kGemmUnroll, PD of kGemmUnroll or twice it
#pragma unroll
        for (int u = 0; u < kGemmUnroll; ++u) step(s, u);
    }
}

// ------------------------------------------------------------------ multiplying waves
// A wave's sums of the hi hi products and of the small ones: (row tile i) x (strip c).
template <class T>
struct GemmAcc {
    f32x4 hi[T::TR][T::TC], low[T::NLOW][T::TR][T::TC];
    __device__ __forceinline__ f32x4 small(int i, int c) const { return T::NLOW == 2 ? low[0][i][c] + low[1][i][c] : low[0][i][c]; }
    __device__ __forceinline__ void sum(f32x4 (&acc)[T::TR][T::TC]) const {
#pragma unroll
        for (int i = 0; i < T::TR; ++i)
#pragma unroll
            for (int c = 0; c < T::TC; ++c) acc[i][c] = hi[i][c] + small(i, c);
    }
    // Whether gemm_refine is needed.  An operand that is not finite shows in the small products of
    // its whole row, a weight (or one past the largest BF16) in those of its whole column.
    __device__ __forceinline__ bool suspect() const {
        float t = 0.0f;
#pragma unroll
        for (int i = 0; i < T::TR; ++i) {
            const f32x4 v = small(i, 0);
            t += (v[0] + v[1]) + (v[2] + v[3]);
        }
#pragma unroll
        for (int c = 1; c < T::TC; ++c) t += T::NLOW == 2 ? low[0][0][c][0] + low[1][0][c][0] : low[0][0][c][0];
        return __ballot(not_finite(t)) != 0;
    }
};
// acc over nst k steps.  ars: the split operand; aoff(i, s): this
// lane's byte offset of row tile i at k step s (of nst), and the part of it that is uniform.  The
// next strip's weights are read from LDS while the current one's matrix instructions run (the
// first strip of step s + 1 too: the loading waves finished it before the barrier ahead of step s).
struct GemmOff {
    uint32_t lane, uniform;
};
template <class T, class AOff>
__device__ __forceinline__ void gemm_compute(const uint16_t* ring, __amdgpu_buffer_rsrc_t ars, AOff aoff, int nst, int wc, int lane,
                                             GemmAcc<T>& acc) {
    bf16x8 av[T::NA][T::TR][3], bv[2][T::PB];
#pragma unroll
    for (int q = 0; q < T::NLOW; ++q)
#pragma unroll
        for (int i = 0; i < T::TR; ++i)
#pragma unroll
            for (int c = 0; c < T::TC; ++c) acc.low[q][i][c] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto load_a = [&](int set, int s, int i, int p) {  // plane p of row tile i; steps past the last reread it
        const GemmOff o = aoff(i, min(s, nst - 1));
        av[set][i][p] = __builtin_bit_cast(bf16x8, gemm_load16(ars, o.lane + p * kPlaneElems * 2, o.uniform));
    };
#pragma unroll
    for (int i = 0; i < T::TR; ++i)
#pragma unroll
        for (int c = 0; c < T::TC; ++c) acc.hi[i][c] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int g = lane >> 4;
    const uint16_t* src = ring + wc * T::TC * T::PB * kPlaneElems + (16 * g + ((lane & 15) ^ (2 * g))) * 8;
    int buf = 0;
    auto load_b = [&](int set, int b, int c, int p) {
        bv[set][p] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(src + b * T::kStepElems + (c * T::PB + p) * kPlaneElems));
    };
#pragma unroll
    for (int s = 0; s < T::NA - 1; ++s)
#pragma unroll
        for (int q = 0; q < 3 * T::TR; ++q) load_a(s, s, q / 3, q % 3);
    __syncthreads();
#pragma unroll
    for (int p = 0; p < T::PB; ++p) load_b(0, 0, 0, p);
    // The products of a strip, one group of TR matrix instructions each, in order of the operand
    // planes.  A group takes at most one operand load and one weight read with it: a 1 KB load
    // occupies the CU's address path for 16 cycles and four waves share it, so nine loads
    // issued at once held a wave's matrix instructions back by up to 576 cycles per step.
    constexpr int NP = T::PB == 3 ? 6 : 3, NG = T::TC * NP, NQ = 3 * T::TR;
    constexpr int pa[6] = {0, 2, T::PB == 3 ? 0 : 1, 1, 1, 0}, pb[6] = {0, 0, T::PB == 3 ? 2 : 0, 1, 0, 1};
    static_assert(NQ <= NG, "one operand load per group");
    auto step = [&](int s, int u) {
        const int nbuf = buf + 1 == kGemmRing ? 0 : buf + 1;
#pragma unroll
        for (int c = 0; c < T::TC; ++c) {
            const int cur = (u * T::TC + c) & 1;
#pragma unroll
            for (int g = 0; g < NP; ++g) {
                const int gi = c * NP + g, q = gi * NQ / NG;
                if (gi == 0 || q != (gi - 1) * NQ / NG) load_a((u + T::NA - 1) % T::NA, s + u + T::NA - 1, q / 3, q % 3);
                if (g < T::PB) {
                    if (c + 1 < T::TC) load_b(cur ^ 1, buf, c + 1, g);
                    else load_b(cur ^ 1, nbuf, 0, g);
                }
                __builtin_amdgcn_sched_barrier(0);
                auto& d = g == 0 ? acc.hi : acc.low[(g + 1) % T::NLOW];
#pragma unroll
                for (int i = 0; i < T::TR; ++i)
                    d[i][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[u % T::NA][i][pa[g]], bv[cur][pb[g]], d[i][c], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        buf = nbuf;
        __syncthreads();
    };
    // Register sets come round after U steps; nst is a multiple of kGemmUnroll.
    constexpr int U = T::NA == 3 ? 3 * kGemmUnroll : kGemmUnroll;
    int s = 0;
    for (; s + U <= nst; s += U) {
#pragma unroll
        for (int u = 0; u < U; ++u) step(s, u);
    }
    if constexpr (U > kGemmUnroll) {
        if (s < nst) {
#pragma unroll
            for (int u = 0; u < kGemmUnroll; ++u) step(s, u);
            if (s + kGemmUnroll < nst) {
#pragma unroll
                for (int u = kGemmUnroll; u < 2 * kGemmUnroll; ++u) step(s, u);
            }
        }
    }
}

// ------------------------------------------------------------------ placement and results
// A value held in a register at this point of the program: an empty asm takes it.  The
// epilogues form every output (and read every loaded operand) before the first row's store
// this way; left to the compiler, each row's arithmetic sank into that row's branch, where the
// use of a load still in flight made it wait for every memory access outstanding, the
// earlier rows' stores included (one store completion per row).
template <typename T>
__device__ __forceinline__ void pin_value(T v) {
    asm volatile("" ::"v"(v));
}

// Workgroup L runs on XCD L % 8 (round-robin dispatch).  The logical index j gives each XCD one
// contiguous range, row blocks (y) fastest, then splits (z), then column tiles (x), so the
// workgroups sharing a column tile's weights mostly share one L2.
struct GemmPlace {
    int x, y, z;
};
__device__ __forceinline__ GemmPlace gemm_place() {
    const int nwg = gridDim.x * gridDim.y * gridDim.z;
    const int L = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    const int per = nwg / 8, rem = nwg % 8, xcd = L % 8;
    const int j = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + L / 8;
    return {j / static_cast<int>(gridDim.y * gridDim.z), j % static_cast<int>(gridDim.y), (j / static_cast<int>(gridDim.y)) % static_cast<int>(gridDim.z)};
}

// A wave's results lie at rows 16 (tile0 + i) + rq + r (rq = 4 (lane / 16)), columns col0 + 16 c:
// acc[i][c][r].  Raw partial sums to ws[M][N].  Every destination's 32-bit element offset is
// formed before the first store (M x N < 2^31): with one register pair reused for each row's
// address, the compiler let only about two stores be in flight at a time.
template <class T>
__device__ __forceinline__ void gemm_store_partial(float* ws, int M, int N, int tile0, int col0, int lane, const f32x4 (&acc)[T::TR][T::TC]) {
    const int rq = 4 * (lane >> 4);
    uint32_t off[T::TR][4];
#pragma unroll
    for (int i = 0; i < T::TR; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            off[i][r] = static_cast<uint32_t>(((tile0 + i) * 16 + rq + r) * N + col0);
            pin_value(off[i][r]);
        }
#pragma unroll
    for (int i = 0; i < T::TR; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if ((tile0 + i) * 16 + rq + r < M) {
#pragma unroll
                for (int c = 0; c < T::TC; ++c) ws[off[i][r] + 16 * c] = acc[i][c][r];
            }
}

// The epilogue of a suspect tile: each sum that is not finite is formed again, dot(m, n) for row m
// and column n of the wave's tile, and store(m, n, v) takes them all (rows past M too).  The tile
// passes through the wave's part of LDS (the ring is no longer read), so that the loop is over
// memory and not over registers, and the ordinary epilogue stays as it is (155 rows, 3840 x 1280:
// 22.0 us without this and with it; sums corrected in their registers took 22.7, by the copies
// and by the stores that had to wait for the test).  For epilogues that only add: another copy of
// a function's code may round a finite value differently (gemm_store_split).
template <class T, class Dot, class Store>
__device__ __forceinline__ void gemm_refine(uint8_t* lds, int M, int tile0, int wave, int lane, const GemmAcc<T>& acc, Dot dot, Store store) {
    constexpr int W = 16 * T::TC, S = W + 4;
    float* buf = reinterpret_cast<float*>(lds) + wave * T::kEpiFloats;
#pragma unroll
    for (int i = 0; i < T::TR; ++i) {
#pragma unroll
        for (int c = 0; c < T::TC; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float l = T::NLOW == 2 ? acc.low[0][i][c][r] + acc.low[1][i][c][r] : acc.low[0][i][c][r];
                asm volatile("" : "+v"(l));  // an addition of this branch, not shared with the ordinary epilogue's
                buf[(4 * (lane >> 4) + r) * S + 16 * c + (lane & 15)] = acc.hi[i][c][r] + l;
            }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma clang loop unroll(disable)
        for (int q = lane; q < 16 * W; q += 64) {
            const int n = q % W, m = (tile0 + i) * 16 + q / W;
            float v = buf[q / W * S + n];
            if (m < M && not_finite(v)) v = dot(m, n);
            store(m, n, v);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

// Results as split rows of the next GEMM's operand ([.][on], from row row_off on): each wave
// passes its row tiles through its own part of LDS (the ring is no longer read), so that a lane
// holds eight consecutive columns.  f(i, c, r) is the value of acc[i][c][r]; with PAIRS, of a
// column pair, given in its even lane, and `oc0` counts pairs.  `suspect`: values that are not
// finite are replaced by again(m, n), row m and column (pair) n of the wave's tile, the value from
// sums formed again.
template <class T, bool PAIRS, class F, class G>
__device__ __forceinline__ void gemm_store_split(uint8_t* lds, int wave, int lane, uint16_t* out, int M, int on, int row_off, int tile0, int oc0, F f,
                                                 bool suspect, G again) {
    constexpr int W = PAIRS ? 8 * T::TC : 16 * T::TC, S = W + 4;  // columns written; row stride
    float* buf = reinterpret_cast<float*>(lds) + wave * T::kEpiFloats;
    const int rq = 4 * (lane >> 4);
#pragma unroll
    for (int i = 0; i < T::TR; ++i) {
#pragma unroll
        for (int c = 0; c < T::TC; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float v = f(i, c, r);
                if constexpr (PAIRS) {
                    if (!(lane & 1)) buf[(rq + r) * S + 8 * c + (lane & 15) / 2] = v;
                } else {
                    buf[(rq + r) * S + 16 * c + (lane & 15)] = v;
                }
            }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (__builtin_expect(suspect, 0)) {
#pragma clang loop unroll(disable)
            for (int q = lane; q < 16 * W; q += 64) {
                const int n = q % W, m = (tile0 + i) * 16 + q / W;
                if (m < M && not_finite(buf[q / W * S + n])) buf[q / W * S + n] = again(m, n);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        for (int q = lane; q < 2 * W; q += 64) {
            const int r = q & 15, e0 = 8 * (q >> 4), row = (tile0 + i) * 16 + r;
            float x[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = buf[r * S + e0 + e];
            if (row < M) split_store_piece(out, split_off(row + row_off, oc0 + e0, on), x);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

// ------------------------------------------------------------------ few rows
// Up to four row tiles: a workgroup of eight waves takes 16 columns and its K range whole,
// wave w the k steps w, w + 8, ... of it, each with its weights straight from memory to the
// matrix operand (no LDS, no barrier until the end), two to five steps requested at once.  With so few
// rows the weights are read once either way and the time is the memory's: 64-column tiles
// need K splits (and a kernel to add them) to reach every CU, and their steps wait on one
// another.  More rows: the operand, read by every workgroup, becomes the larger stream.
constexpr int kSmallWaves = 8;
constexpr int kSmallK = 32 * kSmallWaves;  // K ranges are multiples of this
template <int RT>
struct GemmSmallLds {
    float sum[kSmallWaves][RT][16][17];
};
// Thread t ends with the sum (over the waves, in order) of row t / 16, column t % 16 for
// t < 256 RT / (RT > 2 ? 2 : 1); with RT > 2, also of row t / 16 + 32 in `out[1]`.  w: the
// workgroup's first weight row at its first k; a_row_bytes: bytes of a row tile of the operand.
// Sums of rows below M that are not finite are formed again: value(m, k) as gemm_refine's a.
template <typename WT, int RT, class A>
__device__ __forceinline__ void gemm_small(GemmSmallLds<RT>& lds, const WT* w, int K, int nst, __amdgpu_buffer_rsrc_t ars, uint32_t a0,
                                           uint32_t a_row_bytes, int M, A value, float (&out)[2]) {
    constexpr int NL = sizeof(WT) == 4 ? 2 : 1;
    constexpr int kBatch = RT == 1 ? 5 : 2;  // two workgroups per CU up to two row tiles
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, c = lane & 15;
    const __amdgpu_buffer_rsrc_t rs = gemm_rsrc(w, static_cast<uint32_t>((static_cast<size_t>(15) * K + nst * 32) * sizeof(WT)));
    const uint32_t boff = static_cast<uint32_t>((static_cast<size_t>(c) * K + 8 * g) * sizeof(WT));
    uint32_t aoff[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) aoff[i] = a0 + static_cast<uint32_t>(min(i, (M - 1) >> 4)) * a_row_bytes + lane * 16;
    f32x4 acc[RT], low[2][RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) acc[i] = low[0][i] = low[1][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s0 = wave; s0 < nst; s0 += kSmallWaves * kBatch) {
        u32x4 b[kBatch][NL];
        bf16x8 a[kBatch][RT][3];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {  // steps past the last: out of range, zeros, no memory access
            const int s = s0 + kSmallWaves * u;
            const uint32_t o = s < nst ? boff + static_cast<uint32_t>(s) * 32 * sizeof(WT) : 0x40000000u;
#pragma unroll
            for (int q = 0; q < NL; ++q) b[u][q] = gemm_load16(rs, o + 16 * q, 0);
        }
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            const int s = s0 + kSmallWaves * u;
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int p = 0; p < 3; ++p)
                    a[u][i][p] = __builtin_bit_cast(
                        bf16x8, gemm_load16(ars, s < nst ? aoff[i] + static_cast<uint32_t>(s) * (kTileElems * 2) + p * kPlaneElems * 2 : 0x7ffffff0u, 0));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            u32x4 h, m, l;
            if constexpr (NL == 2) {
                float x[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) x[i] = __uint_as_float(b[u][i >> 2][i & 3]);
                split_piece(x, h, m, l);
            } else {
                h = b[u][0];
            }
            const bf16x8 bh = __builtin_bit_cast(bf16x8, h), bm = __builtin_bit_cast(bf16x8, m), bl = __builtin_bit_cast(bf16x8, l);
            auto mul = [&](int p, bf16x8 y, f32x4 (&d)[RT]) {
#pragma unroll
                for (int i = 0; i < RT; ++i) d[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u][i][p], y, d[i], 0, 0, 0);
            };
            mul(0, bh, acc);
            mul(2, bh, low[0]);
            mul(1, bh, low[1]);
            if constexpr (NL == 2) {
                mul(0, bl, low[0]);
                mul(0, bm, low[1]);
                mul(1, bm, low[0]);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) lds.sum[wave][i][4 * g + r][c] = acc[i][r] + (low[0][i][r] + low[1][i][r]);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < (RT > 2 ? 2 : 1); ++q) {
        const int row = (tid >> 4) + 32 * q, i = row >> 4;
        float v = 0.0f;
        if (i < RT) {
#pragma unroll
            for (int z = 0; z < kSmallWaves; ++z) v += lds.sum[z][i][row & 15][tid & 15];
        }
        if (__builtin_expect(not_finite(v) && row < M, 0))
            v = gemm_dot(w + static_cast<size_t>(tid & 15) * K, nst * 32, [&](int k) { return value(row, k); });
        out[q] = v;
    }
}
// Its cut, or splits 0 where the 64-column tiles are faster.  Measured on MI355X in both kernels
// (one GEMM with what follows it, weights from HBM, us, 64-column tiles -> this):
//   at most one workgroup per CU (256) and 1280 k each: 3840 x 1280 at 20 rows 11.0 -> 8.1, at 60 rows
//   13.1 -> 11.4; 1280 x 1280 at 32 / 60 rows 8.1 -> 6.9 / 9.5 -> 8.2; 1024 x 3072 at 48 rows 10.5 -> 9.8;
//   5120 x 1280, 320 workgroups: 8 rows 12.9 -> 11.0, but 20 rows 13.5 -> 15.3 (some CUs have two,
//   and every one reads the whole operand); 1280 x 5120 at 20 rows 12.7 -> 17.8;
//   BF16 weights (the operand outweighs them sooner): 3840 x 1280 at 32 rows 7.9 -> 6.5, at 63 rows
//   8.5 -> 9.4.
struct GemmSmallPlan {
    int splits, kchunk;
};
GemmSmallPlan gemm_small_plan(int M, int N, int K, int max_splits, bool bf16);

// How one GEMM is cut: a tile shape, its row blocks, and K cut into `splits` ranges of kchunk (a
// multiple of kGemmK).  `reduce`: the splits are added by a kernel of their own (else by one that
// runs anyway).
struct GemmPlan {
    int tile, mblocks, splits, kchunk;
};
GemmPlan gemm_plan(int M, int N, int K, int max_splits, bool bf16, bool reduce);
// Row tiles of the tile shapes (each 64 columns).  128-column tiles (8 x 8 and 12 x 8) halve
// the operand reads per product but need more than 256 registers or leave half the CUs idle:
// slower at every size measured.
constexpr int kTileRt[] = {1, 2, 4, 8, 12}, kTiles = 5, kGemmBn = 64;
template <typename WT, class F>
void gemm_tile(int tile, F f) {  // f(GemmTile<...>{}) for the plan's tile shape
    switch (tile) {
        case 0: f(GemmTile<WT, 1, 1, 1>{}); break;
        case 1: f(GemmTile<WT, 2, 1, 2>{}); break;
        case 2: f(GemmTile<WT, 4, 1, 4>{}); break;
        case 3: f(GemmTile<WT, 4, 2, 4>{}); break;
        default: f(GemmTile<WT, 4, 3, 4>{}); break;
    }
}

}  // namespace itts
