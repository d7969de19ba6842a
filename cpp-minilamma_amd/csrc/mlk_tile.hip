// mlk_tile.hip -- many-row linear layers on the fp16 matrix cores:
// y[T, O] = x[T, K] W[O, K]^T (+ bias), W fp32, Q8_0 / Q4_0 / Q4_1 blocks or
// planar Q8_0 / Q4_0, for more than 32 rows (F32 from 5, Q8_0 and Q4_0 blocks
// from 17: TileChosen) and K a multiple of 32, at least 256 (other shapes:
// mlk_linear.hip, mlk_gemm.hip).  Semantics as there
// (LinearQ80 / Q40 / Q41, src/quant.cc:393-463; cublasSgemm,
// src/cuda_matmul.cc:142-186): fp32 products and sums, in an order of this
// kernel's choosing.
//
// Products.  Each row of x (and of fp32 or Q4_1 weights, decoded to the
// reference's fp32 values) is scaled by a power of two and split into two
// fp16 pieces, the value rounded to fp16 and the rest rounded to fp16:
// together the value to within one unit of its fp32 last place.
//   codes (Q8_0, Q4_0)    a code is a small integer, exact in fp16, so a
//       block's sum S = sum code (x0 + x1) is two v_mfma_f32_16x16x32_f16,
//       then acc += d S + d' S' for a pair of blocks, in fp32 (one rounding
//       of acc for two blocks: with one per block the sums were 2.2e-7 off
//       at K = 4096 instead of 1.7e-7, and the kernel 5% faster).
//   values (F32, Q4_1)    x1 w0 + x0 w1 + x0 w0, three MFMAs straight into
//       the accumulators; x1 w1, below 2^-22 of the product, is left out.
// Three bf16 pieces per x (exact products) and the fp32 MFMA, which these
// replace, took 3 and, at an eighth of the rate, 8 times the matrix work.
// Errors against float64 (relative 2-norm, normal x and weights, K = 4096
// unsplit): Q8_0 1.7e-7 (three pieces: 2.1e-7), F32 7.1e-7 and Q4_1 6.8e-7
// (fp32 MFMA: 1.1e-6).  Time at 4096 rows, K = 4096, 14336 outputs: Q8_0 1366
// -> 1170 us, F32 3649 -> 1460, Q4_1 3807 -> 1450; at 64 rows Q8_0 91 -> 41.
//
// Scales.  A row's power of two puts the mean magnitude of its first 64
// inputs in [2, 4): fp16 then holds values up to 16000 times that mean, and
// the second piece's subnormals reach 2^-25.  Every thread keeps the largest
// magnitude of the rows it loads; a row whose largest scaled value leaves
// [2^-3, 65504), infinities among them, is marked at the end of the K loop
// and its outputs are summed again in order in fp32 (SlowOutputs), so no
// finite or infinite input is lost.  NaNs pass through the products.
//
// Work.  A workgroup owns BM token rows x BN outputs (32 x 64, 2 waves, 64 x
// 128, 4 waves, or 128 x 256, 8 waves), a wave a 16 MI x 16 NJ part of them, K in stages of 32
// through LDS; while stages are multiplied the next ones, already in
// registers, are split, decoded and written to the other LDS buffers, and
// the ones after them are requested from memory.  Few tiles: K is split over
// workgroups, partial sums reduced in split order (mlk_gemm.hip).
//
// Bound: a stage of a 128 x 256 tile (T = 4096, Q8_0) takes about 2800
// cycles where its MFMAs take 1024 a SIMD; without the loads from memory 2080,
// without loads, splits, decodes and LDS writes 1850, the scale FMAs 190 of
// it (timing-only copies).  Not the order of instructions, deeper requests (3
// and 4 stages ahead), coalesced weight pieces through LDS, or the two halves
// of the waves half a stage apart: each the same or slower.
#include "mlk_quant.h"

#include <type_traits>

namespace mlk {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_a2 __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kWF32 = -1;
constexpr int kBK = 32;  // inputs per stage: one quantization block

template <int WT>
constexpr bool kCodes = WT == MLK_Q8_0 || WT == MLK_Q4_0 || WT == kWPlanarQ8 || WT == kWPlanarQ4;

template <int WT>
constexpr bool kPlanar = WT == kWPlanarQ8 || WT == kWPlanarQ4;

__device__ inline uint32_t AsU32(h2 v) { return __builtin_bit_cast(uint32_t, v); }

// ------------------------------------------------------------ fp16 pieces
// v * s = p0 + p1 + (at most one unit in the last place of fp32), p0 and p1
// fp16; 8 values, two a dword.
__device__ inline void Split8(const float4 (&v)[2], float s, u32x4* p0, u32x4* p1) {
    const float f[8] = {v[0].x, v[0].y, v[0].z, v[0].w, v[1].x, v[1].y, v[1].z, v[1].w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float a = f[2 * i], b = f[2 * i + 1];
        h2 hi, lo;
        hi.x = static_cast<_Float16>(a * s);
        hi.y = static_cast<_Float16>(b * s);
        lo.x = static_cast<_Float16>(fmaf(a, s, -static_cast<float>(hi.x)));
        lo.y = static_cast<_Float16>(fmaf(b, s, -static_cast<float>(hi.y)));
        (*p0)[i] = AsU32(hi);
        (*p1)[i] = AsU32(lo);
    }
}

__device__ inline float AbsSum8(const float4 (&v)[2]) {
    return ((fabsf(v[0].x) + fabsf(v[0].y)) + (fabsf(v[0].z) + fabsf(v[0].w))) +
           ((fabsf(v[1].x) + fabsf(v[1].y)) + (fabsf(v[1].z) + fabsf(v[1].w)));
}

__device__ inline float AbsMax8(const float4 (&v)[2], float m) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        m = fmaxf(fmaxf(m, fabsf(v[i].x)), fabsf(v[i].y));
        m = fmaxf(fmaxf(m, fabsf(v[i].z)), fabsf(v[i].w));
    }
    return m;
}

// The power of two that brings `mean` into [2, 4) and its inverse (within
// 2^-61 .. 2^61; 1 for zero, subnormal, infinite and NaN means).
struct PieceScale {
    float s = 1.0f, inv = 1.0f;
    __device__ PieceScale() {}
    __device__ explicit PieceScale(float mean) {
        int e = static_cast<int>((__float_as_uint(mean) >> 23) & 255u);
        e = e == 0 || e == 255 ? 128 : (e < 66 ? 66 : (e > 188 ? 188 : e));
        s = __uint_as_float(static_cast<uint32_t>(255 - e) << 23);
        inv = __uint_as_float(static_cast<uint32_t>(e - 1) << 23);
    }
    // inv, or 0 when the row's largest magnitude leaves the pieces' range
    // (all zero stays in it)
    __device__ float Checked(float most) const {
        const float m = most * s;
        return m == 0.0f || (m >= 0.125f && m < 65504.0f) ? inv : 0.0f;
    }
};

// ------------------------------------------------------------ weights
// One thread's part of a stage's weight rows, as loaded: 16 inputs (half h
// of the block) of row tid / 2, or for fp32 inputs 8 (tid % 4) .. of rows
// tid / 4 and tid / 4 + (rows per tile) / 2 (4 lanes read a row's 128
// bytes).  Addresses are a uniform base for the tile and the stage plus a
// 32-bit offset of the thread's row.
template <int WT>
struct RawW {
    uint32_t d;
    u32x4 q;
    __device__ void Load(const uint8_t* base, uint32_t off, int h) {
        const uint8_t* b = base + off;
        if constexpr (WT == MLK_Q4_1) {
            d = *reinterpret_cast<const uint32_t*>(b);
            q = *reinterpret_cast<const u32x4_a4*>(b + 4);
        } else {
            d = *reinterpret_cast<const uint16_t*>(b);
            q = *reinterpret_cast<const u32x4_a2*>(b + 2 + (WT == MLK_Q8_0 ? 16 * h : 0));
        }
    }
};
template <>
struct RawW<kWF32> {
    float4 v[2][2];
};
template <int QT>
struct RawPlanar {
    uint32_t d;
    u32x4 q;
    __device__ void Load(const uint8_t* base, uint32_t off, const uint8_t* sbase, uint32_t soff) {
        d = *reinterpret_cast<const uint16_t*>(sbase + soff);
        if constexpr (QT == MLK_Q8_0) {
            const uint2 a = *reinterpret_cast<const uint2*>(base + off);
            const uint2 b = *reinterpret_cast<const uint2*>(base + off + 256);
            q = u32x4{a.x, a.y, b.x, b.y};
        } else {
            q.x = *reinterpret_cast<const uint32_t*>(base + off);
            q.y = *reinterpret_cast<const uint32_t*>(base + off + 256);
        }
    }
};
template <>
struct RawW<kWPlanarQ8> : RawPlanar<MLK_Q8_0> {};
template <>
struct RawW<kWPlanarQ4> : RawPlanar<MLK_Q4_0> {};

// 4 unsigned bytes u as two dwords of fp16 pairs u + bias (exact: 1024 + u
// is the fp16 with low byte u).
__device__ inline void Bytes4(uint32_t u, _Float16 bias, uint32_t* o) {
    const h2 b = {bias, bias};
    o[0] = AsU32(__builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) + b);
    o[1] = AsU32(__builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) + b);
}

// The thread's 16 codes as fp16 pairs, in input order.
template <int WT>
__device__ inline void Codes16(const RawW<WT>& r, int h, u32x4 (&o)[2]) {
    uint32_t t[8];
    if constexpr (WT == MLK_Q8_0 || WT == kWPlanarQ8) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            Bytes4(r.q[i] ^ 0x80808080u, static_cast<_Float16>(-1152.0f), &t[2 * i]);
        }
    } else if constexpr (WT == MLK_Q4_0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            Bytes4((r.q[i] >> (4 * h)) & 0x0F0F0F0Fu, static_cast<_Float16>(-1032.0f), &t[2 * i]);
        }
    } else {  // planar Q4_0: low nibbles inputs 0..3 of 8, high nibbles 4..7, two's complement
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t u = r.q[i] ^ 0x88888888u;
            Bytes4(u & 0x0F0F0F0Fu, static_cast<_Float16>(-1032.0f), &t[4 * i]);
            Bytes4((u >> 4) & 0x0F0F0F0Fu, static_cast<_Float16>(-1032.0f), &t[4 * i + 2]);
        }
    }
    o[0] = u32x4{t[0], t[1], t[2], t[3]};
    o[1] = u32x4{t[4], t[5], t[6], t[7]};
}

// The thread's 16 Q4_1 weights, the reference's fp32 values.
__device__ inline void Values16(const RawW<MLK_Q4_1>& r, int h, float4 (&v)[2][2]) {
    const float sc = HalfHw(r.d & 0xFFFFu), mn = HalfHw(r.d >> 16);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t u = (r.q[i] >> (4 * h)) & 0x0F0F0F0Fu;
        float4& e = v[i / 2][i % 2];
        e.x = __fadd_rn(__fmul_rn(sc, static_cast<float>(u & 0xFFu)), mn);
        e.y = __fadd_rn(__fmul_rn(sc, static_cast<float>((u >> 8) & 0xFFu)), mn);
        e.z = __fadd_rn(__fmul_rn(sc, static_cast<float>((u >> 16) & 0xFFu)), mn);
        e.w = __fadd_rn(__fmul_rn(sc, static_cast<float>(u >> 24)), mn);
    }
}

// One weight of row o (SlowOutputs).
template <int WT>
__device__ inline float Weight(const uint8_t* w, int64_t O, int64_t K, int64_t row_bytes,
                               int64_t o, int64_t k) {
    const int64_t kb = k / 32;
    const int e = static_cast<int>(k % 32);
    if constexpr (WT == kWF32) {
        return reinterpret_cast<const float*>(w + o * row_bytes)[k];
    } else if constexpr (WT == kWPlanarQ8 || WT == kWPlanarQ4) {
        const int64_t rt = o / 16, r = o % 16;
        const int64_t tile = (WT == kWPlanarQ8 ? 16 : 8) * K;
        const int lane = 16 * (e / 8) + static_cast<int>(r), e8 = e % 8;
        const uint8_t* s = w + (O + 15) / 16 * tile + ((rt * (K / 256) + kb / 8) * 16 + r) * 16;
        const float d = HalfHw(reinterpret_cast<const uint16_t*>(s)[kb % 8]);
        if constexpr (WT == kWPlanarQ8) {
            const uint8_t* c = w + rt * tile + ((kb / 2) * 64 + lane) * 16 + (kb & 1) * 8;
            return d * static_cast<float>(static_cast<int8_t>(c[e8]));
        } else {
            const uint8_t* c = w + rt * tile + ((kb / 4) * 64 + lane) * 16 + (kb % 4) * 4;
            const int n = (e8 < 4 ? c[e8] : c[e8 - 4] >> 4) & 15;
            return d * static_cast<float>((n ^ 8) - 8);
        }
    } else {
        const uint8_t* b = w + o * row_bytes + kb * Fmt<WT>::kBytes;
        const float d = HalfHw(*reinterpret_cast<const uint16_t*>(b));
        if constexpr (WT == MLK_Q8_0) {
            return d * static_cast<float>(static_cast<int8_t>(b[2 + e]));
        } else if constexpr (WT == MLK_Q4_0) {
            const int n = e < 16 ? b[2 + e] & 15 : b[2 + e - 16] >> 4;
            return d * static_cast<float>(n - 8);
        } else {
            const int n = e < 16 ? b[4 + e] & 15 : b[4 + e - 16] >> 4;
            return __fadd_rn(__fmul_rn(d, static_cast<float>(n)),
                             HalfHw(*reinterpret_cast<const uint16_t*>(b + 2)));
        }
    }
}

// ------------------------------------------------------------ the kernel
// Epilogues.  kStore: y = sum + bias per segment, or partial sums; kAdd: y =
// y + (sum + bias), mlk_add_f32's value (the layer's residual stream);
// kSwiGlu: segments 0 and 1 are gate and up, a tile holds both for the same
// outputs and y of segment 1 gets SwiGlu(gate, up), mlk_swiglu_f32's value.
enum TileEpi { kStore = 0, kAdd = 1, kSwiGlu = 2 };

// Up to three weight matrices with the same K: their output tiles are
// numbered one segment after another (first tile tn0).  With partial sums
// (partial != null, [splits][T][cols]) segment columns start at col0.
struct TileSeg {
    const uint8_t* w;
    const float* bias;
    float* y;
    int64_t rows, col0;
    int tn0;
};

struct TileArgs {
    const float* x;
    TileSeg seg[3];
    int n_seg;
    int64_t T, K, row_bytes;
    int tiles_m, tiles;
    int64_t per_split;
    float* partial;
    int64_t cols;
};

template <int WT, int BM, int BN, int KB>
struct __align__(16) TileSmem {
    uint32_t x[2 * KB][2][BM * 16];
    uint32_t w[2 * KB][kCodes<WT> ? 1 : 2][BN * 16];
    float d[2 * KB][kCodes<WT> ? BN : 4];
};

// dword offset of 16-byte group g of row r in a [rows][32 fp16] stage plane:
// the operand reads of 8 lanes (8 rows, one g) and the writes (4 groups of a
// row) meet distinct bank quads
__device__ inline int At(int r, int g) { return r * 16 + ((g ^ ((r >> 1) & 3)) << 2); }

// over the N lanes that hold one row
template <int N>
__device__ inline float RowSum(float v) {
#pragma unroll
    for (int m = 1; m < N; m *= 2) v += __shfl_xor(v, m, kWave);
    return v;
}
template <int N>
__device__ inline float RowMax(float v) {
#pragma unroll
    for (int m = 1; m < N; m *= 2) v = fmaxf(v, __shfl_xor(v, m, kWave));
    return v;
}

__device__ inline f32x4 Mfma(h8 a, h8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// The outputs of marked rows (rinv 0) and, for split weights, of marked
// outputs (cinv 0) of a tile: one thread an output, its inputs k0 .. k1 - 1
// in order in fp32.
template <int WT, int EPI, int BM, int BN>
__device__ inline void SlowOutputs(const TileArgs& a, const TileSeg& g,
                                                      const float* rinv, const float* cinv,
                                                      int64_t m0, int64_t n0, int64_t k0,
                                                      int64_t k1, float* out, int64_t ldo,
                                                      bool bias) {
    constexpr bool kDual = EPI == kSwiGlu;
    constexpr int kCols = kDual ? BN / 2 : BN;
    for (int e = threadIdx.x; e < BM * kCols; e += static_cast<int>(blockDim.x)) {
        const int r = e / kCols, c = e % kCols;
        const int64_t row = m0 + r, col = n0 + c;
        if (row >= a.T || col >= g.rows) continue;
        bool take = rinv[r] == 0.0f;
        if constexpr (!kCodes<WT>) {
            take = take || cinv[c] == 0.0f || (kDual && cinv[c + BN - kCols] == 0.0f);
        }
        if (!take) continue;
        const auto sum = [&](const TileSeg& sg) {
            float v = 0.0f;
#pragma unroll 8
            for (int64_t k = k0; k < k1; ++k) {
                v = fmaf(a.x[row * a.K + k], Weight<WT>(sg.w, g.rows, a.K, a.row_bytes, col, k), v);
            }
            return v + (bias && sg.bias != nullptr ? sg.bias[col] : 0.0f);
        };
        float* const o = out + row * ldo + col;
        if constexpr (kDual) {
            *o = SwiGluF(sum(g), sum(a.seg[1]));
        } else {
            *o = EPI == kAdd ? *o + sum(g) : sum(g);
        }
    }
}

template <int WT, int MI, int NJ, int WM, int WN, int EPI, int KB>
__global__ __launch_bounds__(64 * WM * WN, 2) void GemmTile(TileArgs a) {
    constexpr int kThreads = 64 * WM * WN;
    constexpr int BM = 16 * MI * WM, BN = 16 * NJ * WN;
    constexpr int kXN = BM * 4 / kThreads;    // 8-input groups of x per thread and stage
    constexpr int kWN = WT == kWF32 ? 2 : 1;  // weight rows per thread and stage
    constexpr int kPl = kCodes<WT> ? 1 : 2;   // weight planes
    constexpr bool kDual = EPI == kSwiGlu;
    static_assert(BN * 2 == kThreads && BM * 4 % kThreads == 0, "one half block per thread");
    static_assert(KB == 1 || kCodes<WT>, "two blocks a stage: codes only");
    using Smem = TileSmem<WT, BM, BN, KB>;
    __shared__ Smem sm;
    __shared__ __align__(16) float rinv[BM];
    __shared__ float cinv[kCodes<WT> ? 4 : BN];
    const int tile = static_cast<int>(blockIdx.x) % a.tiles;
    const int sp = static_cast<int>(blockIdx.x) / a.tiles;
    const int tm = tile % a.tiles_m, tn = tile / a.tiles_m;
    const int sel = !kDual && a.n_seg > 1 && tn >= a.seg[1].tn0
                        ? (a.n_seg > 2 && tn >= a.seg[2].tn0 ? 2 : 1)
                        : 0;
    const TileSeg g = a.seg[sel];
    const int64_t O = g.rows;
    const int64_t m0 = static_cast<int64_t>(tm) * BM;
    const int64_t n0 = static_cast<int64_t>(tn - g.tn0) * (kDual ? BN / 2 : BN);
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int wm = wave % WM, wn = wave / WM;
    const int i16 = lane & 15, kq = lane >> 4;

    const int64_t all = a.K / kBK;
    const int64_t s0 = sp * a.per_split;
    const int64_t s1 = s0 + a.per_split < all ? s0 + a.per_split : all;

    // x: inputs 8 (tid % 4) .. of rows tid / 4 + (kThreads / 4) i.  Rows past
    // T (weight rows past O) read the last one: their outputs are not stored.
    const char* const xbase = reinterpret_cast<const char*>(a.x + m0 * a.K);
    uint32_t xoff[kXN];
#pragma unroll
    for (int i = 0; i < kXN; ++i) {
        const int64_t row = m0 + (tid >> 2) + kThreads / 4 * i;
        xoff[i] = static_cast<uint32_t>(((row < a.T ? row : a.T - 1) - m0) * a.K * 4) +
                  32 * (tid & 3);
    }
    // weights: the tile's rows are rows n0 .. of the segment, or (kDual) its
    // first half of gate and its second of up
    const int h = tid & 1;
    const auto wrow_of = [&](int r) {  // row r of the tile, from n0
        const int64_t row = kDual && r >= BN / 2 ? r - BN / 2 : r;
        return n0 + row < O ? row : O - 1 - n0;
    };
    const int64_t tile_bytes = (WT == kWPlanarQ8 ? 16 : 8) * a.K;
    const int64_t n0_bytes = kPlanar<WT> ? n0 / 16 * tile_bytes : n0 * a.row_bytes;
    const uint8_t* const wb[2] = {g.w + n0_bytes, kDual ? a.seg[1].w + n0_bytes : g.w + n0_bytes};
    // planar: from there to the scales of the same row tile
    const int64_t s_bytes = (O + 15) / 16 * tile_bytes - n0_bytes + n0 / 16 * (a.K / 256) * 256;
    const uint8_t* const wbase = wb[kDual && wave >= WM * WN / 2];  // of row tid / 2
    uint32_t woff[kWN], soff = 0;
    if constexpr (WT == kWF32) {
#pragma unroll
        for (int i = 0; i < kWN; ++i) {
            woff[i] = static_cast<uint32_t>(wrow_of((tid >> 2) + BN / 2 * i) * a.row_bytes) +
                      32 * (tid & 3);
        }
    } else if constexpr (kPlanar<WT>) {
        const int64_t row = wrow_of(tid >> 1);
        woff[0] = static_cast<uint32_t>(row / 16 * tile_bytes + (32 * h + row % 16) * 16);
        soff = static_cast<uint32_t>((row / 16 * (a.K / 256) * 16 + row % 16) * 16);
    } else {
        woff[0] = static_cast<uint32_t>(wrow_of(tid >> 1) * a.row_bytes);
    }
    float4 xv[2][kXN][2];
    RawW<WT> wr[2];
    auto load = [&](int b, int64_t s) {
#pragma unroll
        for (int i = 0; i < kXN; ++i) {
            const float4* p = reinterpret_cast<const float4*>(xbase + s * (kBK * 4) + xoff[i]);
            xv[b][i][0] = p[0];
            xv[b][i][1] = p[1];
        }
        if constexpr (WT == kWF32) {
#pragma unroll
            for (int i = 0; i < kWN; ++i) {
                const float4* p = reinterpret_cast<const float4*>(wb[i] + s * (kBK * 4) + woff[i]);
                wr[b].v[i][0] = p[0];
                wr[b].v[i][1] = p[1];
            }
        } else if constexpr (WT == kWPlanarQ8) {
            wr[b].Load(wbase + s / 2 * 1024 + s % 2 * 8, woff[0],
                       wbase + s_bytes + s / 8 * 256 + s % 8 * 2, soff);
        } else if constexpr (WT == kWPlanarQ4) {
            wr[b].Load(wbase + s / 4 * 1024 + s % 4 * 4, woff[0],
                       wbase + s_bytes + s / 8 * 256 + s % 8 * 2, soff);
        } else {
            wr[b].Load(wbase + s * Fmt<WT>::kBytes, woff[0], h);
        }
    };
    load(0, s0);
    load(1, s0 + 1 < s1 ? s0 + 1 : s0);
    // the rows' scales, from their first 64 inputs
    PieceScale xs[kXN], wsc[kWN];
    float xmost[kXN], wmost[kWN];
#pragma unroll
    for (int i = 0; i < kXN; ++i) {
        xs[i] = PieceScale(RowSum<4>(AbsSum8(xv[0][i]) + AbsSum8(xv[1][i])) * (1.0f / 64.0f));
        xmost[i] = 0.0f;
    }
#pragma unroll
    for (int i = 0; i < kWN; ++i) {
        wmost[i] = 0.0f;
        if constexpr (WT == kWF32) {
            wsc[i] = PieceScale(RowSum<4>(AbsSum8(wr[0].v[i]) + AbsSum8(wr[1].v[i])) *
                                (1.0f / 64.0f));
        } else if constexpr (WT == MLK_Q4_1) {
            float4 e[2][2], f[2][2];
            Values16(wr[0], h, e);
            Values16(wr[1], h, f);
            wsc[i] = PieceScale(RowSum<2>((AbsSum8(e[0]) + AbsSum8(e[1])) +
                                          (AbsSum8(f[0]) + AbsSum8(f[1]))) *
                                (1.0f / 64.0f));
        }
    }

    // a stage's registers b into LDS buffer buf
    auto store = [&](int buf, int b) {
        u32x4 p0, p1;
#pragma unroll
        for (int i = 0; i < kXN; ++i) {
            Split8(xv[b][i], xs[i].s, &p0, &p1);
            xmost[i] = AbsMax8(xv[b][i], xmost[i]);
            const int at = At((tid >> 2) + kThreads / 4 * i, tid & 3);
            *reinterpret_cast<u32x4*>(&sm.x[buf][0][at]) = p0;
            *reinterpret_cast<u32x4*>(&sm.x[buf][1][at]) = p1;
        }
        if constexpr (kCodes<WT>) {
            u32x4 c[2];
            Codes16<WT>(wr[b], h, c);
            *reinterpret_cast<u32x4*>(&sm.w[buf][0][At(tid >> 1, 2 * h)]) = c[0];
            *reinterpret_cast<u32x4*>(&sm.w[buf][0][At(tid >> 1, 2 * h + 1)]) = c[1];
            sm.d[buf][tid >> 1] = HalfHw(wr[b].d & 0xFFFFu);
        } else {
            float4 q[2][2];
            if constexpr (WT == MLK_Q4_1) Values16(wr[b], h, q);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                if constexpr (WT == kWF32) {
                    q[i][0] = wr[b].v[i][0];
                    q[i][1] = wr[b].v[i][1];
                }
                const int k = WT == kWF32 ? i : 0;
                Split8(q[i], wsc[k].s, &p0, &p1);
                wmost[k] = AbsMax8(q[i], wmost[k]);
                const int at = WT == kWF32 ? At((tid >> 2) + BN / 2 * i, tid & 3)
                                           : At(tid >> 1, 2 * h + i);
                *reinterpret_cast<u32x4*>(&sm.w[buf][0][at]) = p0;
                *reinterpret_cast<u32x4*>(&sm.w[buf][kPl - 1][at]) = p1;
            }
        }
    };

    f32x4 acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    // KB stages from s on, in LDS buffers KB u ..  The next KB stages wait in
    // registers and go into the other buffers, the ones after them are
    // requested (past the last stage: the last again, not used).  One basic
    // block, one barrier.
    auto step = [&](int64_t s, int u) {
        h8 b[KB][kPl][NJ];
        float dj[KB][NJ];
#pragma unroll
        for (int k = 0; k < KB; ++k) {
            const int buf = KB * u + k;
            if constexpr (KB == 1) load(u, s + 2 < s1 ? s + 2 : s1 - 1);
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int row = wn * 16 * NJ + 16 * j + i16;
#pragma unroll
                for (int p = 0; p < kPl; ++p) {
                    b[k][p][j] = *reinterpret_cast<const h8*>(&sm.w[buf][p][At(row, kq)]);
                }
                if constexpr (kCodes<WT>) dj[k][j] = sm.d[buf][row];
            }
        }
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            if (i % (MI / KB) == 0) {
                constexpr int kh = MI / KB;
                if (i > 0) __builtin_amdgcn_sched_barrier(0);
                store(KB * (u ^ 1) + i / kh, KB == 1 ? u ^ 1 : i / kh);
                if constexpr (KB == 2) load(i / kh, s + 4 + i / kh < s1 ? s + 4 + i / kh : s1 - 1);
            }
            h8 hi[KB], lo[KB];
            const int at = At(wm * 16 * MI + 16 * i + i16, kq);
#pragma unroll
            for (int k = 0; k < KB; ++k) {
                hi[k] = *reinterpret_cast<const h8*>(&sm.x[KB * u + k][0][at]);
                lo[k] = *reinterpret_cast<const h8*>(&sm.x[KB * u + k][1][at]);
            }
            if constexpr (kCodes<WT>) {
                f32x4 S[KB][NJ];
#pragma unroll
                for (int k = 0; k < KB; ++k) {
#pragma unroll
                    for (int j = 0; j < NJ; ++j) {
                        S[k][j] = Mfma(lo[k], b[k][0][j], f32x4{0.f, 0.f, 0.f, 0.f});
                    }
#pragma unroll
                    for (int j = 0; j < NJ; ++j) S[k][j] = Mfma(hi[k], b[k][0][j], S[k][j]);
                }
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        if constexpr (KB == 2) {  // one rounding of acc for two blocks
                            acc[i][j][r] += fmaf(dj[1][j], S[KB - 1][j][r], dj[0][j] * S[0][j][r]);
                        } else {
                            acc[i][j][r] += dj[0][j] * S[0][j][r];
                        }
                    }
                }
            } else {
#pragma unroll
                for (int j = 0; j < NJ; ++j) acc[i][j] = Mfma(lo[0], b[0][0][j], acc[i][j]);
#pragma unroll
                for (int j = 0; j < NJ; ++j) acc[i][j] = Mfma(hi[0], b[0][kPl - 1][j], acc[i][j]);
#pragma unroll
                for (int j = 0; j < NJ; ++j) acc[i][j] = Mfma(hi[0], b[0][0][j], acc[i][j]);
            }
        }
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
    };
    store(0, 0);
    if constexpr (KB == 2) {
        store(1, 1);
        load(0, s0 + 2 < s1 ? s0 + 2 : s1 - 1);
        load(1, s0 + 3 < s1 ? s0 + 3 : s1 - 1);
    }
    __syncthreads();
    int64_t s = s0;
    for (; s + KB < s1; s += 2 * KB) {
        step(s, 0);
        step(s + KB, 1);
    }
    if (s < s1) step(s, 0);

    // the factors that undo the scales; 0 marks a row whose values leave the
    // pieces' range
    bool bad = false;
#pragma unroll
    for (int i = 0; i < kXN; ++i) {
        const float inv = xs[i].Checked(RowMax<4>(xmost[i]));
        rinv[(tid >> 2) + kThreads / 4 * i] = inv;
        bad |= inv == 0.0f;
    }
    if constexpr (!kCodes<WT>) {
#pragma unroll
        for (int i = 0; i < kWN; ++i) {
            const float inv = wsc[i].Checked(RowMax<WT == kWF32 ? 4 : 2>(wmost[i]));
            cinv[WT == kWF32 ? (tid >> 2) + BN / 2 * i : tid >> 1] = inv;
            bad |= inv == 0.0f;
        }
    }
    const bool any_bad = __syncthreads_or(bad) != 0;

    const bool part = a.partial != nullptr;
    const int64_t ldo = part ? a.cols : O;
    float* const out = part ? a.partial + sp * a.T * a.cols + g.col0 : (kDual ? a.seg[1].y : g.y);
    const auto value = [&](int i, int j, int r, float ri) {
        if constexpr (kCodes<WT>) {
            return acc[i][j][r] * ri;
        } else {
            return acc[i][j][r] * (ri * cinv[wn * 16 * NJ + 16 * j + i16]);
        }
    };
    const auto factors = [&](int i) {
        return *reinterpret_cast<const f32x4*>(&rinv[wm * 16 * MI + 16 * i + 4 * kq]);
    };
    if constexpr (kDual) {
        // The stage buffers are free.  Gate wave (wm, wn) and up wave
        // (wm, wn + WN / 2) hold the same outputs in the same registers:
        // lane l of one hands lane l of the other its sums.
        static_assert(sizeof(Smem) >= sizeof(float4) * MI * NJ * 64 * WM * (WN / 2),
                      "the gate sums fit the stage buffers");
        float4* const xch =
            reinterpret_cast<float4*>(&sm) + (wm * (WN / 2) + wn % (WN / 2)) * MI * NJ * 64 + lane;
        const bool up = wn >= WN / 2;
        if (!up) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int64_t col = n0 + wn * 16 * NJ + 16 * j + i16;
                const float bg = g.bias != nullptr && col < O ? g.bias[col] : 0.0f;
#pragma unroll
                for (int i = 0; i < MI; ++i) {
                    const f32x4 ri = factors(i);
                    xch[(NJ * i + j) * 64] =
                        make_float4(value(i, j, 0, ri[0]) + bg, value(i, j, 1, ri[1]) + bg,
                                    value(i, j, 2, ri[2]) + bg, value(i, j, 3, ri[3]) + bg);
                }
            }
        }
        __syncthreads();
        if (up) {
            const float* const bias = a.seg[1].bias;
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int64_t col = n0 + (wn - WN / 2) * 16 * NJ + 16 * j + i16;
                if (col >= O) continue;
                const float bu = bias != nullptr ? bias[col] : 0.0f;
                bool bad_col = false;
                if constexpr (!kCodes<WT>) {
                    const int c = wn * 16 * NJ + 16 * j + i16;
                    bad_col = cinv[c] == 0.0f || cinv[c - BN / 2] == 0.0f;
                }
#pragma unroll
                for (int i = 0; i < MI; ++i) {
                    const f32x4 ri = factors(i);
                    const float4 g4 = xch[(NJ * i + j) * 64];
                    const float gv[4] = {g4.x, g4.y, g4.z, g4.w};
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int64_t row = m0 + wm * 16 * MI + 16 * i + 4 * kq + r;
                        if (row >= a.T || bad_col || ri[r] == 0.0f) continue;
                        out[row * ldo + col] = SwiGluF(gv[r], value(i, j, r, ri[r]) + bu);
                    }
                }
            }
        }
    } else {
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int64_t col = n0 + wn * 16 * NJ + 16 * j + i16;
            if (col >= O) continue;
            const float bb = !part && g.bias != nullptr ? g.bias[col] : 0.0f;
            bool bad_col = false;
            if constexpr (!kCodes<WT>) bad_col = cinv[wn * 16 * NJ + 16 * j + i16] == 0.0f;
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                const f32x4 ri = factors(i);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int64_t row = m0 + wm * 16 * MI + 16 * i + 4 * kq + r;
                    if (row >= a.T || bad_col || ri[r] == 0.0f) continue;
                    float* const o = out + row * ldo + col;
                    if constexpr (EPI == kAdd) {
                        *o = *o + (value(i, j, r, ri[r]) + bb);
                    } else {
                        *o = value(i, j, r, ri[r]) + bb;
                    }
                }
            }
        }
    }
    if (any_bad) {
        SlowOutputs<WT, EPI, BM, BN>(a, g, rinv, cinv, m0, n0, s0 * kBK, s1 * kBK, out, ldo, !part);
    }
}


// ------------------------------------------------------------ launches
// Tile shape and K splits of a launch.
//   128 x 256 (one workgroup a CU) for more than 64 rows, where up to 8
//       splits (more while each keeps 16 stages) give 3/4 of a workgroup a
//       CU; past that K is not split: T = 389 over 14336 outputs (224 tiles,
//       Q8_0) took 150 us unsplit, 176 us in two splits of 1.75 rounds.
//   32 x 64 up to 32 rows, split to 4 workgroups a CU (33 KB of LDS each),
//       each split at least 8 stages.  16 rows of F32: w_gate 52 us (fp32
//       MFMA 52), wo 19.9 (20.2); 32 rows of Q8_0 / Q4_0: w_gate 42 / 40 us
//       (skinny kernel, fp32 MFMA, 48 / 47), 128256 outputs 263 / 216 (355 /
//       366, whose 8 splits' partial sums alone are 131 MB).  On 64 x 128
//       tiles the same take 46, 21.7, 40 / 39 and 265 / 228, Q8_0 wo 22 (19.3
//       here).
//   64 x 128 otherwise, split to 1.5 workgroups a CU, each split at least 8
//       stages.  Q8_0: T = 64 over 4096 x 14336 39.6 us in 16 splits (512
//       workgroups), 46 in 8; 128 rows over 4096 x 4096 31 us against 34-37
//       on 128 x 256, over 14336 x 4096 70 against 55.
// Measured beside these: 128 x 128 tiles (4 waves) 7-14% slower than 128 x
// 256 at every T from 200 to 4096.
struct TilePlan {
    int bm = 64;
    int splits = 1;
    int64_t per_split = 0, tiles_m = 0, tiles = 0;
    int Bm() const { return bm; }
    int Bn() const { return 2 * bm; }
};

// rows: outputs per segment; dual: gate and up in one tile
TilePlan MakeTilePlan(int64_t T, int64_t K, const int64_t* rows, int n_seg, bool dual, bool split) {
    const int64_t cus = ComputeUnits(), stages = K / kBK;
    TilePlan p;
    const auto count = [&](int bm) {
        p.bm = bm;
        p.tiles_m = (T + p.Bm() - 1) / p.Bm();
        int64_t tn = 0;
        for (int i = 0; i < (dual ? 1 : n_seg); ++i) {
            const int64_t bn = dual ? p.Bn() / 2 : p.Bn();
            tn += (rows[i] + bn - 1) / bn;
        }
        p.tiles = p.tiles_m * tn;
    };
    int64_t sp = 1;
    bool wide = T > 64;
    if (wide) {
        count(128);
        while (p.tiles * sp * 4 < 3 * cus && stages / (2 * sp) >= 16 && sp < 32) sp *= 2;
        wide = p.tiles * sp * 4 >= 3 * cus;
    }
    if (!wide) {
        count(T <= 32 ? 32 : 64);
        const int64_t half_wgs = T <= 32 ? 8 : 3;  // per CU
        sp = 1;
        while (p.tiles * sp * 2 < half_wgs * cus && stages / (2 * sp) >= 8 && sp < 32) sp *= 2;
    }
    if (!split) sp = 1;
    p.per_split = (stages + sp - 1) / sp;
    if (stages % 2 == 0) p.per_split += p.per_split % 2;  // whole pairs of blocks
    p.splits = static_cast<int>((stages + p.per_split - 1) / p.per_split);
    return p;
}

template <int WT, int EPI>
void LaunchEpi(const TilePlan& p, hipStream_t s, const TileArgs& a) {
    const dim3 grid(static_cast<unsigned>(p.tiles * p.splits));
    constexpr int kPair = kCodes<WT> ? 2 : 1;
    const bool pair = kCodes<WT> && a.K % 64 == 0;
    if (p.bm == 128) {
        if (pair) {
            hipLaunchKernelGGL((GemmTile<WT, 4, 4, 2, 4, EPI, kPair>), grid, dim3(512), 0, s, a);
        } else {
            hipLaunchKernelGGL((GemmTile<WT, 4, 4, 2, 4, EPI, 1>), grid, dim3(512), 0, s, a);
        }
    } else if (p.bm == 32) {
        if (pair) {
            hipLaunchKernelGGL((GemmTile<WT, 2, 2, 1, 2, EPI, kPair>), grid, dim3(128), 0, s, a);
        } else {
            hipLaunchKernelGGL((GemmTile<WT, 2, 2, 1, 2, EPI, 1>), grid, dim3(128), 0, s, a);
        }
    } else if (pair) {
        hipLaunchKernelGGL((GemmTile<WT, 2, 4, 2, 2, EPI, kPair>), grid, dim3(256), 0, s, a);
    } else {
        hipLaunchKernelGGL((GemmTile<WT, 2, 4, 2, 2, EPI, 1>), grid, dim3(256), 0, s, a);
    }
}

template <int WT>
void LaunchWt(const TilePlan& p, int epi, hipStream_t s, const TileArgs& a) {
    if constexpr (kPlanar<WT>) {
        LaunchEpi<WT, kStore>(p, s, a);
    } else if (epi == kAdd) {
        LaunchEpi<WT, kAdd>(p, s, a);
    } else if (epi == kSwiGlu) {
        LaunchEpi<WT, kSwiGlu>(p, s, a);
    } else {
        LaunchEpi<WT, kStore>(p, s, a);
    }
}

// Fills a's tiles from the plan and launches; segments' w, bias, y, rows set.
mlk_status Run(int wt, const TilePlan& p, int epi, TileArgs& a, float* partial, hipStream_t s) {
    if (p.tiles * p.splits > 0x7FFFFFFF) {
        return Fail(MLK_ERR_INVALID, "linear: %lld tiles exceed one launch",
                    static_cast<long long>(p.tiles * p.splits));
    }
    int64_t col = 0, tn = 0;
    for (int i = 0; i < a.n_seg; ++i) {
        a.seg[i].col0 = col;
        a.seg[i].tn0 = static_cast<int>(tn);
        col += a.seg[i].rows;
        if (epi != kSwiGlu) tn += (a.seg[i].rows + p.Bn() - 1) / p.Bn();
    }
    a.cols = col;
    a.tiles_m = static_cast<int>(p.tiles_m);
    a.tiles = static_cast<int>(p.tiles);
    a.per_split = p.per_split;
    a.partial = partial;
    switch (wt) {
        case MLK_Q8_0: LaunchWt<MLK_Q8_0>(p, epi, s, a); break;
        case MLK_Q4_0: LaunchWt<MLK_Q4_0>(p, epi, s, a); break;
        case MLK_Q4_1: LaunchWt<MLK_Q4_1>(p, epi, s, a); break;
        case kWPlanarQ8: LaunchWt<kWPlanarQ8>(p, epi, s, a); break;
        case kWPlanarQ4: LaunchWt<kWPlanarQ4>(p, epi, s, a); break;
        default: LaunchWt<kWF32>(p, epi, s, a); break;
    }
    return CheckLaunch("GemmTile");
}

bool WorkspaceOk(const void* workspace, size_t bytes, int64_t need) {
    return workspace != nullptr && Aligned(workspace, 16) && bytes >= static_cast<size_t>(need);
}

}  // namespace

bool TileApplies(int wt, int64_t T, int64_t K) {
    // the 32-bit row offsets of a tile hold 256 rows of 2^22 fp32 inputs
    return T > 0 && K >= 256 && K <= (int64_t{1} << 22) &&
           K % (wt == kWPlanarQ8 || wt == kWPlanarQ4 ? 256 : 32) == 0;
}

bool TileChosen(int wt, int64_t T, int64_t K, int64_t cols, bool fused) {
    if (!TileApplies(wt, T, K)) return false;
    if (T > 32) return true;
    const int64_t n = K * cols;
    if (wt == kWF32) return T >= 8 || (T >= 5 && n >= kFewRowsMin);
    return (wt == MLK_Q8_0 || wt == MLK_Q4_0) && T > 16 && n >= (fused ? kLayerGroupMin : kFewRowsMin);
}

bool TileWeightAligned(int wt, const void* w) {
    return Aligned(w, wt == kWF32 ? 16 : (wt == MLK_Q4_1 ? 4 : 2));
}

int64_t TileWorkspaceBytes(int64_t T, int64_t K, int64_t O) {
    return TileFusedPlan(T, K, &O, 1).bytes;
}

mlk_status LaunchTile(int wt, const float* x, const void* w, const float* bias, float* y, int64_t T,
                      int64_t K, int64_t O, int64_t row_bytes, void* workspace,
                      size_t workspace_bytes, hipStream_t s) {
    TilePlan p = MakeTilePlan(T, K, &O, 1, false, true);
    if (p.splits > 1 && !WorkspaceOk(workspace, workspace_bytes, p.splits * T * O * 4)) {
        p = MakeTilePlan(T, K, &O, 1, false, false);
    }
    TileArgs a{};
    a.x = x;
    a.seg[0] = TileSeg{static_cast<const uint8_t*>(w), bias, y, O, 0, 0};
    a.n_seg = 1;
    a.T = T;
    a.K = K;
    a.row_bytes = row_bytes;
    float* partial = p.splits > 1 ? static_cast<float*>(workspace) : nullptr;
    const mlk_status st = Run(wt, p, kStore, a, partial, s);
    if (st != MLK_OK || partial == nullptr) return st;
    return ReduceSplits(partial, p.splits, bias, y, T, O, s);
}

TileFused TileFusedPlan(int64_t T, int64_t K, const int64_t* rows, int n_seg) {
    const TilePlan p = MakeTilePlan(T, K, rows, n_seg, false, true);
    TileFused f;
    f.splits = p.splits;
    if (p.splits > 1) {
        for (int i = 0; i < n_seg; ++i) f.bytes += p.splits * T * rows[i] * 4;
    }
    return f;
}

mlk_status LinearTileFused(int wt, const float* x, int64_t T, int64_t K, const StreamArgs& sa,
                           int mode, void* workspace, size_t workspace_bytes, hipStream_t s) {
    const bool block = wt == MLK_Q8_0 || wt == MLK_Q4_0 || wt == MLK_Q4_1;
    if ((!block && wt != kWF32) || !TileApplies(wt, T, K) || !Aligned(x, 16) || sa.n_seg < 1 ||
        sa.n_seg > 3 || (mode == kStreamAdd && sa.n_seg != 1) ||
        (mode == kStreamSwiGlu && (sa.n_seg != 2 || sa.seg[0].rows != sa.seg[1].rows)) ||
        (mode == kStreamQkvRope && !QkvRopeArgsOk(sa))) {
        return Fail(MLK_ERR_INVALID, "linear (tiles, fused): unsupported shape");
    }
    TileArgs a{};
    int64_t rows[3] = {0, 0, 0};
    for (int i = 0; i < sa.n_seg; ++i) {
        const StreamSeg& g = sa.seg[i];
        const bool out = mode != kStreamSwiGlu || i == 1;  // gate's y is not written
        if (g.w == nullptr || !TileWeightAligned(wt, g.w) || g.rows <= 0 ||
            (out && g.y == nullptr) || (mode == kStreamAdd && g.res != g.y) ||
            // outputs are written while other workgroups still read x
            (out && g.y < x + T * K && x < g.y + T * g.rows)) {
            return Fail(MLK_ERR_INVALID, "linear (tiles, fused): bad segment %d", i);
        }
        rows[i] = g.rows;
        a.seg[i] = TileSeg{g.w, g.bias, g.y, g.rows, 0, 0};
    }
    a.x = x;
    a.n_seg = sa.n_seg;
    a.T = T;
    a.K = K;
    a.row_bytes = block ? K / 32 * BlockBytes(wt) : K * 4;
    TilePlan p = MakeTilePlan(T, K, rows, sa.n_seg, false, true);
    if (p.splits > 1) {
        const int64_t need = TileFusedPlan(T, K, rows, sa.n_seg).bytes;
        if (!WorkspaceOk(workspace, workspace_bytes, need)) {
            return Fail(MLK_ERR_INVALID, "linear (tiles, fused): workspace of %lld bytes needed",
                        static_cast<long long>(need));
        }
        float* partial = static_cast<float*>(workspace);
        const mlk_status st = Run(wt, p, kStore, a, partial, s);
        if (st != MLK_OK) return st;
        return ReduceSplitsFused(partial, p.splits, T, a.cols, sa, mode, s);
    }
    if (mode == kStreamQkvRope) {
        return Fail(MLK_ERR_INVALID, "linear (tiles, fused): RoPE only in a reduction");
    }
    if (mode == kStreamSwiGlu) {
        p = MakeTilePlan(T, K, rows, 2, true, false);
        return Run(wt, p, kSwiGlu, a, nullptr, s);
    }
    return Run(wt, p, mode == kStreamAdd ? kAdd : kStore, a, nullptr, s);
}

mlk_status LinearTilePartials(int wt, const float* x, const void* w, int64_t T, int64_t K,
                              int64_t O, void* workspace, size_t workspace_bytes, hipStream_t s,
                              float** partial, int* splits) {
    const bool block = wt == MLK_Q8_0 || wt == MLK_Q4_0 || wt == MLK_Q4_1;
    const TilePlan p = MakeTilePlan(T, K, &O, 1, false, true);
    if ((!block && wt != kWF32) || !TileApplies(wt, T, K) || !Aligned(x, 16) ||
        !TileWeightAligned(wt, w) || p.splits < 2 ||
        !WorkspaceOk(workspace, workspace_bytes, p.splits * T * O * 4)) {
        return Fail(MLK_ERR_INVALID, "linear (tiles): no partial sums for this call");
    }
    TileArgs a{};
    a.x = x;
    a.seg[0] = TileSeg{static_cast<const uint8_t*>(w), nullptr, nullptr, O, 0, 0};
    a.n_seg = 1;
    a.T = T;
    a.K = K;
    a.row_bytes = block ? K / 32 * BlockBytes(wt) : K * 4;
    *partial = static_cast<float*>(workspace);
    *splits = p.splits;
    return Run(wt, p, kStore, a, *partial, s);
}

}  // namespace mlk
