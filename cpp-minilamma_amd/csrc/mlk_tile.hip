// mlk_tile.hip -- many-row linear layers on the fp16 matrix cores:
// y[T, O] = x[T, K] W[O, K]^T (+ bias), W fp32, Q8_0 / Q4_0 / Q4_1 blocks or
// planar Q8_0 / Q4_0, for more than 32 rows (F32 from 5, Q8_0 and Q4_0 blocks
// from 17 where the weights are large: TileChosen) and K a multiple of 32, at
// least 256 (other shapes: mlk_linear.hip, mlk_gemm.hip).  Semantics as there
// (LinearQ80 / Q40 / Q41, src/quant.cc:393-463; cublasSgemm,
// src/cuda_matmul.cc:142-186): fp32 products and sums, in an order of this
// kernel's choosing.
//
// Products.  Each row of x (and of fp32 or Q4_1 weights, decoded to the
// reference's fp32 values) is scaled by a power of two s and split into two
// fp16 pieces: x s = x0 + 2^-11 x1, x0 the value rounded to fp16, x1 the rest
// times 2^11 rounded to fp16.  Where |x s| >= 2^-14 the pieces hold it to
// 2^-23 of itself, below to 2^-36.
//   codes (Q8_0, Q4_0)    a code is a small integer, exact in fp16 also
//       times 2^-11, so a block's sum S = sum (code x0 + (2^-11 code) x1) is
//       two v_mfma_f32_16x16x32_f16, then acc += d S + d' S' for a pair of
//       blocks, in fp32 (one rounding of acc for two blocks: with one per
//       block the sums were 2.2e-7 off at K = 4096 instead of 1.7e-7, and the
//       kernel 5% faster).
//   values (F32, Q4_1)    S = x1 w0 + x0 w1, acc += x0 w0 (three MFMAs), then
//       acc += 2^-11 S; x1 w1 is left out.  (S kept over all stages instead:
//       within 1% at 8 rows of F32, Q4_1 437 -> 466 us at 800 rows.)
// Three bf16 pieces per x (exact products) and the fp32 MFMA, which these
// replace, took 3 and, at an eighth of the rate, 8 times the matrix work.
// Errors against float64 (relative 2-norm, normal x and weights, K = 4096
// unsplit): Q8_0 1.7e-7 (three pieces: 2.1e-7), F32 and Q4_1 4.6e-7 (fp32
// MFMA: 1.15e-6).  Time at 4096 rows, K = 4096, 14336 outputs: Q8_0 1363 ->
// 1217 us, F32 3659 -> 1678, Q4_1 3827 -> 1551; at 64 rows Q8_0 91 -> 43.
//
// Scales and range.  s puts the largest of a row's first 64 inputs of the K
// split (where those are zero, the first that are not of 64 at 7 places
// further on) at [2^7, 2^8), weights' at [2^10, 2^11).  Every thread keeps the
// largest and the smallest nonzero magnitude of the rows it loads, in fp32 (of
// Q4_1 blocks bounds of both from d and m).  After the K loop a row is marked
// unless every value is below 65504 / s (infinities are not) and every nonzero
// one at least 2^-11 / (K s), for values 2^-10 / (K s); and for values also a
// row of x whose smallest scaled magnitude times the tile's smallest is below
// 2^-25 / K.  A product of an unmarked output is then within
//   codes   (4 + K / 2) u |x w|, the K only for x at that lower bound (the
//           pieces' 2^-36 against it; u = 2^-24)
//   values  (8 + K / 4 + K / 4 + K / 2) u |x w|, the terms in K for x and w at
//           the lower bounds and x1 w1 (up to 2^-50) at the bound of the pair
// of its exact value, whatever the row's other values are and whichever of
// them meet weights of zero.  Marked outputs are summed again as fp32 products
// (MarkedRow, MarkedOutputs).  A row's values do not depend on the tile's other
// rows, but for the order of a marked row's sums (one for up to 8 marked rows,
// one for more).  Rows are marked that reach about 2^8 above or 2^(18 + log2 K)
// below their first inputs; of normal rows about one in 10^5, of SwiGLU's
// outputs one in 10^4.  Time (Q8_0, 4096 rows, K = 4096, 14336 outputs): one
// marked row in every tile 1217 -> 1540 us, all rows marked 7160; first inputs
// zero: no difference.  NaNs pass through the products.  Keeping both
// magnitudes takes about 4% of the call, scaling the second pieces 3%.
//
// Work.  A workgroup owns BM token rows x BN outputs (32 x 64, 2 waves, 64 x
// 128, 4 waves, or 128 x 256, 8 waves), a wave a 16 MI x 16 NJ part of them,
// K in stages of 32 through LDS; while stages are multiplied the next ones, already in
// registers, are split, decoded and written to the other LDS buffers, and
// the ones after them are requested from memory.  Few tiles: K is split over
// workgroups, partial sums reduced in split order (mlk_gemm.hip).
//
// Bound: a stage of a 128 x 256 tile (T = 4096, Q8_0) takes about 2900
// cycles where its MFMAs take 1024 a SIMD; before the range was kept and the
// second pieces scaled 2800, then without the loads from memory 2080, without
// loads, splits, decodes and LDS writes 1850, the scale FMAs 190 of it
// (timing-only copies).  Not the order of instructions, deeper requests (3
// and 4 stages ahead), coalesced weight pieces through LDS, or the two halves
// of the waves half a stage apart: each the same or slower.
#include "mlk_quant.h"

#include <type_traits>

namespace mlk {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef uint16_t us2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_a2 __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kWF32 = -1;
constexpr int kBK = 32;  // inputs per stage: one quantization block

template <int WT>
constexpr bool kCodes = WT == MLK_Q8_0 || WT == MLK_Q4_0 || WT == kWPlanarQ8 || WT == kWPlanarQ4;

template <int WT>
constexpr bool kPlanar = WT == kWPlanarQ8 || WT == kWPlanarQ4;

constexpr float kLowUp = 2048.0f;  // second pieces are kept times 2^11

__device__ inline uint32_t AsU32(h2 v) { return __builtin_bit_cast(uint32_t, v); }

// ------------------------------------------------------------ fp16 pieces
// v s = p0 + 2^-11 p1 (+ at most 2^-23 of v s, or 2^-36 where that is more),
// p0 and p1 fp16; 8 values, two a dword.  (The asm hides where p0 came from,
// which would otherwise be rounded twice: Q8_0 at 4096 rows 1203 -> 1183 us.)
__device__ inline void Split8(const float4 (&v)[2], float s, u32x4* p0, u32x4* p1) {
    const float f[8] = {v[0].x, v[0].y, v[0].z, v[0].w, v[1].x, v[1].y, v[1].z, v[1].w};
    const float s2 = s * kLowUp;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float a = f[2 * i] * s2, b = f[2 * i + 1] * s2;
        h2 hi, lo;
        hi.x = static_cast<_Float16>(a * (1.0f / kLowUp));
        hi.y = static_cast<_Float16>(b * (1.0f / kLowUp));
        uint32_t u = AsU32(hi);
        asm("" : "+v"(u));
        hi = __builtin_bit_cast(h2, u);
        lo.x = static_cast<_Float16>(fmaf(static_cast<float>(hi.x), -kLowUp, a));
        lo.y = static_cast<_Float16>(fmaf(static_cast<float>(hi.y), -kLowUp, b));
        (*p0)[i] = u;
        (*p1)[i] = AsU32(lo);
    }
}

__device__ inline float AbsMax8(const float4 (&v)[2], float m) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        m = fmaxf(fmaxf(m, fabsf(v[i].x)), fabsf(v[i].y));
        m = fmaxf(fmaxf(m, fabsf(v[i].z)), fabsf(v[i].w));
    }
    return m;
}

// Smallest magnitude but zero, as a key that orders like it (infinities and
// NaNs above every finite value, zero above all).
constexpr uint32_t kNoKey = 0xFFFFFFFFu;
__device__ inline uint32_t LeastKey(float v) { return (__float_as_uint(v) << 1) - 1u; }
__device__ inline uint32_t LeastKey8(const float4 (&v)[2], uint32_t m) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        m = min(min(m, LeastKey(v[i].x)), LeastKey(v[i].y));
        m = min(min(m, LeastKey(v[i].z)), LeastKey(v[i].w));
    }
    return m;
}
__device__ inline float KeyValue(uint32_t k) {
    return k == kNoKey ? INFINITY : __uint_as_float((k + 1u) >> 1);
}

// The power of two that brings `first`, the largest magnitude of a row's
// first inputs, into [2^at, 2^(at + 1)) and its inverse (2^at for zero,
// subnormal, infinite and NaN values; within 2^(at - 61) .. 2^(at + 61)).  x
// takes at = 7: room for activations of 250 times that magnitude; weights 10.
struct PieceScale {
    float s = 1.0f, inv = 1.0f;
    __device__ PieceScale() {}
    __device__ PieceScale(float first, int at) {
        int e = static_cast<int>((__float_as_uint(first) >> 23) & 255u);
        e = e == 0 || e == 255 ? 127 : (e < 66 ? 66 : (e > 188 ? 188 : e));
        s = __uint_as_float(static_cast<uint32_t>(254 + at - e) << 23);
        inv = __uint_as_float(static_cast<uint32_t>(e - at) << 23);
    }
    // whether a row's values lie in the pieces' range: its largest magnitude
    // and its smallest but zero
    __device__ bool Fits(float most, float least, float low_min) const {
        return most == 0.0f || (most * s < 65504.0f && least * s >= low_min);
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

// A Q4_1 block's range from its scale d and minimum m: no value is above
// |m| + 15 |d|, and as a multiple of the spacing of both no value but zero is
// below the smaller spacing (2^(e - 25) at exponent field e).
__device__ inline float BlockMost(const RawW<MLK_Q4_1>& r) {
    return fmaf(15.0f, fabsf(HalfHw(r.d & 0xFFFFu)), fabsf(HalfHw(r.d >> 16)));
}
// both magnitudes less one: zero above all
__device__ inline us2 BlockKeys(const RawW<MLK_Q4_1>& r) {
    return __builtin_bit_cast(us2, r.d & 0x7FFF7FFFu) - us2{1, 1};
}
__device__ inline float KeySpacing(us2 k) {
    const uint32_t m = k.x < k.y ? k.x : k.y;
    if (m == 0xFFFFu) return INFINITY;
    const uint32_t e = (m + 1u) >> 10;
    return __uint_as_float((102u + (e > 0 ? e : 1)) << 23);
}

// 8 weights of row o in block kb: inputs e .. e + 3 and 16 + e .. 16 + e + 3
// of its 32 (e = 0, 4, 8 or 12), as loaded and as the reference's fp32 values
// (codes: exact).
template <int WT>
struct Raw8 {
    uint32_t d, u[2];  // scale (Q4_1: and minimum), 4 codes each
    __device__ void Load(const uint8_t* w, int64_t O, int64_t K, int64_t row_bytes, int64_t o,
                         int64_t kb, int e) {
        typedef uint32_t u32_a2 __attribute__((aligned(2)));
        if constexpr (kPlanar<WT>) {
            const int64_t rt = o / 16, r = o % 16;
            const int64_t tile = (WT == kWPlanarQ8 ? 16 : 8) * K;
            const uint8_t* s = w + (O + 15) / 16 * tile;
            d = *reinterpret_cast<const uint16_t*>(
                s + ((rt * (K / 256) + kb / 8) * 16 + r) * 16 + kb % 8 * 2);
#pragma unroll
            for (int c = 0; c < 2; ++c) {  // 8 inputs from 16 c + e / 8 * 8 on
                const int64_t at = 16 * (2 * c + e / 8) + r;
                const uint8_t* q =
                    WT == kWPlanarQ8 ? w + rt * tile + (kb / 2 * 64 + at) * 16 + kb % 2 * 8 + e % 8
                                     : w + rt * tile + (kb / 4 * 64 + at) * 16 + kb % 4 * 4;
                u[c] = *reinterpret_cast<const uint32_t*>(q);
            }
        } else {
            const uint8_t* b = w + o * row_bytes + kb * Fmt<WT>::kBytes;
            if constexpr (WT == MLK_Q4_1) {
                d = *reinterpret_cast<const uint32_t*>(b);
                u[0] = u[1] = *reinterpret_cast<const uint32_t*>(b + 4 + e);
            } else {
                d = *reinterpret_cast<const uint16_t*>(b);
                u[0] = *reinterpret_cast<const u32_a2*>(b + 2 + e);
                u[1] = WT == MLK_Q8_0 ? *reinterpret_cast<const u32_a2*>(b + 18 + e) : u[0];
            }
        }
    }
    __device__ f32x4 Values(int c, int e) const {
        const float s = HalfHw(d & 0xFFFFu);
        // Q4: the nibbles of these inputs as bytes
        uint32_t v = u[c];
        if constexpr (WT == MLK_Q4_0 || WT == MLK_Q4_1) v = (v >> (4 * c)) & 0x0F0F0F0Fu;
        if constexpr (WT == kWPlanarQ4) v = ((v >> e % 8) & 0x0F0F0F0Fu) ^ 0x08080808u;
        f32x4 o;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t q = v >> (8 * i) & 0xFFu;
            if constexpr (WT == MLK_Q4_1) {
                o[i] = __fadd_rn(__fmul_rn(s, static_cast<float>(q)), HalfHw(d >> 16));
            } else {
                o[i] = s * static_cast<float>(WT == MLK_Q8_0 || WT == kWPlanarQ8
                                                  ? static_cast<int>(static_cast<int8_t>(q))
                                                  : static_cast<int>(q) - 8);
            }
        }
        return o;
    }
};
template <>
struct Raw8<kWF32> {
    f32x4 u[2];
    __device__ void Load(const uint8_t* w, int64_t, int64_t, int64_t row_bytes, int64_t o,
                         int64_t kb, int e) {
        const float* p = reinterpret_cast<const float*>(w + o * row_bytes) + kb * 32 + e;
        u[0] = *reinterpret_cast<const f32x4*>(p);
        u[1] = *reinterpret_cast<const f32x4*>(p + 16);
    }
    __device__ f32x4 Values(int c, int) const { return u[c]; }
};

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
__device__ inline float RowMax(float v) {
#pragma unroll
    for (int m = 1; m < N; m *= 2) v = fmaxf(v, __shfl_xor(v, m, kWave));
    return v;
}
template <int N>
__device__ inline uint32_t RowMin(uint32_t v) {
#pragma unroll
    for (int m = 1; m < N; m *= 2) {
        v = min(v, static_cast<uint32_t>(__shfl_xor(static_cast<int>(v), m, kWave)));
    }
    return v;
}

__device__ inline f32x4 Mfma(h8 a, h8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// Over the wave, in every lane.
__device__ inline float WaveSum(float v) {
#define MLK_DPP_ADD(ctrl, rows)                                                             \
    v += __uint_as_float(static_cast<uint32_t>(__builtin_amdgcn_update_dpp(                 \
        0, static_cast<int>(__float_as_uint(v)), ctrl, rows, 0xF, false)))
    MLK_DPP_ADD(0xB1, 0xF);   // quad_perm 1 0 3 2
    MLK_DPP_ADD(0x4E, 0xF);   // quad_perm 2 3 0 1
    MLK_DPP_ADD(0x141, 0xF);  // row_half_mirror
    MLK_DPP_ADD(0x140, 0xF);  // row_mirror
    MLK_DPP_ADD(0x142, 0xA);  // row_bcast15 into rows 1, 3
    MLK_DPP_ADD(0x143, 0xC);  // row_bcast31 into rows 2, 3
#undef MLK_DPP_ADD
    return __uint_as_float(static_cast<uint32_t>(
        __builtin_amdgcn_readlane(static_cast<int>(__float_as_uint(v)), 63)));
}

// The outputs n .. n + N - 1 of one marked row as fp32 products and sums: the
// wave's lanes take consecutive blocks (their inputs in registers), every
// output's sum is reduced over them and kept by one lane.
template <int WT, int EPI, int N>
__device__ inline void MarkedRow(const TileArgs& a, const TileSeg& g, int64_t row, int64_t n,
                                 int64_t s0, int64_t s1, float* out, int64_t ldo, bool bias) {
    constexpr int kMat = EPI == kSwiGlu ? 2 : 1;
    const int lane = threadIdx.x & (kWave - 1);
    float sum[kMat] = {};
    for (int64_t z = s0; z < s1; z += kWave) {
        // codes: the lane's block; fp32: its 4 inputs of every 256
        const int64_t kb = z + lane < s1 ? z + lane : s1 - 1;
        const auto at = [&](int i) {
            if constexpr (WT != kWF32) return kb * kBK + 4 * i;
            const int64_t k = z * kBK + 4 * kWave * i + 4 * lane;
            return k < s1 * kBK ? k : s1 * kBK - 4;
        };
        const auto in = [&](int i) {
            return WT == kWF32 ? z * kBK + 4 * kWave * i + 4 * lane < s1 * kBK : z + lane < s1;
        };
        f32x4 x[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            x[i] = *reinterpret_cast<const f32x4*>(a.x + row * a.K + at(i));
        }
        // G outputs' weights are loaded while the G before them are summed
        constexpr int G = WT == kWF32 ? 1 : 4;
        using LaneW = typename std::conditional<WT == kWF32, f32x4[8], Raw8<WT>[4]>::type;
#pragma unroll
        for (int p = 0; p < kMat; ++p) {
            const uint8_t* const w = p == 0 ? g.w : a.seg[1].w;
            LaneW lw[2][G];
            const auto load = [&](int c0, LaneW (&l)[G]) {
#pragma unroll
                for (int c = 0; c < G; ++c) {
                    const int64_t o = n + (c0 + c < N ? c0 + c : N - 1);
                    const int64_t oc = o < g.rows ? o : g.rows - 1;
                    if constexpr (WT == kWF32) {
#pragma unroll
                        for (int i = 0; i < 8; ++i) {
                            l[c][i] =
                                *reinterpret_cast<const f32x4*>(w + oc * a.row_bytes + at(i) * 4);
                        }
                    } else {
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            l[c][q].Load(w, g.rows, a.K, a.row_bytes, oc, kb, 4 * q);
                        }
                    }
                }
            };
            const auto dot = [&](int c0, const LaneW (&l)[G]) {
#pragma unroll
                for (int c = 0; c < G; ++c) {
                    float part = 0.0f;
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        f32x4 v;
                        if constexpr (WT == kWF32) {
                            v = l[c][i];
                        } else {
                            v = l[c][i % 4].Values(i / 4, 4 * (i % 4));
                        }
                        float t = 0.0f;
#pragma unroll
                        for (int e = 0; e < 4; ++e) t = fmaf(x[i][e], v[e], t);
                        part += in(i) ? t : 0.0f;
                    }
                    part = WaveSum(part);
                    if (lane == c0 + c) sum[p] += part;
                }
            };
            load(0, lw[0]);
            for (int c = 0; c < N; c += 2 * G) {
                load(c + G, lw[1]);
                dot(c, lw[0]);
                load(c + 2 * G, lw[0]);
                dot(c + G, lw[1]);
            }
        }
    }
    const int64_t col = n + lane;
    if (lane >= N || col >= g.rows) return;
    const float b0 = bias && g.bias != nullptr ? g.bias[col] : 0.0f;
    float* const o = out + row * ldo + col;
    if constexpr (kMat == 2) {
        const float* const b1 = a.seg[1].bias;
        *o = SwiGluF(sum[0] + b0, sum[1] + (b1 != nullptr ? b1[col] : 0.0f));
    } else {
        *o = EPI == kAdd ? *o + (sum[0] + b0) : sum[0] + b0;
    }
}

// The marked outputs of a wave's rows m .. m + 16 MI - 1 (bit r of `rows`) and
// outputs n .. n + 16 NB - 1 (bit c of `cols`: the output of every row) as
// fp32 products and sums over blocks s0 .. s1 - 1, the operands straight from
// memory, two blocks' loads at a time.  MFMA step st of 16 inputs from k on
// multiplies inputs k + 4 kq + st.
template <int WT, int EPI, int MI, int NB>
__device__ inline void MarkedOutputs(const TileArgs& a, const TileSeg& g, uint64_t rows,
                                     uint64_t cols, int64_t m, int64_t n, int64_t s0, int64_t s1,
                                     float* out, int64_t ldo, bool bias) {
    constexpr int kMat = EPI == kSwiGlu ? 2 : 1;
    const int i16 = threadIdx.x & 15, kq = (threadIdx.x >> 4) & 3;
    const float* xp[MI];
    bool take[MI];
    f32x4 e[MI][kMat][NB];
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        take[i] = cols != 0 || ((rows >> (16 * i)) & 0xFFFFu) != 0;
        const int64_t row = m + 16 * i + i16;
        xp[i] = a.x + (row < a.T ? row : a.T - 1) * a.K + 4 * kq;
#pragma unroll
        for (int p = 0; p < kMat; ++p) {
#pragma unroll
            for (int j = 0; j < NB; ++j) e[i][p][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    if (rows == 0 && cols == 0) return;
    for (int64_t z = s0; z < s1; z += 2) {
        Raw8<WT> w[2][kMat][NB];
        f32x4 x[2][MI][2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int64_t kb = z + b < s1 ? z + b : z;
#pragma unroll
            for (int p = 0; p < kMat; ++p) {
#pragma unroll
                for (int j = 0; j < NB; ++j) {
                    const int64_t col = n + 16 * j + i16;
                    w[b][p][j].Load(p == 0 ? g.w : a.seg[1].w, g.rows, a.K, a.row_bytes,
                                    col < g.rows ? col : g.rows - 1, kb, 4 * kq);
                }
            }
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                if (!take[i]) continue;
                x[b][i][0] = *reinterpret_cast<const f32x4*>(xp[i] + kb * kBK);
                x[b][i][1] = *reinterpret_cast<const f32x4*>(xp[i] + kb * kBK + 16);
            }
        }
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            if (z + b >= s1) continue;
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                f32x4 wv[kMat][NB];
#pragma unroll
                for (int p = 0; p < kMat; ++p) {
#pragma unroll
                    for (int j = 0; j < NB; ++j) wv[p][j] = w[b][p][j].Values(c, 4 * kq);
                }
#pragma unroll
                for (int i = 0; i < MI; ++i) {
                    if (!take[i]) continue;
#pragma unroll
                    for (int p = 0; p < kMat; ++p) {
#pragma unroll
                        for (int j = 0; j < NB; ++j) {
#pragma unroll
                            for (int st = 0; st < 4; ++st) {
                                e[i][p][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                                    x[b][i][c][st], wv[p][j][st], e[i][p][j], 0, 0, 0);
                            }
                        }
                    }
                }
            }
        }
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const int64_t col = n + 16 * j + i16;
        if (col >= g.rows) continue;
        const bool cb = (cols >> (16 * j + i16)) & 1;
        const float b0 = bias && g.bias != nullptr ? g.bias[col] : 0.0f;
        const float b1 = kMat == 2 && a.seg[1].bias != nullptr ? a.seg[1].bias[col] : 0.0f;
#pragma unroll
        for (int i = 0; i < MI; ++i) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t row = m + 16 * i + 4 * kq + r;
                if (row >= a.T || !(cb || (rows >> (16 * i + 4 * kq + r) & 1))) continue;
                float* const o = out + row * ldo + col;
                if constexpr (EPI == kSwiGlu) {
                    *o = SwiGluF(e[i][0][j][r] + b0, e[i][kMat - 1][j][r] + b1);
                } else {
                    *o = EPI == kAdd ? *o + (e[i][0][j][r] + b0) : e[i][0][j][r] + b0;
                }
            }
        }
    }
}

// Waves a SIMD that a workgroup's registers leave room for: three for the 64 x
// 128 tiles of fp32 and Q4_1 weights, whose LDS fits a CU three times (F32, 64
// rows of w_gate: 69.5 us with two, 66.3 with three; the 32 x 64 tiles, 8
// rows: 50 us, 55 with their registers held to three).
template <int WT, int BM>
constexpr int kTileWaves = !kCodes<WT> && BM == 64 ? 3 : 2;

template <int WT, int MI, int NJ, int WM, int WN, int EPI, int KB>
__global__ __launch_bounds__(64 * WM * WN,
                             (kTileWaves<WT, 16 * MI * WM>)) void GemmTile(TileArgs a) {
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
    __shared__ uint32_t wlow;  // values: the weight rows' smallest scaled magnitude
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
    // the rows' scales, from their first 64 inputs: the thread's part of the
    // two stages in registers
    PieceScale xs[kXN], wsc[kWN];
    float xmost[kXN], wmost[kWN];
    uint32_t xleast[kXN], wleast[kWN];  // LeastKeys
    us2 wkeys = {0xFFFF, 0xFFFF};       // Q4_1
    const auto first_x = [&](int i) {
        return RowMax<4>(AbsMax8(xv[1][i], AbsMax8(xv[0][i], 0.0f)));
    };
    const auto first_w = [&](int i) {
        if constexpr (WT == kWF32) {
            return RowMax<4>(AbsMax8(wr[1].v[i], AbsMax8(wr[0].v[i], 0.0f)));
        } else if constexpr (WT == MLK_Q4_1) {
            return fmaxf(BlockMost(wr[0]), BlockMost(wr[1]));
        } else {
            return 1.0f;
        }
    };
    bool none = false;
#pragma unroll
    for (int i = 0; i < kXN; ++i) {
        xmost[i] = first_x(i);
        none |= xmost[i] == 0.0f;
    }
#pragma unroll
    for (int i = 0; i < kWN; ++i) {
        wmost[i] = first_w(i);
        none |= wmost[i] == 0.0f;
    }
    if (__any(none)) {  // rows that begin with zeros: 64 inputs at 7 places further on
        for (int k = 1; k < 8 && __any(none); ++k) {
            const int64_t z = s0 + (s1 - s0) * k / 8;
            load(0, z);
            load(1, z + 1 < s1 ? z + 1 : z);
            none = false;
#pragma unroll
            for (int i = 0; i < kXN; ++i) {
                const float m = first_x(i);
                if (xmost[i] == 0.0f) xmost[i] = m;
                none |= xmost[i] == 0.0f;
            }
#pragma unroll
            for (int i = 0; i < kWN; ++i) {
                const float m = first_w(i);
                if (wmost[i] == 0.0f) wmost[i] = m;
                none |= wmost[i] == 0.0f;
            }
        }
        load(0, s0);
        load(1, s0 + 1 < s1 ? s0 + 1 : s0);
    }
#pragma unroll
    for (int i = 0; i < kXN; ++i) {
        xs[i] = PieceScale(xmost[i], 7);
        xmost[i] = 0.0f;
        xleast[i] = kNoKey;
    }
#pragma unroll
    for (int i = 0; i < kWN; ++i) {
        wsc[i] = PieceScale(wmost[i], 10);
        wmost[i] = 0.0f;
        wleast[i] = kNoKey;
    }

    // LDS offsets of the thread's writes and operand reads; rows a multiple of
    // 8 apart have the same swizzle, so the others lie constants away
    const int xw = At(tid >> 2, tid & 3);
    const int ww = WT == kWF32 ? xw : At(tid >> 1, 2 * h), ww1 = At(tid >> 1, 2 * h + 1);
    const int xr = wm * 256 * MI + At(i16, kq), wrd = wn * 256 * NJ + At(i16, kq);

    // a stage's registers b into LDS buffer buf
    auto store = [&](int buf, int b) {
        u32x4 p0, p1;
#pragma unroll
        for (int i = 0; i < kXN; ++i) {
            Split8(xv[b][i], xs[i].s, &p0, &p1);
            xmost[i] = AbsMax8(xv[b][i], xmost[i]);
            xleast[i] = LeastKey8(xv[b][i], xleast[i]);
            const int at = xw + kThreads * 4 * i;
            *reinterpret_cast<u32x4*>(&sm.x[buf][0][at]) = p0;
            *reinterpret_cast<u32x4*>(&sm.x[buf][1][at]) = p1;
        }
        if constexpr (kCodes<WT>) {
            u32x4 c[2];
            Codes16<WT>(wr[b], h, c);
            *reinterpret_cast<u32x4*>(&sm.w[buf][0][ww]) = c[0];
            *reinterpret_cast<u32x4*>(&sm.w[buf][0][ww1]) = c[1];
            sm.d[buf][tid >> 1] = HalfHw(wr[b].d & 0xFFFFu);
        } else {
            float4 q[2][2];
            if constexpr (WT == MLK_Q4_1) {
                Values16(wr[b], h, q);
                wmost[0] = fmaxf(wmost[0], BlockMost(wr[b]));
                wkeys = __builtin_elementwise_min(wkeys, BlockKeys(wr[b]));
            }
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int k = WT == kWF32 ? i : 0;
                if constexpr (WT == kWF32) {
                    q[i][0] = wr[b].v[i][0];
                    q[i][1] = wr[b].v[i][1];
                }
                Split8(q[i], wsc[k].s, &p0, &p1);
                if constexpr (WT == kWF32) {
                    wmost[i] = AbsMax8(q[i], wmost[i]);
                    wleast[i] = LeastKey8(q[i], wleast[i]);
                }
                const int at = WT == kWF32 ? ww + BN * 8 * i : (i == 0 ? ww : ww1);
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
        h8 bl[KB][NJ];  // codes for the second pieces, times 2^-11
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
                    b[k][p][j] = *reinterpret_cast<const h8*>(&sm.w[buf][p][wrd + 256 * j]);
                }
                if constexpr (kCodes<WT>) {
                    bl[k][j] = b[k][0][j] * static_cast<_Float16>(1.0f / kLowUp);
                    dj[k][j] = sm.d[buf][row];
                }
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
            const int at = xr + 256 * i;
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
                        S[k][j] = Mfma(lo[k], bl[k][j], f32x4{0.f, 0.f, 0.f, 0.f});
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
                f32x4 S[NJ];  // the products with a second piece, times 2^11
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    S[j] = Mfma(lo[0], b[0][0][j], f32x4{0.f, 0.f, 0.f, 0.f});
                }
#pragma unroll
                for (int j = 0; j < NJ; ++j) S[j] = Mfma(hi[0], b[0][kPl - 1][j], S[j]);
#pragma unroll
                for (int j = 0; j < NJ; ++j) acc[i][j] = Mfma(hi[0], b[0][0][j], acc[i][j]);
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        acc[i][j][r] = fmaf(S[j][r], 1.0f / kLowUp, acc[i][j][r]);
                    }
                }
            }
        }
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (!kCodes<WT>) {
        if (tid == 0) wlow = 0x7F800000u;
    }
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
    // pieces' range (head comment)
    const float low_min = 1.0f / ((kCodes<WT> ? 2048.0f : 1024.0f) * static_cast<float>(a.K));
    const float low_pair = 1.0f / (33554432.0f * static_cast<float>(a.K));
    bool bad = false;
    float low = INFINITY;  // values: the smallest scaled weight of the tile
    if constexpr (!kCodes<WT>) {
#pragma unroll
        for (int i = 0; i < kWN; ++i) {
            const float most = WT == kWF32 ? RowMax<4>(wmost[i]) : wmost[i];
            const float least =
                WT == kWF32 ? KeyValue(RowMin<4>(wleast[i])) : KeySpacing(wkeys);
            const bool fits = wsc[i].Fits(most, least, low_min);
            cinv[WT == kWF32 ? (tid >> 2) + BN / 2 * i : tid >> 1] = fits ? wsc[i].inv : 0.0f;
            bad |= !fits;
            if (fits) low = fminf(low, least * wsc[i].s);
        }
        atomicMin(&wlow, __float_as_uint(low));
        __syncthreads();
        low = __uint_as_float(wlow);
    }
#pragma unroll
    for (int i = 0; i < kXN; ++i) {
        const float least = KeyValue(RowMin<4>(xleast[i]));
        bool fits = xs[i].Fits(RowMax<4>(xmost[i]), least, low_min);
        if constexpr (!kCodes<WT>) fits = fits && !(least * xs[i].s * low < low_pair);
        rinv[(tid >> 2) + kThreads / 4 * i] = fits ? xs[i].inv : 0.0f;
        bad |= !fits;
    }
    const bool any_bad = __syncthreads_or(bad) != 0;

    const bool part = a.partial != nullptr;
    const int64_t ldo = part ? a.cols : O;
    float* const out = part ? a.partial + sp * a.T * a.cols + g.col0 : (kDual ? a.seg[1].y : g.y);
    const auto factors = [&](int i) {
        return *reinterpret_cast<const f32x4*>(&rinv[wm * 16 * MI + 16 * i + 4 * kq]);
    };
    const auto value = [&](int i, int j, int r, float ri) {
        if constexpr (kCodes<WT>) {
            return acc[i][j][r] * ri;
        } else {
            return acc[i][j][r] * (ri * cinv[wn * 16 * NJ + 16 * j + i16]);
        }
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
    if (__builtin_expect(any_bad, 0)) {
        // up to 8 marked rows one by one, each wave a part of the outputs;
        // more, and marked outputs, by the matrix cores, each wave its rows
        // and, of the tile's outputs, 1 / WN
        constexpr int NB = kDual ? NJ / 2 : NJ;
        const auto marked = [](const float* f, int n, int l) {
            return __ballot(l < n && f[l < n ? l : 0] == 0.0f);
        };
        uint64_t all_rows[WM];
        int n_rows = 0;
#pragma unroll
        for (int i = 0; i < WM; ++i) {
            const int64_t left = a.T - m0 - 16 * MI * i;  // (rows past T are copies of the last)
            all_rows[i] = marked(rinv + 16 * MI * i,
                                 left < 16 * MI ? static_cast<int>(left) : 16 * MI, lane);
            n_rows += __popcll(all_rows[i]);
        }
        bool any_col = false;
        uint64_t cols = 0;
        if constexpr (!kCodes<WT>) {
            for (int i = 0; i < BN; i += kWave) any_col |= marked(cinv + i, kWave, lane) != 0;
            const float* const f = cinv + wn * 16 * NB;
            cols = marked(f, 16 * NB, lane);
            if (kDual) cols |= marked(f + BN / 2, 16 * NB, lane);
        }
        if (n_rows <= 8 && !any_col) {
            constexpr int N = (kDual ? BN / 2 : BN) / (WM * WN);
#pragma unroll
            for (int i = 0; i < WM; ++i) {
                for (uint64_t b = all_rows[i]; b != 0; b &= b - 1) {
                    const int64_t row = m0 + 16 * MI * i + __builtin_ctzll(b);
                    MarkedRow<WT, EPI, N>(a, g, row, n0 + wave * N, s0, s1, out, ldo, !part);
                }
            }
        } else {
            MarkedOutputs<WT, EPI, MI, NB>(a, g, all_rows[wm], cols, m0 + wm * 16 * MI,
                                           n0 + wn * 16 * NB, s0, s1, out, ldo, !part);
        }
    }
}

// ------------------------------------------------------------ launches
// Tile shape and K splits of a launch.
//   128 x 256 (one workgroup a CU) for more than 64 rows, where up to 8
//       splits (more while each keeps 16 stages) give 3/4 of a workgroup a
//       CU; past that K is not split: T = 389 over 14336 outputs (224 tiles,
//       Q8_0) takes 160 us unsplit, 17% more in two splits of 1.75 rounds.
//   32 x 64 up to 32 rows, split to 4 workgroups a CU (33 KB of LDS each),
//       each split at least 8 stages.  16 rows of F32: w_gate 50.6 us (fp32
//       MFMA 51.2); 32 rows of Q8_0 / Q4_0: w_gate 41.7 / 40.5 us (skinny
//       kernel, fp32 MFMA, 49.5 / 48.4), 128256 outputs 273 / 222 (350 / 360,
//       whose 8 splits' partial sums alone are 131 MB).  On 64 x 128 tiles
//       those took as long or longer.
//   64 x 128 otherwise, split to 1.5 workgroups a CU, each split at least 8
//       stages.  Q8_0: T = 64 over 4096 x 14336 43 us in 16 splits (512
//       workgroups), 16% more in 8; 128 rows over 4096 x 4096 31 us against
//       34-37 on 128 x 256, over 14336 x 4096 61 there against 70.
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
    return (wt == MLK_Q8_0 || wt == MLK_Q4_0) && T > 16 &&
           n >= (fused ? kLayerGroupMin : kFewRowsMin);
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
