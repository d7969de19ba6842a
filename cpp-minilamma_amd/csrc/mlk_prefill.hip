// mlk_prefill.hip -- causal attention of a prompt chunk on the matrix cores.
//
// Tokens t < T sit at positions pos0 + t; token t's head h attends to cache
// positions 0 .. pos0 + t of its KV head g = h / (H / KV) (the reference's
// ForwardAttention per token, src/forward.cc:265-298, with the chunk's own
// K/V rows already written to the cache):
//   s_j = (q . k_j) * (1 / sqrt(hd)),  p = softmax(s),  out = sum_j p_j v_j
// in fp32.  The dot products and the weighted sum run on
// v_mfma_f32_16x16x4_f32, so their fp32 summation order differs from the
// reference's serial loops; the result is held to the same float64 error
// bound as the decode kernel's (every order of the fp32 sums meets it).
//
// Work layout: a workgroup of 4 waves owns 16 consecutive tokens and 4 query
// heads of one KV head (wave w: head 4 * head_block + w of the group), so
// the 4 waves share each K/V tile.  Workgroups run in reverse token order,
// the longest prefixes first.  Per tile of 32 cache positions (staged
// through two LDS buffers, rows hd + 4 floats apart; the next tile's global
// loads are issued before the current tile's MFMAs):
//   - S^T = K Q^T (16 positions x 16 queries per instruction block): K rows
//     come from LDS, each lane's q row (query l % 16, dims 16c + 4(l / 16)
//     .. + 3) lives in registers for the whole kernel.  S^T rather than S,
//     because the MFMA output layout of S^T (lane l, register r: position
//     4(l / 16) + r, query l % 16) is exactly the B-operand layout of
//     O^T = V^T P^T, so p never goes through LDS or a transpose.
//   - Online softmax per query: the running max needs 2 cross-lane
//     shuffles per tile (the 4 lane groups of a query); the running sum
//     stays per lane and is reduced once at the end.
//   - O^T += V^T P^T: V read from LDS one float per lane and step (16
//     consecutive dims per 16 lanes), 32 accumulators per lane at hd = 128.
// Positions past the workgroup's last token are clamped on load and masked
// (-inf score) per query.  A wave whose head is past its group (head counts
// per KV head that are not a multiple of 4) computes on head 0's query and
// stores nothing: no branch around the loop body.  FLOPs: 4 * hd * H * sum_t (pos0 + t + 1).
//
// fp16 products (kF16: every launch at head_dim 128; head_dim 64 keeps the
// fp32 instruction above): K, V, q and p are each scaled by a power of two and
// split into two fp16 pieces, the value rounded to fp16 and the rest rounded
// to fp16 (together within one unit of its last of 23 bits; for values far
// below their tile's largest, within 2^-39 of that).  The scale comes from the
// largest finite magnitude of a K tile, of a V tile (32 positions x 128 dims)
// and of a q row, which it brings into [2^14, 2^15); p, at most 1, is scaled by
// 2^14 and by the V tile's factor relative to the largest so far, so the
// accumulators keep one unit.  Each product is lo hi + hi lo + hi hi, three
// v_mfma_f32_16x16x32_f16 (32 dims or the tile's 32 positions each); lo lo,
// below 2^-22, is left out.  Six bf16 piece products (three pieces a value)
// took twice the matrix work and half as much LDS again: Llama-3-8B heads,
// 4096 tokens from position 0, 721 us before, 484 with these (284 TFLOP/s of
// q.k and p.v), error against float64 1.6e-7 before, 1.2e-7 after; 64 decode
// tokens over 1000 positions 66 -> 62 us.  Scores stay within
// the gamma_{hd+1} bound with the fp32 sums; values add at most 16 u of
// sum_j p_j |v_jd| to the sums' (n + 6) u.
// Tile buffers of 37.9 KB: two when the grid has at most one workgroup per
// compute unit; otherwise one, with a barrier before each restage, so several
// workgroups share a unit and one's softmax and staging overlap the others'
// matrix work.  The value MFMA's k index is the lane's own 8 probabilities:
// slot 8 kq + j is position 16 (j / 4) + 4 kq + j % 4 of the tile, the order
// V^T is staged in.
#include "mlk_attention.h"

#include <cmath>
#include <type_traits>

namespace mlk {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kPfThreads = 256;
constexpr int kPfTokens = 16;  // tokens per workgroup: the MFMA's 16 query columns
constexpr int kPfTile = 32;    // cache positions per K/V tile
constexpr int kPfHeads = 4;    // query heads per workgroup, one per wave

template <int HD>
struct __align__(16) PrefillSmem {
    float k[2][kPfTile * (HD + 4)];
    float v[2][kPfTile * (HD + 4)];
};

// The next K and V tiles in registers: thread tid holds float4 tid + 256 i
// of the [32][HD] tiles (positions past max_pos read max_pos's row).  The
// registers are native 4-vectors: with HIP's float4 struct, each copy is an
// aggregate memcpy, and the optimizer fuses load and LDS store into one
// global-to-LDS copy at the store, so the prefetch would not happen.
template <int HD>
struct KvTile {
    static constexpr int NL = kPfTile * HD / 4 / kPfThreads;
    f32x4 k[NL], v[NL];  // vectors, not float4 structs (see Load)
    const float* kb;
    const float* vb;
    int64_t slot, max_pos;
    __device__ void Load(int64_t p0) {
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int idx = static_cast<int>(threadIdx.x) + kPfThreads * i;
            const int64_t p = p0 + idx / (HD / 4);
            const int64_t pos = p <= max_pos ? p : max_pos;
            const int c4 = idx % (HD / 4);
            k[i] = *reinterpret_cast<const f32x4*>(kb + pos * slot + 4 * c4);
            v[i] = *reinterpret_cast<const f32x4*>(vb + pos * slot + 4 * c4);
        }
    }
    __device__ void Store(float* ks, float* vs) const {
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int idx = static_cast<int>(threadIdx.x) + kPfThreads * i;
            const int o = (idx / (HD / 4)) * (HD + 4) + 4 * (idx % (HD / 4));
            *reinterpret_cast<f32x4*>(ks + o) = k[i];
            *reinterpret_cast<f32x4*>(vs + o) = v[i];
        }
    }
};

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
constexpr int kPad = 8;             // fp16 padding per K plane row (rows 16 bytes apart in bank terms)
constexpr int kVLd = kPfTile + 8;   // V^T plane row: 32 slots + 8 padding

// K planes [piece][32 positions][HD + 8] and V^T planes [piece][HD][40] of
// a tile, fp16, and the waves' largest K and V magnitudes of the next tile.
template <int HD, int NBUF>
struct __align__(16) PrefillSmemF16 {
    uint16_t k[NBUF][2 * kPfTile * (HD + kPad)];
    uint16_t v[NBUF][2 * HD * kVLd];
    uint32_t most[2][4];
};

// 4 floats times s as two fp16 pieces, 4 per dword pair (low half first).
__device__ inline void Split4(f32x4 x, float s, uint2 (&o)[2]) {
    h2 hi[2], lo[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const float a = x[2 * i], b = x[2 * i + 1];
        hi[i].x = static_cast<_Float16>(a * s);
        hi[i].y = static_cast<_Float16>(b * s);
        lo[i].x = static_cast<_Float16>(fmaf(a, s, -static_cast<float>(hi[i].x)));
        lo[i].y = static_cast<_Float16>(fmaf(b, s, -static_cast<float>(hi[i].y)));
    }
    o[0] = make_uint2(__builtin_bit_cast(uint32_t, hi[0]), __builtin_bit_cast(uint32_t, hi[1]));
    o[1] = make_uint2(__builtin_bit_cast(uint32_t, lo[0]), __builtin_bit_cast(uint32_t, lo[1]));
}

// 8 floats times s as the pieces' operands.
__device__ inline void Split8(f32x4 a, f32x4 b, float s, h8 (&o)[2]) {
    uint2 pa[2], pb[2];
    Split4(a, s, pa);
    Split4(b, s, pb);
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        o[p] = __builtin_bit_cast(h8, make_uint4(pa[p].x, pa[p].y, pb[p].x, pb[p].y));
    }
}

// Magnitudes as unsigned keys: twice the bits plus 2^24, which wraps for
// infinities and NaNs to below every finite value's key, so the largest key
// is the largest finite magnitude's.
__device__ inline uint32_t MagKey(float x) { return (__float_as_uint(x) << 1) + 0x01000000u; }

template <int N>
__device__ inline uint32_t MagKeys(const f32x4 (&x)[N]) {
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < N; ++i) {
#pragma unroll
        for (int e = 0; e < 4; ++e) m = max(m, MagKey(x[i][e]));
    }
    return m;
}

// Largest over the wave, in every lane (uniform).
__device__ inline uint32_t WaveMaxU32(uint32_t v) {
#define MLK_DPP_MAX(ctrl, rows)                                                              \
    v = max(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(                            \
                   static_cast<int>(v), static_cast<int>(v), ctrl, rows, 0xF, false)))
    MLK_DPP_MAX(0xB1, 0xF);   // quad_perm 1 0 3 2
    MLK_DPP_MAX(0x4E, 0xF);   // quad_perm 2 3 0 1
    MLK_DPP_MAX(0x141, 0xF);  // row_half_mirror
    MLK_DPP_MAX(0x140, 0xF);  // row_mirror
    MLK_DPP_MAX(0x142, 0xA);  // row_bcast15 into rows 1, 3
    MLK_DPP_MAX(0x143, 0xC);  // row_bcast31 into rows 2, 3
#undef MLK_DPP_MAX
    return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), 63));
}

// The power of two that brings the key's magnitude into [2^14, 2^15) (at
// most 2^126), and its inverse.
struct MagScale {
    int fe;  // the inverse's exponent field, 1 .. 240
    float s, f;
    __device__ explicit MagScale(uint32_t key) {
        const int e = static_cast<int>(key >> 24) - 1;  // the exponent field, -1 .. 254
        const int b = 268 - e < 253 ? 268 - e : 253;
        fe = 254 - b;
        s = __uint_as_float(static_cast<uint32_t>(b) << 23);
        f = __uint_as_float(static_cast<uint32_t>(fe) << 23);
    }
};

// 2^(e - 127), 0 below the smallest normal.
__device__ inline float Pow2Field(int e) {
    return __uint_as_float(static_cast<uint32_t>(e > 0 ? e : 0) << 23);
}

// The next tile for the fp16 kernel: thread tid holds one 4 x 4 block of K
// and one of V, at positions 4 a .. 4 a + 3 and dims 4 c4 .. 4 c4 + 3
// (head_dim 128).  K takes a = tid / 32, c4 = tid % 32 (a 16-lane group
// writes 128 contiguous bytes of a plane row); V takes a = tid % 8, c4 =
// tid / 8, so a group's V^T writes (8 position groups x 2 dim rows, 80 bytes
// apart) meet each LDS bank once.  Positions past load_pos read its row.
struct KvBlock {
    f32x4 k[4], v[4];
    const float* kb;
    const float* vb;
    int64_t slot, load_pos;
    __device__ void Load(int64_t p0) {
        const int tid = static_cast<int>(threadIdx.x);
        const int ak = tid / 32, ck = tid % 32, av = tid % 8, cv = tid / 8;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int64_t p = p0 + 4 * ak + r;
            const int64_t pos = p <= load_pos ? p : load_pos;
            k[r] = *reinterpret_cast<const f32x4*>(kb + pos * slot + 4 * ck);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int64_t p = p0 + 4 * av + r;
            const int64_t pos = p <= load_pos ? p : load_pos;
            v[r] = *reinterpret_cast<const f32x4*>(vb + pos * slot + 4 * cv);
        }
    }
    // V at positions past mp (within the tile) is zero: their probabilities
    // are 0, whatever a later token's V holds
    __device__ void DropV(int64_t mp) {
        const int av = static_cast<int>(threadIdx.x) % 8;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (4 * av + r > mp) v[r] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    // K rows 4 a + r; V^T rows 4 c4 + e at slots s0 .. s0 + 3, where
    // positions 4 a .. 4 a + 3 sit (slot 8 kq + j: position 16 (j / 4) +
    // 4 kq + j % 4)
    // KL / VLD: the K and V^T plane row strides (the LDS layout's, or the
    // unpadded images of KvPieces)
    template <int KL = 128 + kPad, int VLD = kVLd>
    __device__ void Store(uint16_t* ks, uint16_t* vs, float k_scale, float v_scale) const {
        constexpr int HD = 128;
        const int tid = static_cast<int>(threadIdx.x);
        const int a = tid / 32, c4 = tid % 32, av = tid % 8, cv = tid / 8;
        const int s0 = av < 4 ? 8 * av : 8 * (av - 4) + 4;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            uint2 pc[2];
            Split4(k[r], k_scale, pc);
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                *reinterpret_cast<uint2*>(ks + (p * kPfTile + 4 * a + r) * KL + 4 * c4) = pc[p];
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            uint2 pc[2];
            Split4(f32x4{v[0][e], v[1][e], v[2][e], v[3][e]}, v_scale, pc);
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                *reinterpret_cast<uint2*>(vs + (p * HD + 4 * cv + e) * VLD + s0) = pc[p];
            }
        }
    }
};

// The tile's largest K and V keys: each wave's into most[][wave], and after a
// barrier the largest of the four.
__device__ inline void PutMost(uint32_t (&most)[2][4], const KvBlock& t) {
    const uint32_t k = WaveMaxU32(MagKeys(t.k)), v = WaveMaxU32(MagKeys(t.v));
    if (threadIdx.x % kWave == 0) {
        most[0][threadIdx.x / kWave] = k;
        most[1][threadIdx.x / kWave] = v;
    }
}
__device__ inline uint32_t GetMost(const uint32_t (&most)[4]) {
    const uint4 m = *reinterpret_cast<const uint4*>(most);
    return __builtin_amdgcn_readfirstlane(max(max(m.x, m.y), max(m.z, m.w)));
}

// Pre-split tiles (head_dim 128): per KV head g and tile t of 32 cache
// positions, the K planes [2][32][128] and the V^T planes [2][128][32] in
// fp16, exactly what KvBlock::Store writes to LDS, without the row padding:
// one 32 KB image a tile, images of head g at g * n_tiles + t, then the
// tiles' largest K and V keys (uint2 each, in the same order).  A prompt
// chunk's workgroups each stage every tile of their prefix, so the split
// (most of the VALU work of a tile) is done once here instead of once per 16
// tokens.
constexpr int kPieceHalves = 2 * kPfTile * 128;          // fp16 of a K (or V^T) image
constexpr int kPieceTileU4 = 2 * kPieceHalves * 2 / 16;  // uint4 of a tile's two images

__global__ __launch_bounds__(kPfThreads) void KvPieces(const float* __restrict__ kc,
                                                       const float* __restrict__ vc,
                                                       int64_t slot, int KV, int64_t max_pos,
                                                       int64_t n_tiles,
                                                       uint16_t* __restrict__ images,
                                                       uint2* __restrict__ keys) {
    __shared__ __align__(16) uint32_t most[2][4];
    const int64_t t = blockIdx.x / KV;
    const int g = static_cast<int>(blockIdx.x % KV);
    KvBlock tile;
    tile.kb = kc + static_cast<int64_t>(g) * 128;
    tile.vb = vc + static_cast<int64_t>(g) * 128;
    tile.slot = slot;
    tile.load_pos = max_pos;  // positions past it read its row
    tile.Load(t * kPfTile);
    PutMost(most, tile);
    __syncthreads();
    const uint32_t kk = GetMost(most[0]), kv = GetMost(most[1]);
    const int64_t at = static_cast<int64_t>(g) * n_tiles + t;
    uint16_t* ks = images + at * (2 * kPieceHalves);
    tile.Store<128, kPfTile>(ks, ks + kPieceHalves, MagScale(kk).s, MagScale(kv).s);
    if (threadIdx.x == 0) keys[at] = make_uint2(kk, kv);
}

// The next tile from KvPieces' images: thread tid copies uint4 tid + 256 i
// (i < 4) of the K image and of the V^T image.  K image uint4 u: piece
// u / 512, row (u / 16) % 32, dims 8 (u % 16) ..; V^T image: piece u / 512,
// dim (u / 4) % 128, slots 8 (u % 4) ...
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct KvBlockPre {
    u32x4 k[4], v[4];   // native vectors, not uint4 structs (see KvTile::Load)
    uint2 key;
    const u32x4* base;  // head g's first image
    const uint2* keys;  // and its key
    __device__ void Load(int64_t p0) {
        const u32x4* src = base + (p0 / kPfTile) * kPieceTileU4;
        const int tid = static_cast<int>(threadIdx.x);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            k[i] = src[tid + kPfThreads * i];
            v[i] = src[kPieceTileU4 / 2 + tid + kPfThreads * i];
        }
        key = keys[p0 / kPfTile];
    }
    // as KvBlock::DropV
    __device__ void DropV(int64_t mp) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            // slots 8 q4 + 2d, + 1 (dword d): positions 16 (d / 2) + 4 q4 +
            // 2 (d % 2), + 1
            const int64_t b = 4 * ((threadIdx.x + kPfThreads * i) % 4);
            const auto keep = [&](int64_t pl) {
                return (pl <= mp ? 0x0000FFFFu : 0u) | (pl + 1 <= mp ? 0xFFFF0000u : 0u);
            };
            v[i].x &= keep(b);
            v[i].y &= keep(b + 2);
            v[i].z &= keep(b + 16);
            v[i].w &= keep(b + 18);
        }
    }
    __device__ void Store(uint16_t* ks, uint16_t* vs, float, float) const {
        constexpr int KL = 128 + kPad;
        const int tid = static_cast<int>(threadIdx.x);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int u = tid + kPfThreads * i;
            *reinterpret_cast<u32x4*>(ks + ((u / 512) * kPfTile + (u / 16) % kPfTile) * KL +
                                      8 * (u % 16)) = k[i];
            *reinterpret_cast<u32x4*>(vs + ((u / 512) * 128 + (u / 4) % 128) * kVLd + 8 * (u % 4)) =
                v[i];
        }
    }
};

// kChunked (decode tokens at any positions, AttnDecodeTile below): the
// token's position comes from `positions`, and the workgroup covers one
// chunk of cache positions, writing partials for AttnCombine.
struct TileChunks {
    const int32_t* positions;  // per token, or null: pos0 + t
    int64_t max_ctx;
    int chunk, n_chunks;
    float* ws_acc;  // [T, H, n_chunks, hd]
    float* ws_ml;   // [T, H, n_chunks, 2]
    int32_t* err;
};

template <int HD, bool kChunked, bool kF16, int NBUF = 2, bool kPre = false>
__global__ __launch_bounds__(kPfThreads) void AttnPrefill(
    const float* __restrict__ q, int64_t q_stride, const float* __restrict__ kc,
    const float* __restrict__ vc, int64_t slot, int KV, int H, int32_t pos0, int64_t T,
    float scale, float* __restrict__ out, int head_blocks, TileChunks tc,
    const uint16_t* __restrict__ images, const uint2* __restrict__ image_keys,
    int64_t n_image_tiles, uint32_t* __restrict__ a_planes) {
#pragma clang fp contract(off)
    static_assert(!kF16 || HD == 128, "fp16 products: head_dim 128");
    static_assert(!kPre || kF16, "pre-split tiles: fp16 products");
    static_assert(NBUF == 2 || (NBUF == 1 && kF16), "one tile buffer: fp16 products only");
    constexpr int LD = HD + 4;
    constexpr int NC = HD / 16;                          // 16-dim chunks
    constexpr int KL = HD + kPad;                        // K plane row (fp16)
    __shared__ typename std::conditional<kF16, PrefillSmemF16<HD, NBUF>, PrefillSmem<HD>>::type sm;
    const int group = H / KV;
    const int64_t n_tb = (T + kPfTokens - 1) / kPfTokens;
    int64_t bid = blockIdx.x;
    const int hb = static_cast<int>(bid % head_blocks);
    bid /= head_blocks;
    const int g = static_cast<int>(bid % KV);
    bid /= KV;
    int ck = 0;  // the chunk (kChunked)
    if constexpr (kChunked) {
        ck = static_cast<int>(bid / n_tb);
        bid %= n_tb;
    }
    const int64_t t0 = (n_tb - 1 - bid) * kPfTokens;
    const int wave = threadIdx.x / kWave;
    const int lane = threadIdx.x % kWave;
    const int i16 = lane & 15, kq = lane >> 4;
    const int hq = hb * kPfHeads + wave;  // query head within the group
    const bool active = hq < group;
    const int h = g * group + (active ? hq : 0);
    const int64_t last_t = (t0 + kPfTokens < T ? t0 + kPfTokens : T) - 1;
    const int64_t t = t0 + i16 <= last_t ? t0 + i16 : last_t;  // this lane's query token
    int64_t my_pos = pos0 + t;
    int64_t max_pos = pos0 + last_t;
    int64_t p_begin = 0, p_end = max_pos + 1;  // cache positions of this workgroup
    bool valid = true;
    if constexpr (kChunked) {
        const int32_t pt = tc.positions != nullptr ? tc.positions[t] : pos0 + static_cast<int32_t>(t);
        valid = pt >= 0 && pt < tc.max_ctx;
        if (!valid && ck == 0 && hb == 0 && g == 0 && t0 + i16 <= last_t) RaiseFlag(tc.err, 1);
        my_pos = valid ? pt : -1;  // an invalid token attends nothing
        // the block's last position: the maximum over its 16 tokens
        int32_t mx = static_cast<int32_t>(my_pos);
#pragma unroll
        for (int o = 1; o < 16; o *= 2) mx = max(mx, __shfl_xor(mx, o, kWave));
        max_pos = mx;
        p_begin = static_cast<int64_t>(ck) * tc.chunk;
        p_end = p_begin + tc.chunk < max_pos + 1 ? p_begin + tc.chunk : max_pos + 1;
        if (p_begin >= p_end) {  // no token of the block reaches this chunk
            if (tc.n_chunks == 1 && active && t0 + i16 <= last_t) {
                // every token invalid, and no merge follows: zero rows
                float* orow = out + (t * H + h) * static_cast<int64_t>(HD) + 4 * kq;
#pragma unroll
                for (int cc = 0; cc < NC; ++cc) {
                    *reinterpret_cast<float4*>(orow + 16 * cc) = make_float4(0.f, 0.f, 0.f, 0.f);
                }
            }
            return;
        }
    }

    f32x4 qv[NC];        // fp32: dims 16 c + 4 kq .. + 3
    h8 qp[2][HD / 32];   // fp16: pieces of dims 32 c + 8 kq .. + 7
    float q_factor = 1.0f;
    if constexpr (kF16) {
        const float* qrow = q + t * q_stride + static_cast<int64_t>(h) * HD + 8 * kq;
        f32x4 qr[2 * (HD / 32)];
#pragma unroll
        for (int c = 0; c < HD / 32; ++c) {
            qr[2 * c] = *reinterpret_cast<const f32x4*>(qrow + 32 * c);
            qr[2 * c + 1] = *reinterpret_cast<const f32x4*>(qrow + 32 * c + 4);
        }
        uint32_t key = MagKeys(qr);  // the row's, over its 4 lanes
        key = max(key, static_cast<uint32_t>(__shfl_xor(static_cast<int>(key), 16, kWave)));
        key = max(key, static_cast<uint32_t>(__shfl_xor(static_cast<int>(key), 32, kWave)));
        const MagScale ms(key);
        q_factor = ms.f;
#pragma unroll
        for (int c = 0; c < HD / 32; ++c) {
            h8 pc[2];
            Split8(qr[2 * c], qr[2 * c + 1], ms.s, pc);
            qp[0][c] = pc[0];
            qp[1][c] = pc[1];
        }
    } else {
        const float* qrow = q + t * q_stride + static_cast<int64_t>(h) * HD + 4 * kq;
#pragma unroll
        for (int c = 0; c < NC; ++c) qv[c] = *reinterpret_cast<const f32x4*>(qrow + 16 * c);
    }

    typename std::conditional<kPre, KvBlockPre,
                              typename std::conditional<kF16, KvBlock, KvTile<HD>>::type>::type
        tile;
    if constexpr (kPre) {
        tile.base = reinterpret_cast<const u32x4*>(images) +
                    static_cast<int64_t>(g) * n_image_tiles * kPieceTileU4;
        tile.keys = image_keys + static_cast<int64_t>(g) * n_image_tiles;
    } else {
        tile.kb = kc + static_cast<int64_t>(g) * HD;
        tile.vb = vc + static_cast<int64_t>(g) * HD;
        tile.slot = slot;
        if constexpr (kF16) {
            // a prompt chunk's tiles as KvPieces reads them, to the chunk's
            // last token, so their scales are the images'
            tile.load_pos = kChunked ? max_pos : pos0 + T - 1;
        } else {
            tile.max_pos = max_pos;
        }
    }
    auto load = [&](int64_t p0) { tile.Load(p0); };
    // fp16: true K = stored K * k_factor, true V = stored V * 2^(v_exp - 127)
    float k_factor = 1.0f;
    int v_exp = 127;
    // the tile at p0 from its registers into buffer buf (fp16 without images:
    // after PutMost and a barrier)
    auto store = [&](int buf, int64_t p0) {
        if constexpr (kF16) {
            uint32_t kk, kv;
            if constexpr (kPre) {
                kk = __builtin_amdgcn_readfirstlane(tile.key.x);
                kv = __builtin_amdgcn_readfirstlane(tile.key.y);
            } else {
                kk = GetMost(sm.most[0]);
                kv = GetMost(sm.most[1]);
            }
            const MagScale mk(kk), mv(kv);
            k_factor = mk.f;
            v_exp = mv.fe;
            if ((kPre || !kChunked) && max_pos - p0 < kPfTile - 1) tile.DropV(max_pos - p0);
            tile.Store(sm.k[buf], sm.v[buf], mk.s, mv.s);
        } else {
            tile.Store(sm.k[buf], sm.v[buf]);
        }
    };

    f32x4 acc[NC];  // O^T: acc[c][r] = dim 16c + 4 kq + r of query i16
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY;  // running max of query i16 (equal in its 4 lane groups)
    float l = 0.0f;       // this lane's part of the running sum

    const int64_t n_tiles = (p_end - p_begin + kPfTile - 1) / kPfTile;
    load(p_begin);
    if constexpr (kF16 && !kPre) {
        PutMost(sm.most, tile);
        __syncthreads();
    }
    store(0, p_begin);
    __syncthreads();
    int unit = v_exp;  // fp16: true sums = acc * 2^(unit - 127) * 2^-14
    // positions fit in 32 bits (below max_seq); log2-unit score scale
    const int32_t my_pos_32 = static_cast<int32_t>(my_pos);
    const float scale2 = scale * 1.44269504088896340736f * q_factor;
    for (int64_t it = 0; it < n_tiles; ++it) {
        const int buf = NBUF == 2 ? static_cast<int>(it & 1) : 0;
        const int32_t p0_32 = static_cast<int32_t>(p_begin + it * kPfTile);
        load(p_begin + (it + 1 < n_tiles ? it + 1 : it) * kPfTile);
        // Nothing crosses this point: without it the scheduler sinks the
        // next tile's global loads to their LDS stores at the bottom of the
        // loop, and every tile then waits out a full HBM round trip.
        __builtin_amdgcn_sched_barrier(0);
        {  // idle waves (a head block past the group) compute too, unstored
            f32x4 s[2];
#pragma unroll
            for (int pt = 0; pt < 2; ++pt) {
                s[pt] = f32x4{0.f, 0.f, 0.f, 0.f};
                if constexpr (kF16) {
                    const uint16_t* krow = &sm.k[buf][(pt * 16 + i16) * KL + 8 * kq];
#pragma unroll
                    for (int c = 0; c < HD / 32; ++c) {
                        const h8 k0 = *reinterpret_cast<const h8*>(krow + 32 * c);
                        const h8 k1 = *reinterpret_cast<const h8*>(krow + kPfTile * KL + 32 * c);
                        s[pt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(k1, qp[0][c], s[pt], 0, 0, 0);
                        s[pt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(k0, qp[1][c], s[pt], 0, 0, 0);
                        s[pt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(k0, qp[0][c], s[pt], 0, 0, 0);
                    }
                } else {
                    const float* krow = &sm.k[buf][(pt * 16 + i16) * LD + 4 * kq];
#pragma unroll
                    for (int c = 0; c < NC; ++c) {
                        const f32x4 kk = *reinterpret_cast<const f32x4*>(krow + 16 * c);
#pragma unroll
                        for (int st = 0; st < 4; ++st) {
                            s[pt] = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[st], qv[c][st], s[pt],
                                                                         0, 0, 0);
                        }
                    }
                }
            }
            float sv[8];
            float tmax = -INFINITY;
#pragma unroll
            for (int pt = 0; pt < 2; ++pt) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    // scores in log2 units (scale * log2(e)), for exp2 below
                    const int32_t pos = p0_32 + pt * 16 + 4 * kq + r;
                    // (fp16: K's factor, then q's with the scale)
                    const float sr = kF16 ? s[pt][r] * k_factor : s[pt][r];
                    const float x = pos <= my_pos_32 ? sr * scale2 : -INFINITY;
                    sv[pt * 4 + r] = x;
                    tmax = fmaxf(tmax, x);
                }
            }
            tmax = fmaxf(tmax, __shfl_xor(tmax, 16, kWave));
            tmax = fmaxf(tmax, __shfl_xor(tmax, 32, kWave));
            // finite: position 0 is in every query's range.  In a chunk, a
            // token before the chunk (or invalid) sees only -inf: it is
            // referenced to 0 and keeps m = -inf, l = 0 (AttnCombine never
            // reads that partial).
            const float mnew = fmaxf(m, tmax);
            const float mref = kChunked && mnew == -INFINITY ? 0.0f : mnew;
            // rescale only when some query's max moved (the factor is then
            // exactly 1 for the others: skipping it changes nothing), or the
            // accumulators' unit grows to this V tile's
            if (__builtin_amdgcn_ballot_w64(mnew != m) != 0) {
                const float corr = __builtin_amdgcn_exp2f(m - mref);
                l *= corr;
#pragma unroll
                for (int c = 0; c < NC; ++c) acc[c] *= corr;
            }
            if (kF16 && v_exp > unit) {
                const float grow = Pow2Field(127 + unit - v_exp);
#pragma unroll
                for (int c = 0; c < NC; ++c) acc[c] *= grow;
                unit = v_exp;
            }
            float pv[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                pv[i] = __builtin_amdgcn_exp2f(sv[i] - mref);
                l += pv[i];
            }
            m = mnew;
            if constexpr (kF16) {
                // B: this lane's probabilities, slot j = position 16 (j / 4) + 4 kq + j % 4
                h8 pp[2];
                Split8(f32x4{pv[0], pv[1], pv[2], pv[3]}, f32x4{pv[4], pv[5], pv[6], pv[7]},
                       Pow2Field(127 + 14 + v_exp - unit), pp);
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    const uint16_t* vrow = &sm.v[buf][(16 * c + i16) * kVLd + 8 * kq];
                    const h8 v0 = *reinterpret_cast<const h8*>(vrow);
                    const h8 v1 = *reinterpret_cast<const h8*>(vrow + HD * kVLd);
                    acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(v1, pp[0], acc[c], 0, 0, 0);
                    acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(v0, pp[1], acc[c], 0, 0, 0);
                    acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(v0, pp[0], acc[c], 0, 0, 0);
                }
            } else {
#pragma unroll
                for (int c = 0; c < NC; ++c) {
#pragma unroll
                    for (int pt = 0; pt < 2; ++pt) {
#pragma unroll
                        for (int st = 0; st < 4; ++st) {
                            const float vv = sm.v[buf][(pt * 16 + 4 * kq + st) * LD + 16 * c + i16];
                            acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(vv, pv[pt * 4 + st],
                                                                          acc[c], 0, 0, 0);
                        }
                    }
                }
            }
        }
        const int64_t p_next = p_begin + (it + 1 < n_tiles ? it + 1 : it) * kPfTile;
        if constexpr (kF16 && !kPre) PutMost(sm.most, tile);
        // one buffer: every wave is done with the tile before it is replaced;
        // fp16 without images: the next tile's largest magnitudes are known
        if constexpr (NBUF == 1 || (kF16 && !kPre)) __syncthreads();
        store(NBUF == 1 ? 0 : buf ^ 1, p_next);
        __syncthreads();
    }
    if constexpr (kF16) {  // out of the fp16 unit
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[c] = acc[c] * (1.0f / 16384.0f) * Pow2Field(unit);
    }
    l += __shfl_xor(l, 16, kWave);
    l += __shfl_xor(l, 32, kWave);
    if (!active || t0 + i16 > last_t) return;
    if constexpr (kChunked) {
        const int64_t row = t * H + h;
        if (tc.n_chunks > 1) {  // unnormalized partials, merged by AttnCombine
            float* arow = tc.ws_acc + (row * tc.n_chunks + ck) * HD + 4 * kq;
#pragma unroll
            for (int cc = 0; cc < NC; ++cc) {
                *reinterpret_cast<float4*>(arow + 16 * cc) =
                    make_float4(acc[cc][0], acc[cc][1], acc[cc][2], acc[cc][3]);
            }
            if (kq == 0) {  // the max back in natural-log units, as AttnCombine takes it
                tc.ws_ml[(row * tc.n_chunks + ck) * 2] = m * 0.69314718055994530942f;
                tc.ws_ml[(row * tc.n_chunks + ck) * 2 + 1] = l;
            }
            return;
        }
        if (!valid) {  // one chunk: the row is final here
            float* orow = out + row * HD + 4 * kq;
#pragma unroll
            for (int cc = 0; cc < NC; ++cc) {
                *reinterpret_cast<float4*>(orow + 16 * cc) = make_float4(0.f, 0.f, 0.f, 0.f);
            }
            return;
        }
    }
    float* orow = out + (t * H + h) * static_cast<int64_t>(HD) + 4 * kq;
    const float inv = 1.0f / l;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const float4 o = make_float4(acc[c][0] * inv, acc[c][1] * inv, acc[c][2] * inv,
                                     acc[c][3] * inv);
        *reinterpret_cast<float4*>(orow + 16 * c) = o;
        // the output rows [T, H * HD] also as StorePlanes planes (wo's x)
        if (a_planes != nullptr) {
            StorePlanes4(a_planes, T, t, static_cast<int64_t>(h) * HD + 16 * c + 4 * kq, o.x, o.y,
                         o.z, o.w);
        }
    }
}

}  // namespace

bool PrefillSupported(int32_t head_dim, const float* q, int64_t q_row_stride, const float* out,
                      const float* k_cache, const float* v_cache) {
    return (head_dim == 64 || head_dim == 128) && q_row_stride % 4 == 0 && Aligned(q, 16) &&
           Aligned(out, 16) && Aligned(k_cache, 16) && Aligned(v_cache, 16);
}

int64_t PrefillImageBytes(int32_t n_kv_heads, int32_t head_dim, int64_t n_pos) {
    if (head_dim != 128 || n_kv_heads <= 0 || n_pos <= 0) return 0;
    // a tile's image and its two keys (rounded up to 16 bytes)
    return static_cast<int64_t>(n_kv_heads) * ((n_pos + kPfTile - 1) / kPfTile) *
           (kPieceTileU4 * 16 + 16);
}

namespace {

// K and V of positions 0 .. n_pos - 1 into tile images and keys at `images`
// (PrefillImageBytes).
mlk_status LaunchPieces(const float* kc, const float* vc, int64_t slot, int32_t KV, int64_t n_pos,
                        uint16_t* images, uint2** keys, int64_t* n_tiles, hipStream_t s) {
    *n_tiles = (n_pos + kPfTile - 1) / kPfTile;
    if (*n_tiles * KV > 0x7FFFFFFF) {
        return Fail(MLK_ERR_INVALID, "attention prefill: launch too large");
    }
    *keys = reinterpret_cast<uint2*>(images + *n_tiles * KV * (2 * kPieceHalves));
    hipLaunchKernelGGL(KvPieces, dim3(static_cast<unsigned>(*n_tiles * KV)), dim3(kPfThreads), 0, s,
                       kc, vc, slot, KV, n_pos - 1, *n_tiles, images, *keys);
    return CheckLaunch("KvPieces");
}

}  // namespace

mlk_status LaunchPrefill(const float* q, int64_t q_row_stride, const float* kc, const float* vc,
                         int64_t slot, int32_t H, int32_t KV, int32_t head_dim, int32_t pos0,
                         int64_t T, float* out, hipStream_t s, void* workspace,
                         size_t workspace_bytes, uint32_t* a_planes) {
    const int group = H / KV;
    const int head_blocks = (group + kPfHeads - 1) / kPfHeads;
    const int64_t n_tb = (T + kPfTokens - 1) / kPfTokens;
    const int64_t blocks = n_tb * KV * head_blocks;
    if (blocks > 0x7FFFFFFF) return Fail(MLK_ERR_INVALID, "attention prefill: launch too large");
    const float scale = 1.0f / sqrtf(static_cast<float>(head_dim));
    const dim3 grid(static_cast<unsigned>(blocks));
    const TileChunks none{};
    // head_dim 128 with room for the tile images: split K and V once
    // (positions 0 .. pos0 + T - 1), then stage the images
    const int64_t n_pos = pos0 + T;
    const int64_t image_bytes = PrefillImageBytes(KV, head_dim, n_pos);
    if (image_bytes > 0 && T >= kPrefillImageMinTokens && workspace != nullptr &&
        Aligned(workspace, 16) &&
        static_cast<int64_t>(workspace_bytes) >= image_bytes) {
        uint16_t* images = static_cast<uint16_t*>(workspace);
        uint2* keys = nullptr;
        int64_t n_tiles = 0;
        const mlk_status st = LaunchPieces(kc, vc, slot, KV, n_pos, images, &keys, &n_tiles, s);
        if (st != MLK_OK) return st;
        hipLaunchKernelGGL((AttnPrefill<128, false, true, 1, true>), grid, dim3(kPfThreads), 0, s,
                           q, q_row_stride, kc, vc, slot, KV, H, pos0, T, scale, out, head_blocks,
                           none, images, keys, n_tiles, a_planes);
        return CheckLaunch("AttnPrefill");
    }
    if (head_dim == 64) {
        hipLaunchKernelGGL((AttnPrefill<64, false, false>), grid, dim3(kPfThreads), 0, s, q,
                           q_row_stride, kc, vc, slot, KV, H, pos0, T, scale, out, head_blocks,
                           none, nullptr, nullptr, 0, a_planes);
    } else {
        hipLaunchKernelGGL((AttnPrefill<128, false, true, 1>), grid, dim3(kPfThreads), 0, s, q,
                           q_row_stride, kc, vc, slot, KV, H, pos0, T, scale, out, head_blocks,
                           none, nullptr, nullptr, 0, a_planes);
    }
    return CheckLaunch("AttnPrefill");
}

// Positions per chunk: a power of two from 256 up to the whole context,
// halved while the grid has fewer than 512 workgroups.  Large batches then
// take the context in one chunk (no partials, no merge).
int TileChunk(int64_t T, int32_t H, int32_t KV, int64_t max_ctx) {
    const int group = H / KV;
    const int64_t base = (T + kPfTokens - 1) / kPfTokens * KV * ((group + kPfHeads - 1) / kPfHeads);
    int64_t chunk = 256;
    while (chunk < max_ctx && chunk < (int64_t{1} << 30)) chunk *= 2;
    while (chunk > 256 && base * ((max_ctx + chunk - 1) / chunk) < 512) chunk /= 2;
    return static_cast<int>(chunk);
}

int64_t PrefillChunks(int64_t T, int32_t H, int32_t KV, int64_t n_pos, int64_t max_ctx,
                      int* chunk) {
    const int group = H / KV;
    const int64_t base = (T + kPfTokens - 1) / kPfTokens * KV * ((group + kPfHeads - 1) / kPfHeads);
    *chunk = 1 << 30;
    if (base > ComputeUnits() || n_pos < kPrefillSplitMinCtx) return 1;
    // by the positions there are, within the chunks of the workspace's sizing
    const int max_chunk = TileChunk(T, H, KV, max_ctx);
    const int64_t most = (max_ctx + max_chunk - 1) / max_chunk;
    *chunk = TileChunk(T, H, KV, n_pos);
    while ((n_pos + *chunk - 1) / *chunk > most) *chunk *= 2;
    return (n_pos + *chunk - 1) / *chunk;
}

mlk_status LaunchDecodeTile(const float* q, int64_t q_row_stride, const float* kc,
                            const float* vc, int64_t slot, int32_t H, int32_t KV,
                            int32_t head_dim, const int32_t* positions, int32_t pos0, int64_t T,
                            int64_t max_ctx, int chunk, float* out, float* ws_acc, float* ws_ml,
                            int32_t* err, hipStream_t s, void* images_at) {
    const int group = H / KV;
    const int head_blocks = (group + kPfHeads - 1) / kPfHeads;
    const int64_t n_tb = (T + kPfTokens - 1) / kPfTokens;
    const int64_t nc = (max_ctx + chunk - 1) / chunk;
    const int64_t blocks = n_tb * KV * head_blocks * nc;
    if (blocks > 0x7FFFFFFF) return Fail(MLK_ERR_INVALID, "attention decode: launch too large");
    TileChunks tc{positions, max_ctx, chunk, static_cast<int>(nc), ws_acc, ws_ml, err};
    const float scale = 1.0f / sqrtf(static_cast<float>(head_dim));
    const dim3 grid(static_cast<unsigned>(blocks));
    if (head_dim == 64) {
        hipLaunchKernelGGL((AttnPrefill<64, true, false>), grid, dim3(kPfThreads), 0, s, q,
                           q_row_stride, kc, vc, slot, KV, H, pos0, T, scale, out, head_blocks,
                           tc, nullptr, nullptr, 0, nullptr);
    } else if (images_at != nullptr) {
        // (consecutive positions) tiles from images, as LaunchPrefill
        uint16_t* images = static_cast<uint16_t*>(images_at);
        uint2* keys = nullptr;
        int64_t n_tiles = 0;
        const mlk_status st =
            LaunchPieces(kc, vc, slot, KV, pos0 + T, images, &keys, &n_tiles, s);
        if (st != MLK_OK) return st;
        hipLaunchKernelGGL((AttnPrefill<128, true, true, 1, true>), grid, dim3(kPfThreads), 0, s, q,
                           q_row_stride, kc, vc, slot, KV, H, pos0, T, scale, out, head_blocks,
                           tc, images, keys, n_tiles, nullptr);
    } else if (blocks <= ComputeUnits()) {
        // two tile buffers (76 KB of LDS)
        hipLaunchKernelGGL((AttnPrefill<128, true, true>), grid, dim3(kPfThreads), 0, s, q,
                           q_row_stride, kc, vc, slot, KV, H, pos0, T, scale, out, head_blocks,
                           tc, nullptr, nullptr, 0, nullptr);
    } else {
        hipLaunchKernelGGL((AttnPrefill<128, true, true, 1>), grid, dim3(kPfThreads), 0, s, q,
                           q_row_stride, kc, vc, slot, KV, H, pos0, T, scale, out, head_blocks,
                           tc, nullptr, nullptr, 0, nullptr);
    }
    return CheckLaunch("AttnPrefill (decode tokens)");
}

}  // namespace mlk
