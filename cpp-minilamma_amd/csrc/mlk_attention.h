// mlk_attention.h -- the causal prefill attention kernel (mlk_prefill.hip)
// as used by the attention entry points (mlk_attention.hip).
#pragma once

#include "mlk_common.h"

namespace mlk {

// The prefill kernel handles head_dim 64 and 128 with 16-byte aligned q
// rows (q_row_stride % 4 == 0), output and caches.
bool PrefillSupported(int32_t head_dim, const float* q, int64_t q_row_stride, const float* out,
                      const float* k_cache, const float* v_cache);

// Tokens t < T at positions pos0 + t, each attending to cache positions
// 0 .. pos0 + t; kc / vc point at the layer's [max_seq, KV, head_dim] slice,
// slot = KV * head_dim floats per position.  Arguments already validated.
// With a 16-byte aligned workspace of PrefillImageBytes(KV, head_dim,
// pos0 + T) bytes (head_dim 128, PrefillImages), K and V of positions 0 ..
// pos0 + T - 1 are first split into bf16 piece images, one launch, which the
// tiles then copy instead of splitting each tile in every workgroup; the sums
// are the same.  Otherwise no workspace is used.  a_planes (16-byte aligned,
// H * head_dim a multiple of 32), when set, also receives the output rows as
// StorePlanes planes.
// Where the images pay: a tile has to be staged by enough workgroups (Llama-3
// heads, 8B / 70B: 389 tokens after 1500 133 -> 124 / 169 -> 162 us, at 4000
// in chunks 229 -> 221, 128 tokens there 77 -> 83, 1024 from position 0 80 ->
// 77 / 118 -> 114, 4096 763 -> 708 / 1547 -> 1427, but 512 41 -> 40 / 44 ->
// 47).
inline bool PrefillImages(int64_t T, int64_t pos0) { return T >= 1024 || (T >= 384 && pos0 >= T); }
// A prompt chunk whose token blocks are at most one workgroup per compute
// unit, over a context of at least kPrefillSplitMinCtx positions, is split
// over chunks of positions like decode tokens (LaunchDecodeTile): the number
// of chunks of its n_pos positions (1: not split; at most TileChunk's for
// max_ctx) and their length.  Llama-3-8B heads, whole ->
// in chunks: 64 tokens at 4000 267 -> 47 us, 128 at 4000 278 -> 77, 389 at
// 6000 424 -> 328; more blocks than units fill the chip by themselves (700 at
// 2000 took 1.5 times as long in chunks).  Over short contexts the merge costs
// more than the split gives (389 from position 0 took twice as long); over
// 1000 positions it would gain (128 tokens a third), but up to here a call with
// a workspace keeps the sums of the prefill entry, which has none, bit for bit.
constexpr int64_t kPrefillSplitMinCtx = 2048;
int64_t PrefillChunks(int64_t T, int32_t H, int32_t KV, int64_t n_pos, int64_t max_ctx,
                      int* chunk);
int64_t PrefillImageBytes(int32_t n_kv_heads, int32_t head_dim, int64_t n_pos);
mlk_status LaunchPrefill(const float* q, int64_t q_row_stride, const float* kc, const float* vc,
                         int64_t slot, int32_t H, int32_t KV, int32_t head_dim, int32_t pos0,
                         int64_t T, float* out, hipStream_t s, void* workspace = nullptr,
                         size_t workspace_bytes = 0, uint32_t* a_planes = nullptr);

// Decode tokens at any positions (positions[t], or pos0 + t) on the same
// matrix-core tiles: a workgroup holds 16 tokens and shares each K/V tile
// among them, over one chunk of TileChunk() cache positions.  With more than
// one chunk it writes (acc, m, l) partials to ws_acc / ws_ml ([T, H, n_chunks,
// hd] / [.., 2], n_chunks = ceil(max_ctx / chunk)) for AttnCombine; with one
// it writes out.  Invalid positions raise err (their rows are zeroed by the
// merge, or here with one chunk).  images_at (consecutive positions,
// head_dim 128): room for PrefillImageBytes(KV, head_dim, pos0 + T), used as
// in LaunchPrefill.  Arguments already validated.
int TileChunk(int64_t T, int32_t H, int32_t KV, int64_t max_ctx);
mlk_status LaunchDecodeTile(const float* q, int64_t q_row_stride, const float* kc,
                            const float* vc, int64_t slot, int32_t H, int32_t KV,
                            int32_t head_dim, const int32_t* positions, int32_t pos0, int64_t T,
                            int64_t max_ctx, int chunk, float* out, float* ws_acc, float* ws_ml,
                            int32_t* err, hipStream_t s, void* images_at = nullptr);

// Workspace of a prompt chunk (positions == NULL, 16 or more tokens): chunk
// partials and tile images, whichever its call uses.
int64_t PromptAttentionBytes(int64_t T, int32_t H, int32_t KV, int32_t head_dim, int64_t max_ctx);

// mlk_attention_decode_f32 with one more output: when the chunk merge runs
// (more than one chunk of cache positions) and planes is not null, the merge
// also writes out's bf16 planes (StorePlanes1 over rows of n_heads * head_dim,
// which must be a multiple of 32) and sets *planes_written, and so does the
// prefill kernel (positions == NULL, 16 or more tokens); otherwise planes
// are untouched and *planes_written is false.
mlk_status AttentionDecode(const float* q, int64_t q_row_stride, const float* k_cache,
                           const float* v_cache, int64_t n_layers, int64_t max_seq,
                           int32_t n_heads, int32_t n_kv_heads, int32_t head_dim, int64_t layer,
                           const int32_t* positions, int32_t pos0, int64_t n_tokens,
                           int64_t max_ctx, float* out, void* workspace, size_t workspace_bytes,
                           int32_t* err, void* stream, uint32_t* planes, bool* planes_written);

}  // namespace mlk
