// Launch-function declarations: pure-HIP translation units (one per
// kernel family) export these; ext.cpp (the only file that includes
// torch headers) validates tensors and calls them.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

#include "prefill_parts.h"

namespace rlli {

// y = rmsnorm(x) * w           (residual == nullptr)
// r += x; y = rmsnorm(r) * w   (fused residual-add form)
void launch_rmsnorm(const uint16_t* x, uint16_t* residual, const uint16_t* w,
                    uint16_t* y, int rows, int dim, float eps,
                    hipStream_t stream);

// The same with x = the sum of n f32 parts [n, rows, dim]; dim <= 8192.
void launch_rmsnorm_parts(const float* parts, int n, uint16_t* residual,
                          const uint16_t* w, uint16_t* y, int rows, int dim,
                          float eps, hipStream_t stream);

// out[t, i] = silu(gu[t, i]) * gu[t, I + i]   for packed gate|up rows
void launch_silu_mul(const uint16_t* gate_up, uint16_t* out, int rows,
                     int inter, hipStream_t stream);

// In-place RoPE (NeoX-interleaved-halves style) on q and k, then scatter
// k/v into the paged cache at slot_mapping[t].
// q/k/v may be strided slices of one fused [T, (n_q+2*n_kv)*D] qkv
// tensor: *_stride is the per-token element stride of each view.
// Cache pointers are void*: the paged cache stores bf16 (default) or
// OCP fp8-e4m3 (cache_fp8) — see common.h cache codecs.
// FP8-activation emitters for the quantized-weight GEMM path
// (rowwise torch._scaled_mm consumers): normed / activated rows out as
// fp8-e4m3 + one dequant scale per row.
void launch_rmsnorm_fp8(const uint16_t* x, uint16_t* residual,
                        const uint16_t* w, uint8_t* y8, float* scales,
                        int rows, int dim, float eps, hipStream_t stream);
void launch_silu_mul_fp8(const uint16_t* gate_up, uint8_t* out8,
                         float* scales, int rows, int inter,
                         hipStream_t stream);

void launch_rope_kv_append(
    uint16_t* q, uint16_t* k, uint16_t* v,
    const int32_t* positions, const float* cos_sin,   // [max_pos, head_dim]
    void* k_cache, void* v_cache,
    const int32_t* slot_mapping,
    int tokens, int n_q_heads, int n_kv_heads, int head_dim,
    int block_size, int q_stride, int kv_stride, bool cache_fp8,
    hipStream_t stream);

// Paged GQA decode attention, one new query per sequence.  Fused form
// (positions given): q | k | v rows, or their f32 parts, are rotated and
// appended as well (no slot_mapping: queries are rotated, nothing appended).
// decode_attn_shares: equal shares of all sequences' tokens that workgroups
// take per key/value head, for which part_out [n_kv, shares + batch, group,
// head_dim] and part_ml [.., group, 2] are needed; 0: a workgroup takes a
// whole sequence.  ``apart``: sequences that were cut are left in their parts.
int decode_attn_shares(int batch, int n_kv_heads, int max_tokens);
void launch_decode_attn(
    const uint16_t* q,                 // [batch, q_stride], or null:
    const float* parts, int n_parts,   // [n_parts, batch, q_stride]
    void* k_cache,                     // [blocks, n_kv, block_size, head_dim]
    void* v_cache,
    const int32_t* block_table,        // [batch, max_blocks]
    const int32_t* seq_lens,           // [batch]
    const int32_t* positions,          // [batch] or null
    const float* cos_sin, const int32_t* slot_mapping,    // or null
    uint16_t* out,                     // [batch, n_q_heads, head_dim]
    int batch, int n_q_heads, int n_kv_heads, int head_dim, int block_size,
    int max_blocks, float scale, int q_stride, int shares, float* part_out,
    float* part_ml, bool cache_fp8, bool apart, hipStream_t stream);

// What says which pages the rows of a mixed step see: decoding sequences
// first, then tiles of at most 32 prompt rows.
struct RowTables {
  const int32_t *tables_dec, *lens_dec;       // [n_decode, dec_width], [..]
  const int32_t *row0, *pos0, *nrows, *btrow; // [n_tiles]
  const int32_t* tables_pre;                  // [.., pre_width]
  int n_decode, dec_width, n_tiles, pre_width;
};
// tables [rows, wide], lens [rows]
void launch_row_tables(const RowTables& a, int32_t* tables, int32_t* lens,
                       int rows, int wide, hipStream_t stream);

// Varlen causal prefill attention over in-batch q/k/v.
void launch_prefill_attn(
    const uint16_t* q, const uint16_t* k, const uint16_t* v,
    const int32_t* cu_seqlens,         // [n_seqs + 1]
    uint16_t* out,
    int n_seqs, int total_tokens, int n_q_heads, int n_kv_heads,
    int head_dim, float scale, int q_stride, int kv_stride,
    hipStream_t stream);

// Causal attention of whole prompts over a fused qkv tensor; cu_seqlens
// [n_seqs + 1] stays on the device.
void launch_prefill_rows(const uint16_t* qkv, const int32_t* cu_seqlens,
                         uint16_t* out, int n_seqs, int rows, int n_kv_heads,
                         int group, int head_dim, int qkv_stride, float scale,
                         hipStream_t stream);

// The same of sequences of up to 64 rows with the rotation of queries and keys
// and the append to the cache; qkv stays as it is.
void launch_prompt_rows_attn(const uint16_t* qkv, const int32_t* cu_seqlens,
                             const int32_t* positions, const float* cos_sin,
                             void* k_cache, void* v_cache,
                             const int32_t* slot_mapping, uint16_t* out,
                             int n_seqs, int rows, int n_kv_heads, int group,
                             int head_dim, int block_size, int qkv_stride,
                             float scale, bool cache_fp8, hipStream_t stream);

// The same over the paged cache (chunks and mixed batches).
void launch_prefill_paged(const uint16_t* qkv, const void* k_cache,
                          const void* v_cache, const int32_t* chunk_row0,
                          const int32_t* chunk_pos0,
                          const int32_t* chunk_nrows,
                          const int32_t* chunk_btrow,
                          const int32_t* block_tables, uint16_t* out,
                          int n_chunks, int n_kv_heads, int group,
                          int head_dim, int qkv_stride, int max_blocks,
                          int block_size, float scale, bool cache_fp8,
                          const PrefillParts& parts, hipStream_t stream);

// Prompt rows and decoding sequences of a mixed step at once (mixed_attn.hip).
// What the tiles' keys are divided into and the sequences' shares; splits 0:
// not for these sizes; faster: than one after the other.  ``keys``, ``max_tokens``:
// what the tables have room for.
struct MixedPlan {
  int splits, shares;
  bool faster;
};
MixedPlan mixed_attn_plan(int n_tiles, int batch, int n_kv, int group,
                          int head_dim, int keys, int max_tokens, int elem,
                          int block_size);
void launch_mixed_attn(const uint16_t* qkv, void* k_cache, void* v_cache,
                       const int32_t* chunk_row0, const int32_t* chunk_pos0,
                       const int32_t* chunk_nrows, const int32_t* chunk_btrow,
                       const int32_t* tables_pre, int pre_blocks,
                       const int32_t* tables_dec, const int32_t* lens_dec,
                       int dec_blocks, uint16_t* out, int n_tiles, int batch,
                       int n_kv, int group, int head_dim, int stride,
                       float scale, bool cache_fp8, const PrefillParts& parts,
                       int shares, float* part_out, float* part_ml,
                       hipStream_t stream);

// Products of at most 128 rows, y[M, N] = x[M, K] w[N, K]^T (rows_gemm.hip).
// With parts given, f32 [splits, M, N] whose sum is y; otherwise out.
// N % 4 == 0, K % 64 == 0, 16-byte aligned rows.
int rows_gemm_splits(int N, int K);
void launch_rows_gemm(const uint16_t* x, const uint16_t* w, float* parts,
                      uint16_t* out, int M, int N, int K, int splits,
                      hipStream_t stream);
// silu(x w[:I]^T) * (x w[I:]^T) for w [2 I, K]; false where I is so small
// that the product in parts is faster
bool rows_gemm_silu_ok(int inter);
void launch_rows_gemm_silu(const uint16_t* x, const uint16_t* w,
                           uint16_t* out, int M, int inter, int K,
                           hipStream_t stream);
// The same two for one row, the norm of residual + the sum of n parts [n, K],
// which goes to residual_out, where rows_norm_ok.
struct RowsNorm {
  const float* parts;
  const uint16_t* residual;
  uint16_t* residual_out;
  const uint16_t* gain;
  int n;
  float eps;
};
// Of one sequence's attention in parts, which launch_decode_attn left apart:
// its output, at ``whole`` if it was not cut, times w.
struct RowsCombine {
  const float *o, *ml;         // as launch_decode_attn has them
  const uint16_t* whole;       // [K]
  const int32_t* len;
  int shares, group, head_dim;
};
// where that is the faster way, of up to max_tokens
bool rows_combine_ok(int N, int K, int max_tokens);
void launch_rows_combine(const RowsCombine& attn, const uint16_t* w,
                         float* parts, int N, int K, int splits,
                         hipStream_t stream);
bool rows_norm_ok(int N, int K, bool silu);
void launch_rows_norm(const RowsNorm& norm, const uint16_t* w, float* parts,
                      int N, int K, int splits, hipStream_t stream);
void launch_rows_norm_silu(const RowsNorm& norm, const uint16_t* w,
                           uint16_t* out, int inter, int K,
                           hipStream_t stream);
// A norm that two products share, of up to 32 rows.  The first adds its result to
// the streams [M, S, N] (each takes out_w of it and mix [from, to] of all, and in_w
// of each is what is normed) and writes rows times gains and sums of squares
// [N / 16, 16 or 32]; the second takes both, for its squared positive part.
struct RowsAdds {
  float* streams;
  const float *mix, *out_w, *in_w, *gain;
  float* ss;
};
struct RowsScale {
  const float* ss;
  int panels, width;           // N / 16 and N of the first product
  float eps;
};
bool rows_adds_ok(int M, int N, int K, int streams);
void launch_rows_adds(const uint16_t* x, const uint16_t* w, uint16_t* out,
                      int M, int N, int K, int streams, const RowsAdds& adds,
                      hipStream_t stream);
bool rows_scaled_ok(int M, int N, int K);
void launch_rows_scaled_relu2(const uint16_t* x, const uint16_t* w,
                              uint16_t* out, int M, int N, int K,
                              const RowsScale& scale, hipStream_t stream);
// M <= 64 where rows_short_ok; ``relu2``: squared positive part
bool rows_short_ok(int N, int K);
void launch_rows_short(const uint16_t* x, const uint16_t* w, uint16_t* out,
                       int M, int N, int K, bool relu2, hipStream_t stream);
// more rows: tiles of ``rows`` rows by 8 ``eights`` rows of w; ``relu2`` of the
// 16-bit product
struct TallPlan {
  int rows, eights;
};
TallPlan rows_tall_plan(int M, int N);
void launch_rows_tall(const uint16_t* x, const uint16_t* w, uint16_t* out,
                      int M, int N, int K, bool relu2, const TallPlan& plan,
                      hipStream_t stream);
void launch_sum_parts(const float* parts, uint16_t* out, int splits,
                      int64_t n, hipStream_t stream);

// The same product of more rows (tile_gemm.hip): f32 parts [splits, M, N] or, if
// the plan does not divide K, out [M, N]; with an activation, which wants the
// product ``whole``, out [M, N / 2] of w's gate and up rows or its squared
// positive part.  K % 64 == 0, N % 8 == 0 (16 with silu), 16-byte aligned rows,
// operands below 2^32 bytes.
struct TilePlan {
  int mh, nh, splits;
};
enum class TileAct { none, silu, relu2 };
TilePlan tile_gemm_plan(int M, int N, int K, bool whole);
// whether there is such a tile and division of K
bool tile_gemm_ok(const TilePlan& plan, int K, bool whole);
void launch_tile_gemm(const uint16_t* x, const uint16_t* w, float* parts,
                      uint16_t* out, int M, int N, int K, TileAct act,
                      const TilePlan& plan, hipStream_t stream);

// A decode step's buffers, rows of a batch (decode_state.hip).
struct DecodeState {
  int32_t *ids, *positions;
  int32_t* tables;             // [.., width]
  float* temps;
  int64_t* seeds;
  int32_t* slots;              // of what is loaded: or null
  int width;
};
// The first ``bucket`` rows, of which ``batch`` come from a batch with tables
// [batch, wide].
void launch_decode_load(const DecodeState& to, const DecodeState& from,
                        int bucket, int batch, int wide, int scratch_block,
                        int scratch_slot, hipStream_t stream);
void launch_decode_begin(const int32_t* positions, const int32_t* tables,
                         int32_t* slots, int32_t* lens, int batch, int width,
                         int block_size, hipStream_t stream);
void launch_decode_advance(int32_t* ids, int32_t* positions, int64_t* seeds,
                           const int32_t* tokens, int batch,
                           int64_t seed_step, hipStream_t stream);

// Diagnostic: W streamed past the caches, 64 rows by a part of K per workgroup.
void launch_stream_probe(const uint16_t* w, float* sink, int N, int K,
                         int splitk, hipStream_t stream);

// Fused sampling: greedy argmax when temperature[i] == 0, else Gumbel-max
// sampling of softmax(logits / temperature[i]) with an in-kernel counter
// hash RNG keyed on (seed, row, column) — no 32 MB random tensor per step.
int sample_n_split(int batch);       // phase-A split factor (1 = single)
void launch_sample(
    const void* logits, bool f32,      // [batch, vocab] bf16 or f32
    const float* temperatures,         // [batch]
    const uint64_t* seeds,             // [batch] per-request seeds
    uint64_t step,                     // per-sequence step counter (mixed in)
    int32_t* out_tokens,               // [batch]
    int batch, int vocab,
    uint64_t* partials, int n_split,   // [batch, n_split] workspace
    hipStream_t stream);

}  // namespace rlli
