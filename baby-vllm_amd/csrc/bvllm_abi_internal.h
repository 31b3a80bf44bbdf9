// Argument blocks passed from the C-ABI entry points to the kernel launchers.
// All strides are in elements. Tensors are bf16 unless noted.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bvllm_fast_div.h"

namespace bvllm {

struct RopeArgs {
  void* q;        int64_t q_st, q_sh;      // [T, H, D], last-dim stride 1
  void* k;        int64_t k_st, k_sh;      // [T, Hkv, D]
  const void* v;  int64_t v_st, v_sh;      // [T, Hkv, D]
  const void* cos; int64_t cs_st;          // [T, D]
  const void* sin; int64_t sn_st;          // [T, D]
  void* k_cache;  int64_t kc_slot, kc_head;  // flat [NB·BS, Hkv, D] view of kv_cache[0]
  void* v_cache;  int64_t vc_slot, vc_head;  // flat view of kv_cache[1]
  const int64_t* slot_mapping;             // [T]
  int64_t num_slots;                       // NB·BS; slots outside [0, num_slots) are not written
  int32_t num_tokens, num_heads, num_kv_heads, head_dim;
  int32_t has_cache;
  int32_t vec_ok;                          // every row start and stride is 16-byte aligned
};

struct DecodeArgs {
  const void* q;  int64_t q_sb, q_sh;      // [B, H, D]
  const void* k_cache; const void* v_cache;  // [NB, BS, Hkv, D] each
  int64_t c_sb, c_st, c_sh;                // page, token, head strides (shared by K and V)
  int32_t num_pages;                       // NB; table entries are clamped into [0, NB)
  const int32_t* block_tables; int64_t bt_stride; int32_t max_blocks;
  const int32_t* seq_lens;                 // [B]
  float scale_log2;                        // softmax scale · log2(e)
  void* out;      int64_t o_sb, o_sh;      // [B, H, D], written when num_splits == 1
  float* part_out;                         // [B, H, parts, D] fp32 partial outputs
  float* part_lse;                         // [B, H, parts] fp32 (log2 units)
  int32_t num_splits, blocks_per_split;
  int32_t batch, num_heads, num_kv_heads, head_dim;
  int32_t waves;                           // waves per single-pass work-group (4; 0 = default)
  // Set by the launcher for split launches (decode_plan):
  int32_t splits_per_item;                 // consecutive splits one streaming wave computes
  int32_t num_partials;                    // partial states per (row, head) the launch writes
  int32_t ws_partials;                     // partial states per (row, head) the workspace holds
  int32_t item_order;                      // numbering: 0 KV head, unit, row (fastest first); 1 unit, KV head, row;
                                           // 2 as 0 with the empty units last
  // Balanced single pass (RowChunk): chunks aimed at per column group, rows an even
  // share of which keeps every CU busy.
  int32_t chunk_target, row_slots;
  FastDiv by_col_groups, by_units;         // of item orders 0 and 2
  // Prefill view (both null for a decode batch): row b is sequence b of a
  // varlen prefill batch. Only sequences with exactly one query token are
  // computed; their q / out row is query_start_loc[b] and they attend keys
  // 0 .. min(seq_lens[b], context_lens[b] + 1) - 1.
  const int32_t* query_start_loc;
  const int32_t* context_lens;
};

struct PrefillArgs {
  const void* q;  int64_t q_st, q_sh;      // [T, H, D]
  const void* k_cache; const void* v_cache;
  int64_t c_sb, c_st, c_sh;
  int32_t num_pages;
  const int32_t* block_tables; int64_t bt_stride; int32_t max_blocks;
  const int32_t* query_start_loc;          // [S+1]
  const int32_t* seq_lens;                 // [S]
  const int32_t* context_lens;             // [S]
  float scale_log2;
  void* out;      int64_t o_st, o_sh;      // [T, H, D]
  int32_t num_seqs, num_tokens, max_query_len;
  int32_t num_heads, num_kv_heads, head_dim;
  // Sequences with exactly one query token: -1 = unknown, 0 = none. When not 0
  // those sequences run on the decode kernel and the prefill kernel skips them.
  int32_t single_query_seqs;
  // Key ranges (split_tiles > 0): 64-key tiles per range, the number of ranges (the last
  // one runs to the row's end) and their fp32 partials.
  int32_t split_tiles, num_ranges;
  float* part_out;                         // [num_ranges, T, H, D], unnormalized
  float* part_ml;                          // [num_ranges, T, H, 2]: reference max (log2 units), row sum
  // Balanced single-query rows (RowChunk), or null: decode_chunk_slots() results per head.
  float* row_part_out;                     // [slots, H, D]
  float* row_part_lse;                     // [slots, H]
};

struct ArgmaxArgs {
  const void* logits; int64_t row_stride;  // [rows, vocab], unit column stride
  int32_t rows, vocab;
  int32_t fp32;                            // 1: fp32 logits, 0: bf16
  int32_t vec_ok;                          // 16-byte loads cover whole rows exactly
  void* workspace;                         // argmax_workspace_bytes(rows, vocab)
  int64_t* out;                            // [rows]
};

struct NormArgs {
  const void* input; int64_t in_stride;    // [rows, n] bf16
  void* residual;    int64_t res_stride;   // [rows, n] bf16 or null; receives input + residual
  const void* weight;                      // [n], bf16 or fp32
  int32_t weight_fp32;
  void* out;         int64_t out_stride;   // [rows, n] bf16
  int32_t rows, n;
  float eps;
  int32_t vec_ok;                          // 16-byte aligned rows, n % 8 == 0
};

struct SiluArgs {
  const void* gate_up;                     // [rows, 2d] bf16, contiguous
  void* out;                               // [rows, d] bf16, contiguous
  int64_t rows;
  int32_t d;
  int32_t vec_ok;                          // 16-byte aligned, d % 8 == 0
};

struct LinearArgs {
  const void* x; int64_t x_stride;         // [m, k] bf16
  const void* w;                           // [n, k] bf16, or [2n, k] (gate rows, then up rows); contiguous
  const void* bias;                        // [n] bf16 or null
  void* out; int64_t out_stride;           // [m, n] bf16
  float* partials;                         // LinearPlan::partial_bytes
  int32_t m, n, k;
  // Set by the launcher (linear_plan):
  int32_t k_splits, row_groups, unit;
};

struct EmbedArgs {
  const int64_t* ids;                      // [rows]
  const void* table;                       // [vocab, hidden] bf16
  void* out;                               // [rows, hidden] bf16
  const int64_t* positions;                // [rows]
  const float* cos_table; const float* sin_table;  // [max_positions, head_dim]
  void* cos_out; void* sin_out;            // [rows, head_dim] bf16
  int64_t vocab, max_positions;
  int32_t rows, hidden, head_dim;
};
hipError_t embed_rows(const EmbedArgs& a, hipStream_t stream);

// How a linear layer of a few tokens runs (skinny_linear.hip).
struct LinearPlan {
  int32_t rw, kw;          // row waves x k slabs of a work-group; rw = 0: not a shape for this kernel
  int32_t k_splits;        // k ranges over work-groups (> 1: fp32 partials and a second launch)
  int32_t row_groups;      // work-groups per k range, an even split of the output columns ...
  int32_t unit;            // ... in units of 2 or 4 columns
  int64_t partial_bytes;
};
LinearPlan linear_plan(int32_t m, int32_t n, int32_t k, bool gated, bool eager);
hipError_t skinny_linear(const LinearArgs& a, bool gated, bool eager, hipStream_t stream);

hipError_t rope_kv_append(const RopeArgs& a, hipStream_t stream);
int64_t argmax_workspace_bytes(int32_t rows, int32_t vocab);
hipError_t greedy_argmax(const ArgmaxArgs& a, hipStream_t stream);
hipError_t fused_add_rms_norm(const NormArgs& a, hipStream_t stream);
hipError_t silu_mul(const SiluArgs& a, hipStream_t stream);
hipError_t paged_decode(const DecodeArgs& a, hipStream_t stream);
// The single pass with long rows cut into chunks (paged_decode.hip). The partials hold
// decode_chunk_slots() results per query head: [slots, H, D] and [slots, H].
hipError_t paged_decode_balanced(const DecodeArgs& a, hipStream_t stream);
int64_t decode_chunk_slots(int32_t batch, int32_t num_heads, int32_t num_kv_heads);
// Sets the chunking fields of a launch, and merges its chunks (RowChunk).
void decode_set_chunks(DecodeArgs& a);
hipError_t decode_merge_chunks(const DecodeArgs& a, hipStream_t stream);
// Whether a prefill batch's single-query rows (the longest and all of their pages) are
// uneven enough, and long enough beside the other work-groups' key tiles, that cutting them
// pays for the merge.
bool prefill_balance_rows(int32_t num_heads, int32_t num_kv_heads, int64_t longest, int64_t total,
                          int64_t prefill_tiles);

// How a decode launch with the caller's split plan runs (paged_decode.hip).
struct DecodePlan {
  bool single_pass;        // one split: single-pass work-groups, no workspace
  int32_t group;           // consecutive splits folded into one partial (level 2 of the merge)
  int32_t splits_per_item; // splits per streaming wave: 1, or `group` when the wave folds them
  int32_t partials;        // partial states per (row, head) in the workspace
  bool fold_in_reduce;     // the reduce folds the per-split partials into groups
  bool pair;               // one split or group per work-group of two waves (two states each)
  bool quad;               // (with pair) work-groups of four waves: splits of at most 64 pages, long groups
  bool live_first;         // units with live pages before the empty ones (find_live_unit)
};
DecodePlan decode_plan(int32_t batch, int32_t num_kv_heads, int32_t head_dim, int32_t num_splits,
                       int32_t blocks_per_split);
// Column groups of a decode launch: its KV heads, each cut into ceil(G / 16)
// groups of at most 16 query heads (one MFMA tile of columns) when G > 16.
inline int64_t decode_col_groups(const DecodeArgs& a) {
  const int G = a.num_heads / a.num_kv_heads;
  return (int64_t)a.num_kv_heads * ((G + 15) / 16);
}
// Partial states per (row, head) the decode workspace holds: the most any
// plan of these splits writes, independent of the tuning knobs.
int32_t decode_partials(int32_t batch, int32_t num_kv_heads, int32_t num_splits, int32_t blocks_per_split);

// Process-wide tuning switches (bvllm_set_tuning). Knob values: 0 = default.
enum TuneKnob {
  kTuneDecodeSplitMode = 0,         // 1: one wave per split, 2: one wave per group of splits, 3: two
                                    // waves per group, 4: two waves per split also for splits of at most
                                    // 64 pages, 5: four waves per group (same bits); default: decode_plan
  kTunePrefillBlocksPerWg = 1,      // n > 0: prefill column blocks per work-group when the table allows it
  kTuneDecodeOrder = 2,             // 1: split units fastest in the streaming wave numbering (same bits)
  kTuneDecodeSinglePassStream = 3,  // 1: single-pass launches on streaming waves too (same bits)
  kTuneDecodeCached = 4,            // 1: streaming page loads without the nontemporal hint (same bits)
  kTuneAppendChunks = 5,            // 1: aligned appends on the per-chunk kernel (same bits, NaN payloads aside)
  kTunePrefillShortGrid = 6,        // 1: short prefill grids on the single key walk instead of the key split;
                                    // 2: on 64-column blocks also with at most one per CU
  kTuneKnobs = 7,
};
int tuning(int knob);
int set_tuning(int knob, int value);
hipError_t paged_prefill(const PrefillArgs& a, hipStream_t stream);
// Key ranges of a prefill launch: tiles per range (0: no split) for the batch's shape
// (key_tiles: 64-key tiles its 128-column blocks walk per KV head, longest_tiles: those of
// its longest sequence of more than one query; < 0 if unknown).
int32_t prefill_split_tiles(const PrefillArgs& a, int64_t key_tiles, int64_t longest_tiles);
// Ranges of split_tiles tiles that hold keys: those of the longest sequence of more than one
// query, or of the table where its length is unknown (longest_tiles < 0).
inline int32_t prefill_ranges(int32_t max_blocks, int32_t split_tiles, int64_t longest_tiles) {
  int64_t tiles = ((int64_t)max_blocks + 3) / 4;
  if (longest_tiles >= 0 && longest_tiles < tiles) tiles = longest_tiles > 0 ? longest_tiles : 1;
  return (int32_t)((tiles + split_tiles - 1) / split_tiles);
}
// fp32 values of the partials of num_ranges ranges.
inline int64_t prefill_range_floats(int32_t num_ranges, int32_t num_tokens, int32_t num_heads, int32_t head_dim) {
  return (int64_t)num_ranges * num_tokens * num_heads * (head_dim + 2);
}
// Compute units of the current device (cached per device).
int device_cus();

}  // namespace bvllm
