// A model's input rows in one launch: the embedding row of every token and the RoPE
// cos/sin rows of every position (reference: embed_tokens and rotary_emb of
// babyvllm/models/qwen2.py:109-118, tables of babyvllm/layers/rotary.py:17-32).
//
// Latency-bound at decode sizes (16 tokens read 115 KB): torch ran an index_select
// that walks a small index serially and a gather and a cast for each table, five
// dependent launches of 4.4 to 15.4 us in a captured step (33.6 us in all at 16 tokens
// of 3584); here every 16-byte chunk is one thread of one launch (4.6 us).
#include "bvllm_device.h"
#include "bvllm_abi_internal.h"

namespace bvllm {

namespace {

constexpr uint32_t kNaN2 = 0x7fc07fc0u;  // two bf16 NaNs

// Threads [0, rows·hidden/8): 8 embedding elements each; then [rows·d/8] threads: 8
// elements of a cos row and of a sin row each.
__global__ __launch_bounds__(256) void embed_rows_kernel(EmbedArgs a) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int hc = a.hidden / 8, dc = a.head_dim / 8;
  const int64_t embed_items = (int64_t)a.rows * hc;
  if (t < embed_items) {
    const int64_t row = t / hc;
    const int c = (int)(t - row * hc);
    const int64_t id = a.ids[row];
    // An id outside the table gives a row of NaN (there is nothing to read).
    uint4 v = make_uint4(kNaN2, kNaN2, kNaN2, kNaN2);
    if (id >= 0 && id < a.vocab) v = ld16(reinterpret_cast<const uint16_t*>(a.table) + id * a.hidden + 8 * c);
    st16(reinterpret_cast<uint16_t*>(a.out) + row * a.hidden + 8 * c, v);
    return;
  }
  const int64_t u = t - embed_items;
  if (u >= (int64_t)a.rows * dc) return;
  const int64_t row = u / dc;
  const int c = (int)(u - row * dc);
  int64_t p = a.positions[row];
  if (p < 0) p += a.max_positions;  // counted from the table's end, as torch indexing does
  uint4 cv = make_uint4(kNaN2, kNaN2, kNaN2, kNaN2), sv = cv;
  if (p >= 0 && p < a.max_positions) {
    const float* cs = a.cos_table + p * a.head_dim + 8 * c;
    const float* sn = a.sin_table + p * a.head_dim + 8 * c;
    const f32x4_t c0 = *reinterpret_cast<const f32x4_t*>(cs), c1 = *reinterpret_cast<const f32x4_t*>(cs + 4);
    const f32x4_t s0 = *reinterpret_cast<const f32x4_t*>(sn), s1 = *reinterpret_cast<const f32x4_t*>(sn + 4);
    cv = make_uint4(pack_bf16x2_hw(c0[0], c0[1]), pack_bf16x2_hw(c0[2], c0[3]), pack_bf16x2_hw(c1[0], c1[1]),
                    pack_bf16x2_hw(c1[2], c1[3]));
    sv = make_uint4(pack_bf16x2_hw(s0[0], s0[1]), pack_bf16x2_hw(s0[2], s0[3]), pack_bf16x2_hw(s1[0], s1[1]),
                    pack_bf16x2_hw(s1[2], s1[3]));
  }
  st16(reinterpret_cast<uint16_t*>(a.cos_out) + row * a.head_dim + 8 * c, cv);
  st16(reinterpret_cast<uint16_t*>(a.sin_out) + row * a.head_dim + 8 * c, sv);
}

}  // namespace

hipError_t embed_rows(const EmbedArgs& a, hipStream_t stream) {
  const int64_t items = (int64_t)a.rows * (a.hidden / 8 + a.head_dim / 8);
  const int64_t blocks = (items + 255) / 256;
  if (blocks > 0x7fffffff) return hipErrorInvalidValue;
  hipLaunchKernelGGL(embed_rows_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, a);
  return hipGetLastError();
}

}  // namespace bvllm
