// Inputs of a captured decode step, staged in one launch.
//
// A replayed graph reads fixed buffers.  Refreshing them takes, per step, the
// q / k / v rows of every layer, their zeroed padding rows, and the slots,
// lengths and block tables padded with the scratch block
// (nanovllm/engine/model_runner.py:864-869): twelve copies and fills as torch
// operators, each a launch of 2-4 us for kilobytes.  Here one workgroup per
// (layer, bucket row) moves that row's q, k and v and one more workgroup per
// bucket row writes its slot, length and table row.  A replayed step of 8
// layers x 13 rows (32 q / 4 kv heads, contexts 300-3001): 214 us with the
// operators and a copy node per layer for the outputs, 177 us with this
// launch and the decode writing the runner's output buffer.
#include "kvc_internal.h"

namespace kvc {
namespace {

constexpr int kThreads = 256;

struct StageRows {
  const char* src;
  char* dst;
  int64_t src_layer, src_row;  // bytes
  int64_t dst_layer;           // bytes; destination rows are dense
  int vecs;                    // 16-byte vectors of a row
};

struct StageArgs {
  StageRows rows[3];  // q, k, v
  int layers, batch, bucket;
  const void* slots;
  const void* lens;
  int slots64, lens64;
  const int32_t* tables;
  int64_t tables_stride;
  int tables_cols, dst_cols;
  int32_t* slots_dst;
  int32_t* lens_dst;
  int32_t* tables_dst;
  int scratch_slot, scratch_block;
};

__device__ __forceinline__ int32_t index_at(const void* p, int wide, int i) {
  return wide ? int32_t(static_cast<const int64_t*>(p)[i]) : static_cast<const int32_t*>(p)[i];
}

// Latency-bound at decode batches (8 layers x 16 rows of 10 KB: 1.3 MB).
__global__ void __launch_bounds__(kThreads) stage_decode_kernel(StageArgs a) {
  const int rows = a.layers * a.bucket;
  int w = int(blockIdx.x);
  if (w < rows) {
    const int layer = w / a.bucket;
    const int row = w - layer * a.bucket;
    const bool live = row < a.batch;
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      const StageRows& r = a.rows[t];
      const u32x4_t* s =
          reinterpret_cast<const u32x4_t*>(r.src + layer * r.src_layer + row * r.src_row);
      u32x4_t* d = reinterpret_cast<u32x4_t*>(r.dst + layer * r.dst_layer) + int64_t(row) * r.vecs;
      for (int i = threadIdx.x; i < r.vecs; i += kThreads)
        d[i] = live ? s[i] : u32x4_t{0u, 0u, 0u, 0u};
    }
    return;
  }
  const int row = w - rows;
  const bool live = row < a.batch;
  if (threadIdx.x == 0) {
    a.slots_dst[row] = live ? index_at(a.slots, a.slots64, row) : a.scratch_slot;
    a.lens_dst[row] = live ? index_at(a.lens, a.lens64, row) : 1;
  }
  for (int c = threadIdx.x; c < a.dst_cols; c += kThreads)
    a.tables_dst[int64_t(row) * a.dst_cols + c] =
        live && c < a.tables_cols ? a.tables[row * a.tables_stride + c] : a.scratch_block;
}

}  // namespace
}  // namespace kvc

using namespace kvc;

extern "C" int kvc_stage_decode(const void* q, int64_t q_layer_stride, int64_t q_row_stride,
                                const void* k, int64_t k_layer_stride, int64_t k_row_stride,
                                const void* v, int64_t v_layer_stride, int64_t v_row_stride,
                                int64_t q_row_bytes, int64_t kv_row_bytes, int64_t layers,
                                int64_t batch, int64_t bucket, int64_t dst_rows,
                                const void* slot_mapping, int slot_index_bytes,
                                const void* context_lens, int lens_index_bytes,
                                const int32_t* block_tables, int64_t bt_stride, int64_t bt_cols,
                                void* q_dst, void* k_dst, void* v_dst, int32_t* slots_dst,
                                int32_t* lens_dst, int32_t* tables_dst, int64_t dst_cols,
                                int32_t scratch_slot, int32_t scratch_block,
                                kvc_stream_t stream) {
  clear_error();
  KVC_REQUIRE(layers > 0 && batch >= 0 && bucket >= batch && dst_rows >= bucket && bucket > 0 &&
                  bt_cols >= 0 && dst_cols >= bt_cols && q_row_bytes > 0 && kv_row_bytes > 0,
              KVC_ERR_VALUE, "stage_decode: bad shape");
  KVC_REQUIRE((layers + 1) * bucket < (int64_t(1) << 31) && dst_cols < (int64_t(1) << 31) &&
                  q_row_bytes < (int64_t(1) << 31) && kv_row_bytes < (int64_t(1) << 31),
              KVC_ERR_VALUE, "stage_decode: launch too large");
  KVC_REQUIRE((slot_index_bytes == 4 || slot_index_bytes == 8) &&
                  (lens_index_bytes == 4 || lens_index_bytes == 8),
              KVC_ERR_VALUE, "stage_decode: indices are int32 or int64");
  KVC_REQUIRE(slots_dst != nullptr && lens_dst != nullptr &&
                  (tables_dst != nullptr || dst_cols == 0) &&
                  (batch == 0 || (slot_mapping != nullptr && context_lens != nullptr)) &&
                  (batch == 0 || bt_cols == 0 || block_tables != nullptr),
              KVC_ERR_VALUE, "stage_decode: null slots, lengths or tables");
  const void* ptrs[] = {q, k, v, q_dst, k_dst, v_dst};
  for (const void* p : ptrs)
    KVC_REQUIRE(p != nullptr && reinterpret_cast<uintptr_t>(p) % 16 == 0, KVC_ERR_ASSERT,
                "stage_decode: buffers must be 16-byte aligned");
  const int64_t strides[] = {q_layer_stride, q_row_stride, k_layer_stride, k_row_stride,
                             v_layer_stride, v_row_stride, q_row_bytes,    kv_row_bytes};
  for (int64_t s : strides)
    KVC_REQUIRE(s % 16 == 0, KVC_ERR_ASSERT, "stage_decode: strides must be multiples of 16 bytes");
  StageArgs a{};
  a.rows[0] = {static_cast<const char*>(q), static_cast<char*>(q_dst), q_layer_stride,
               q_row_stride, dst_rows * q_row_bytes, int(q_row_bytes / 16)};
  a.rows[1] = {static_cast<const char*>(k), static_cast<char*>(k_dst), k_layer_stride,
               k_row_stride, dst_rows * kv_row_bytes, int(kv_row_bytes / 16)};
  a.rows[2] = {static_cast<const char*>(v), static_cast<char*>(v_dst), v_layer_stride,
               v_row_stride, dst_rows * kv_row_bytes, int(kv_row_bytes / 16)};
  a.layers = int(layers);
  a.batch = int(batch);
  a.bucket = int(bucket);
  a.slots = slot_mapping;
  a.lens = context_lens;
  a.slots64 = slot_index_bytes == 8;
  a.lens64 = lens_index_bytes == 8;
  a.tables = block_tables;
  a.tables_stride = bt_stride;
  a.tables_cols = int(bt_cols);
  a.dst_cols = int(dst_cols);
  a.slots_dst = slots_dst;
  a.lens_dst = lens_dst;
  a.tables_dst = tables_dst;
  a.scratch_slot = scratch_slot;
  a.scratch_block = scratch_block;
  stage_decode_kernel<<<unsigned((layers + 1) * bucket), kThreads, 0, as_stream(stream)>>>(a);
  return check_launch("stage_decode");
}
