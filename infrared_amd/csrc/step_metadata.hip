// A step's device metadata from the scheduler's lists in one launch: the host
// packs block tables, cached lengths (and last tokens) into one staging buffer,
// one copy moves it, and these kernels expand it to what the attention seam
// reads (infrared/engine/cuda_graph.py:105-155, infrared/engine/paged_engine.py:
// 303-314, 461-516, 621-638).
//
// Bound by launches, not by the bytes they write: the same tensors built from
// elementwise library calls took some 25 launches a decode step and 15 a prefill
// step, each 2-5 us of device time and about as much of the host's. A 24-layer
// fp32 graph step of 8 sequences, metadata included: 236 us against 466; 12 short
// prompts through 8 layers: 369 against 557.
#include "common.hpp"
#include "status.hpp"

namespace ir {
namespace {

struct DecodeInputsArgs {
  const int64_t* rows;    // [num_rows][2]: cached tokens, last token
  const int32_t* tables;  // [num_rows][width]
  int num_rows, bucket, width, bs, t_max;
  uint32_t mask_low;  // bits of the mask dtype's finfo.min
  int64_t* ids;
  int64_t* positions;
  int64_t* write_slots;
  int64_t* gather_slots;  // [bucket][t_max]
  void* mask;             // [bucket][t_max]
  int32_t* block_tables;  // [bucket][width]
  int32_t* context_lens;
};

// One thread per (row, key): its gather slot and mask element; the row's first
// threads also copy its block table, thread 0 its scalars. Rows past num_rows
// repeat row 0.
template <typename MaskBits>
__global__ __launch_bounds__(256) void decode_inputs_kernel(DecodeInputsArgs a) {
  const int row = blockIdx.y;
  const int src = row < a.num_rows ? row : 0;
  const int64_t cached = a.rows[2 * src];
  const int32_t* bt = a.tables + (int64_t)src * a.width;
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p < a.t_max) {
    const bool in = p <= cached;
    const int blk = p / a.bs;  // < width: the tables cover t_max tokens
    const int64_t i = (int64_t)row * a.t_max + p;
    a.gather_slots[i] = in ? (int64_t)bt[blk] * a.bs + (p - blk * a.bs) : 0;
    ((MaskBits*)a.mask)[i] = in ? (MaskBits)0 : (MaskBits)a.mask_low;
  }
  if (p < a.width) a.block_tables[(int64_t)row * a.width + p] = bt[p];
  if (p == 0) {
    const int blk = (int)(cached / a.bs);
    a.ids[row] = a.rows[2 * src + 1];
    a.positions[row] = cached;
    a.write_slots[row] = (int64_t)bt[blk] * a.bs + (cached - (int64_t)blk * a.bs);
    a.context_lens[row] = (int32_t)cached + 1;
  }
}

// One thread per packed token: its sequence by bisection of the chunk starts
// (an empty chunk owns no token), then its position's slot.
__global__ __launch_bounds__(256) void packed_write_slots_kernel(const int32_t* tables, int64_t stride, int width,
                                                                 const int32_t* cached, const int32_t* cu,
                                                                 int num_seqs, int total, int bs, int64_t* slots) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= total) return;
  int lo = 0, hi = num_seqs - 1;  // the last sequence starting at or before t
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (cu[mid] <= t)
      lo = mid;
    else
      hi = mid - 1;
  }
  const int pos = cached[lo] + (t - cu[lo]);
  const int blk = pos / bs;
  slots[t] = pos >= 0 && blk < width ? (int64_t)tables[lo * stride + blk] * bs + (pos - blk * bs) : -1;
}

}  // namespace
}  // namespace ir

using namespace ir;

extern "C" int ir_decode_inputs(const void* staging, int num_rows, int bucket, int width, int block_size, int t_max,
                                int mask_dtype, int64_t* ids, int64_t* positions, int64_t* write_slots,
                                int64_t* gather_slots, void* mask, int32_t* block_tables, int32_t* context_lens,
                                ir_stream_t stream) {
  IR_REQUIRE(dtype_bytes(mask_dtype) > 0, "ir_decode_inputs: unknown mask dtype %d", mask_dtype);
  IR_REQUIRE(num_rows > 0 && bucket >= num_rows && bucket < 65536 && block_size > 0 && t_max > 0 &&
                 (int64_t)width * block_size >= t_max,
             "ir_decode_inputs: bad sizes");
  IR_REQUIRE(staging && ids && positions && write_slots && gather_slots && mask && block_tables && context_lens,
             "ir_decode_inputs: null pointer");
  IR_REQUIRE(((uintptr_t)staging & 7u) == 0, "ir_decode_inputs: staging must be 8-byte aligned");
  DecodeInputsArgs a;
  a.rows = (const int64_t*)staging;
  a.tables = (const int32_t*)(a.rows + 2 * (int64_t)num_rows);
  a.num_rows = num_rows;
  a.bucket = bucket;
  a.width = width;
  a.bs = block_size;
  a.t_max = t_max;
  a.mask_low = mask_dtype == IR_DTYPE_F32 ? 0xff7fffffu : mask_dtype == IR_DTYPE_BF16 ? 0xff7fu : 0xfbffu;
  a.ids = ids;
  a.positions = positions;
  a.write_slots = write_slots;
  a.gather_slots = gather_slots;
  a.mask = mask;
  a.block_tables = block_tables;
  a.context_lens = context_lens;
  const int n = t_max > width ? t_max : width;
  const dim3 grid((unsigned)((n + 255) / 256), (unsigned)bucket);
  if (mask_dtype == IR_DTYPE_F32)
    hipLaunchKernelGGL((decode_inputs_kernel<uint32_t>), grid, dim3(256), 0, (hipStream_t)stream, a);
  else
    hipLaunchKernelGGL((decode_inputs_kernel<uint16_t>), grid, dim3(256), 0, (hipStream_t)stream, a);
  return check_launch("ir_decode_inputs");
}

extern "C" int ir_packed_write_slots(const int32_t* block_tables, int64_t bt_stride, int width,
                                     const int32_t* num_cached, const int32_t* cu_seqlens_q, int num_seqs, int total,
                                     int block_size, int64_t* write_slots, ir_stream_t stream) {
  IR_REQUIRE(width >= 0 && num_seqs >= 0 && total >= 0 && block_size > 0, "ir_packed_write_slots: bad sizes");
  if (total == 0) return ok();
  IR_REQUIRE(num_seqs > 0 && block_tables && num_cached && cu_seqlens_q && write_slots,
             "ir_packed_write_slots: null pointer");
  hipLaunchKernelGGL(packed_write_slots_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, block_tables, bt_stride, width, num_cached, cu_seqlens_q, num_seqs, total,
                     block_size, write_slots);
  return check_launch("ir_packed_write_slots");
}
