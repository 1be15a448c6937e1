// Decode-step metadata on the device (replaces the Triton
// _prepare_decode_kernel of engine/decode_init.py:6-65).
//
// One lane per scheduled sequence, written as the closed form of
// engine/decode_init.py:29-36: the new token sits at position seq_len-1, the
// context (including it) is seq_len tokens, and its cache slot is offset
// (seq_len-1) % block_size of the sequence's last block.  input_ids gathers
// the last sampled token through the persistent batch-slot indirection.
#include "nq_device.hpp"

namespace nq {
namespace {

__global__ __launch_bounds__(256) void prepare_decode_kernel(
    const int64_t *__restrict__ sampled_token_ids, const int64_t *__restrict__ batch_slots,
    const int32_t *__restrict__ seq_lens, const int32_t *__restrict__ last_block_ids,
    int64_t *__restrict__ input_ids, int64_t *__restrict__ positions, int32_t *__restrict__ context_lens,
    int32_t *__restrict__ slot_mapping, int num_seqs, int block_size) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= num_seqs) return;
  const int32_t len = seq_lens[i];
  const int32_t last = last_block_ids[i];
  if (sampled_token_ids != nullptr && input_ids != nullptr)
    input_ids[i] = sampled_token_ids[batch_slots[i]];
  positions[i] = static_cast<int64_t>(len) - 1;
  context_lens[i] = len;
  slot_mapping[i] = last * block_size + (len - 1) % block_size;
}

// The static inputs of a captured decode step from a batch's own tensors
// (engine/model_runner.py:325-334), in one launch: blocks 0 .. blocks_rows - 1 a
// row per lane (rows past the batch are padding: slot -1, context 0, as the
// reference's fills leave them), the rest the block table.  Launch-bound: in
// place of seven copies and fills ahead of the replay (a captured step of 8
// layers 220 -> 208 us).
struct StageArgs {
  const int64_t *input_ids, *positions;
  const int32_t *slot_mapping, *context_lens, *block_tables;
  int64_t bt_stride, to_bt_stride;
  int64_t *to_input_ids, *to_positions;
  int32_t *to_slot_mapping, *to_context_lens, *to_block_tables;
  int batch, rows, width, row_blocks;
};
__global__ __launch_bounds__(256) void stage_decode_kernel(const StageArgs a) {
  if (static_cast<int>(blockIdx.x) < a.row_blocks) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= a.rows) return;
    const bool live = i < a.batch;
    if (live) {
      a.to_input_ids[i] = a.input_ids[i];
      a.to_positions[i] = a.positions[i];
    }
    a.to_slot_mapping[i] = live ? a.slot_mapping[i] : -1;
    a.to_context_lens[i] = live ? a.context_lens[i] : 0;
    return;
  }
  const int64_t n = static_cast<int64_t>(a.batch) * a.width;
  for (int64_t e = static_cast<int64_t>(blockIdx.x - a.row_blocks) * 256 + threadIdx.x; e < n;
       e += static_cast<int64_t>(gridDim.x - a.row_blocks) * 256) {
    const int64_t r = e / a.width, c = e - r * a.width;
    a.to_block_tables[r * a.to_bt_stride + c] = a.block_tables[r * a.bt_stride + c];
  }
}

}  // namespace
}  // namespace nq

using namespace nq;

extern "C" int nq_stage_decode(const int64_t *input_ids, const int64_t *positions, const int32_t *slot_mapping,
                               const int32_t *context_lens, const int32_t *block_tables, int64_t bt_stride,
                               int batch, int width, int64_t *to_input_ids, int64_t *to_positions,
                               int32_t *to_slot_mapping, int32_t *to_context_lens, int32_t *to_block_tables,
                               int64_t to_bt_stride, int rows, void *stream) {
  if (batch < 0 || rows < batch || width < 0 || bt_stride < 0 || to_bt_stride < width)
    return fail(NQ_EINVAL, "stage_decode: bad sizes (batch %d of %d rows, width %d)", batch, rows, width);
  if (rows == 0) return NQ_OK;
  if (!to_slot_mapping || !to_context_lens || (batch > 0 && (!input_ids || !positions || !slot_mapping ||
      !context_lens || !to_input_ids || !to_positions)) || (batch > 0 && width > 0 && (!block_tables || !to_block_tables)))
    return fail(NQ_EINVAL, "stage_decode: null pointer");
  StageArgs a{input_ids, positions, slot_mapping, context_lens, block_tables, bt_stride, to_bt_stride, to_input_ids,
              to_positions, to_slot_mapping, to_context_lens, to_block_tables, batch, rows, width, (rows + 255) / 256};
  const int64_t n = static_cast<int64_t>(batch) * width;
  const int table_blocks = static_cast<int>(n < 1024 * 256 ? (n + 255) / 256 : 1024);
  stage_decode_kernel<<<a.row_blocks + table_blocks, 256, 0, static_cast<hipStream_t>(stream)>>>(a);
  return check_launch("stage_decode");
}

extern "C" int nq_prepare_decode(const int64_t *sampled_token_ids, const int64_t *batch_slots,
                                 const int32_t *seq_lens, const int32_t *last_block_ids, int64_t *input_ids,
                                 int64_t *positions, int32_t *context_lens, int32_t *slot_mapping,
                                 int num_seqs, int block_size, void *stream) {
  if (num_seqs == 0) return NQ_OK;
  if (num_seqs < 0 || block_size <= 0) return fail(NQ_EINVAL, "prepare_decode: bad sizes");
  if (!seq_lens || !last_block_ids || !positions || !context_lens || !slot_mapping)
    return fail(NQ_EINVAL, "prepare_decode: null pointer");
  if ((sampled_token_ids == nullptr) != (input_ids == nullptr) || (sampled_token_ids && !batch_slots))
    return fail(NQ_EINVAL, "prepare_decode: sampled_token_ids, batch_slots and input_ids go together");
  const int threads = 256;
  const int blocks = (num_seqs + threads - 1) / threads;
  prepare_decode_kernel<<<blocks, threads, 0, static_cast<hipStream_t>(stream)>>>(
      sampled_token_ids, batch_slots, seq_lens, last_block_ids, input_ids, positions, context_lens,
      slot_mapping, num_seqs, block_size);
  return check_launch("prepare_decode");
}
