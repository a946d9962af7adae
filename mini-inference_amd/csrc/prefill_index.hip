// Where a packed prefill step's tokens go: their positions and pool slots, from the step's row
// offsets, cached lengths and block tables.
//
// Reference semantics: engine/kv_cache.py:562-573 (write_index) and :230-250 (positions), which
// build these on the host: token i of sequence s has position p = ctx_start[s] + i and slot
// table[s][p / block_size] * block_size + p % block_size; the last token of s is packed row
// cu_q[s + 1] - 1.
//
// The tables (a few KB) are on the device anyway; the two index arrays are 16 bytes per token,
// so making them here saves the host their construction (0.3 ms for 17,000 tokens of 64
// sequences in numpy) and most of the step's upload. Bound by the launch: two dependent reads
// and 16 bytes written per token, one workgroup per 256 tokens of a sequence.
#include "mip_common.h"

namespace mip {
namespace {

__global__ __launch_bounds__(256) void prefill_index_kernel(int64_t* positions, int64_t* slots, int64_t* last,
                                                            const int32_t* cu_q, const int32_t* ctx_start,
                                                            const int32_t* tables, int64_t bt_stride, int chunks,
                                                            int log2_bs) {
  const int s = blockIdx.x / chunks, i = (blockIdx.x - s * chunks) * 256 + threadIdx.x;
  const int r0 = cu_q[s], n = cu_q[s + 1] - r0;
  if (i == 0) last[s] = r0 + n - 1;
  if (i >= n) return;
  const int p = ctx_start[s] + i;
  const int64_t blk = tables[s * bt_stride + (p >> log2_bs)];
  positions[r0 + i] = p;
  slots[r0 + i] = (blk << log2_bs) + (p & ((1 << log2_bs) - 1));
}

}  // namespace
}  // namespace mip

using namespace mip;

extern "C" int mip_prefill_index(int64_t* positions, int64_t* slot_mapping, int64_t* last_index, const int32_t* cu_q,
                                 const int32_t* ctx_start, const int32_t* block_tables, int64_t bt_stride,
                                 int32_t num_seqs, int32_t max_q_len, int32_t block_size, void* stream) {
  if (num_seqs < 0 || max_q_len < 0 || !is_pow2(block_size) || bt_stride < 0) return MIP_EINVAL;
  if (num_seqs == 0) return MIP_OK;
  if (!last_index || !cu_q || !ctx_start || !block_tables || (max_q_len > 0 && (!positions || !slot_mapping)))
    return MIP_EINVAL;
  const int64_t chunks = max_q_len > 0 ? (static_cast<int64_t>(max_q_len) + 255) / 256 : 1;
  if (chunks * num_seqs >= (int64_t{1} << 31)) return MIP_EINVAL;
  hipLaunchKernelGGL(prefill_index_kernel, dim3(static_cast<unsigned>(chunks * num_seqs)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), positions, slot_mapping, last_index, cu_q, ctx_start, block_tables,
                     bt_stride, static_cast<int>(chunks), ilog2_exact(block_size));
  return status_from_hip(hipGetLastError());
}
