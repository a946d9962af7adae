// What a decode step needs before its first layer, from device-resident tables: the batch's block
// tables, the slots and lengths of its new tokens; and the rotary tables of any step's tokens.
//
// Reference semantics: engine/kv_cache.py:592-609 (tables, write positions, lengths) and
// engine/model.py:205-213 (cos / sin). In a captured step these were a dozen torch launches of 2 to 4
// us each and a dozen more for cos and sin, every one of them over a few KB: launches are all they
// cost. Here the step takes two (the journal has to land before a row is read), the rotary tables
// one.
#include "mip_common.h"

namespace mip {
namespace {

__global__ __launch_bounds__(256) void journal_kernel(int32_t* rows, const int64_t* flat, const int64_t* block, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) rows[flat[i]] = static_cast<int32_t>(block[i]);
}

// One workgroup per sequence.
__global__ __launch_bounds__(256) void step_rows_kernel(const int32_t* rows, int64_t row_stride, const int64_t* row_ids,
                                                        const int64_t* positions, int32_t* tables, int64_t table_stride,
                                                        int n_blocks, int64_t* slots, int32_t* lens, int log2_bs) {
  const int b = blockIdx.x;
  const int32_t* src = rows + row_ids[b] * row_stride;
  int32_t* dst = tables + b * table_stride;
  if (threadIdx.x == 0) {
    const int64_t p = positions[b];
    slots[b] = (static_cast<int64_t>(src[p >> log2_bs]) << log2_bs) + (p & ((1 << log2_bs) - 1));
    lens[b] = static_cast<int32_t>(p) + 1;
  }
  for (int i = threadIdx.x; i < n_blocks; i += 256) dst[i] = src[i];
}

// cos and sin of position * theta^(-2 j / D) for j < D / 2, both halves of a row alike. The steps and
// their fp32 roundings are torch's (exponent, pow, reciprocal, angle, then cos and sin), which divides
// the exponent by D as a product with 1 / D: another value where D is no power of two.
template <int DT>
__global__ __launch_bounds__(256) void rope_tables_kernel(typename Elem<DT>::S* cos, typename Elem<DT>::S* sin,
                                                          const int64_t* positions, uint32_t total, uint32_t half,
                                                          float theta) {
  const float inv_d = 1.0f / static_cast<float>(2 * half);
  for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < total; i += gridDim.x * 256u) {
    const uint32_t tok = i / half, j = i - tok * half;
    const float e = static_cast<float>(j) * 2.0f * inv_d;
    const float inv = 1.0f / powf(theta, e);
    const float ang = static_cast<float>(positions[tok]) * inv;
    const auto c = from_f32<DT>(cosf(ang)), s = from_f32<DT>(sinf(ang));
    const int64_t at = static_cast<int64_t>(tok) * 2 * half + j;
    cos[at] = c;
    cos[at + half] = c;
    sin[at] = s;
    sin[at + half] = s;
  }
}

}  // namespace
}  // namespace mip

using namespace mip;

extern "C" int mip_decode_prepare(int32_t* rows, int64_t row_stride, const int64_t* journal_flat,
                                  const int64_t* journal_block, int32_t n_journal, const int64_t* row_ids,
                                  const int64_t* positions, int32_t* tables, int64_t table_stride, int32_t n_blocks,
                                  int64_t* slot_mapping, int32_t* context_lens, int32_t batch, int32_t block_size,
                                  void* stream) {
  if (n_journal < 0 || n_blocks <= 0 || batch < 0 || !is_pow2(block_size) || block_size > (1 << 30)) return MIP_EINVAL;
  if (row_stride < n_blocks || table_stride < n_blocks) return MIP_EINVAL;
  if (!rows || (n_journal > 0 && (!journal_flat || !journal_block))) return MIP_EINVAL;
  if (batch > 0 && (!row_ids || !positions || !tables || !slot_mapping || !context_lens)) return MIP_EINVAL;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (n_journal > 0)
    hipLaunchKernelGGL(journal_kernel, dim3((n_journal + 255) / 256), dim3(256), 0, s, rows, journal_flat, journal_block,
                       n_journal);
  if (batch > 0)
    hipLaunchKernelGGL(step_rows_kernel, dim3(batch), dim3(256), 0, s, rows, row_stride, row_ids, positions, tables,
                       table_stride, n_blocks, slot_mapping, context_lens, ilog2_exact(block_size));
  return status_from_hip(hipGetLastError());
}

extern "C" int mip_rope_tables(void* cos, void* sin, const int64_t* positions, int32_t n_tokens, int32_t head_dim,
                               float theta, int32_t dtype, void* stream) {
  if (dtype != MIP_F32 && dtype != MIP_F16 && dtype != MIP_BF16) return MIP_EINVAL;
  if (n_tokens < 0 || head_dim <= 0 || head_dim % 2) return MIP_EINVAL;
  if (n_tokens == 0) return MIP_OK;
  if (!cos || !sin || !positions) return MIP_EINVAL;
  const int64_t total = static_cast<int64_t>(n_tokens) * (head_dim / 2);
  if (total >= (int64_t{1} << 31)) return MIP_EUNSUPPORTED;
  const int64_t want = (total + 255) / 256;
  const dim3 grid(static_cast<unsigned>(want < 65536 ? want : 65536)), block(256);
  const uint32_t n = static_cast<uint32_t>(total), half = static_cast<uint32_t>(head_dim / 2);
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case MIP_F32:
      hipLaunchKernelGGL((rope_tables_kernel<MIP_F32>), grid, block, 0, s, static_cast<float*>(cos), static_cast<float*>(sin),
                         positions, n, half, theta);
      break;
    case MIP_F16:
      hipLaunchKernelGGL((rope_tables_kernel<MIP_F16>), grid, block, 0, s, static_cast<uint16_t*>(cos),
                         static_cast<uint16_t*>(sin), positions, n, half, theta);
      break;
    default:
      hipLaunchKernelGGL((rope_tables_kernel<MIP_BF16>), grid, block, 0, s, static_cast<uint16_t*>(cos),
                         static_cast<uint16_t*>(sin), positions, n, half, theta);
  }
  return status_from_hip(hipGetLastError());
}
