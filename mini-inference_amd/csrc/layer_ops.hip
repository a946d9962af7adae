// The elementwise stretches of a decoder layer, one launch each: residual add + RMS norm, and
// SiLU(gate) * up.
//
// Reference semantics (engine/model.py's RMSNorm, DecoderLayer and MLP, op by op in torch):
//     s   = x + delta                                        rounded to the dtype
//     out = weight * (s.float() * rsqrt(mean(s.float()^2) + eps)).to(dtype)
//     act = silu(gate) * up                                  silu in fp32, rounded, then * up
// Every intermediate that torch stores in the dtype is rounded to it here too, and the sums and
// products in between are fp32, so the values differ from torch's only by the order of the row
// sum (and the last bit of rsqrt / exp).
//
// What bounds them: bytes at many rows (x, delta read once, s and out written once), the launch
// and one memory round trip at few. torch runs seven kernels per norm plus the add, and three
// for the activation. A row stays in registers between its sum and its scaling, so nothing is
// read twice: one wavefront per row up to 256 16-byte chunks (no barrier, no LDS; 4 rows per
// workgroup), four wavefronts per row above that, since one lane would otherwise hold more
// than 4 chunks of x and of delta and the row's loads would queue on a single wavefront.
//
// Measured at the 0.5B widths, bf16: 3,924 rows, add + norm 9.2 us (28 MB), norm alone 5.6, gating
// 22.4 us (115 MB, 5.1 TB/s), where torch's elementwise kernels of one layer took about 150 us; at 8
// rows 3.8 to 4.0 us each, the launch (torch: 7 launches of 2 to 5 us per norm). One row per
// 64-thread workgroup at 256 rows: 5.0 us, no different from 4 rows per workgroup.
#include "mip_common.h"

namespace mip {
namespace {

// The elements of one 16-byte chunk as fp32.
template <int DT, int N> __device__ __forceinline__ void unpack(const uint4& c, float (&f)[N]) {
  typename Elem<DT>::S s[N];
  __builtin_memcpy(s, &c, 16);
#pragma unroll
  for (int e = 0; e < N; ++e) f[e] = widen<DT>(s[e]);
}
template <int DT, int N> __device__ __forceinline__ uint4 pack(const float (&f)[N]) {
  typename Elem<DT>::S s[N];
#pragma unroll
  for (int e = 0; e < N; ++e) s[e] = from_f32<DT>(f[e]);
  uint4 c;
  __builtin_memcpy(&c, s, 16);
  return c;
}

// W wavefronts per row, NC chunks per lane, row of `chunks` 16-byte chunks (<= 64 * W * NC).
template <int DT, int W, int NC, bool ADD>
__global__ __launch_bounds__(256) void add_rms_norm_kernel(const uint4* x, const uint4* delta, const uint4* weight,
                                                           uint4* sum, uint4* out, int rows, int chunks, float eps,
                                                           float inv_dim) {
  constexpr int N = 16 / Elem<DT>::kBytes;
  constexpr int kRows = 4 / W;
  __shared__ float part[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row = blockIdx.x * kRows + wave / W;
  if (W == 1 && row >= rows) return;  // W == 4: one row per workgroup, every one valid
  const int first = (wave % W) * 64 + lane;
  const int64_t base = static_cast<int64_t>(row) * chunks;
  uint4 xc[NC], dc[NC], wc[NC];
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int c = first + i * 64 * W;
    if (c < chunks) {
      xc[i] = x[base + c];
      if (ADD) dc[i] = delta[base + c];
      wc[i] = weight[c];
    }
  }
  float f[NC][N];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int c = first + i * 64 * W;
    if (c < chunks) {
      unpack<DT>(xc[i], f[i]);
      if (ADD) {
        float d[N];
        unpack<DT>(dc[i], d);
#pragma unroll
        for (int e = 0; e < N; ++e) f[i][e] = rnd<DT>(f[i][e] + d[e]);
        sum[base + c] = pack<DT>(f[i]);
      }
#pragma unroll
      for (int e = 0; e < N; ++e) ss += f[i][e] * f[i][e];
    }
  }
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) ss += __shfl_xor(ss, m);
  if (W > 1) {
    if (lane == 0) part[wave] = ss;
    __syncthreads();
    ss = (part[0] + part[1]) + (part[2] + part[3]);
  }
  const float inv = rsqrtf(ss * inv_dim + eps);
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int c = first + i * 64 * W;
    if (c < chunks) {
      float w[N];
      unpack<DT>(wc[i], w);
#pragma unroll
      for (int e = 0; e < N; ++e) w[e] *= rnd<DT>(f[i][e] * inv);
      out[base + c] = pack<DT>(w);
    }
  }
}

// One lane per 16-byte chunk of the output; gate and up are the halves of one row of gate_up.
template <int DT>
__global__ __launch_bounds__(256) void silu_mul_kernel(const uint4* gate_up, uint4* out, uint32_t total,
                                                       uint32_t chunks) {
  constexpr int N = 16 / Elem<DT>::kBytes;
  for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < total; i += gridDim.x * 256u) {
    const uint32_t row = i / chunks, c = i - row * chunks;
    const uint4* src = gate_up + static_cast<int64_t>(row) * 2 * chunks + c;
    const uint4 gc = src[0], uc = src[chunks];
    float g[N], u[N];
    unpack<DT>(gc, g);
    unpack<DT>(uc, u);
#pragma unroll
    for (int e = 0; e < N; ++e) g[e] = rnd<DT>(g[e] / (1.f + expf(-g[e]))) * u[e];
    out[i] = pack<DT>(g);
  }
}

template <int DT, bool ADD>
int launch_norm(const uint4* x, const uint4* d, const uint4* w, uint4* sum, uint4* out, int rows, int chunks, float eps,
                float inv_dim, hipStream_t s) {
  const dim3 four((rows + 3) / 4), one(rows), b(256);
#define MIP_NORM(W, NC, GRID) \
  hipLaunchKernelGGL((add_rms_norm_kernel<DT, W, NC, ADD>), GRID, b, 0, s, x, d, w, sum, out, rows, chunks, eps, inv_dim)
  if (chunks <= 128) MIP_NORM(1, 2, four);
  else if (chunks <= 256) MIP_NORM(1, 4, four);
  else if (chunks <= 512) MIP_NORM(4, 2, one);
  else if (chunks <= 1024) MIP_NORM(4, 4, one);
  else MIP_NORM(4, 8, one);
#undef MIP_NORM
  return status_from_hip(hipGetLastError());
}

template <int DT>
int norm_dtype(const void* x, const void* d, const void* w, void* sum, void* out, int rows, int chunks, float eps,
               float inv_dim, hipStream_t s) {
  const auto *xp = static_cast<const uint4*>(x), *dp = static_cast<const uint4*>(d), *wp = static_cast<const uint4*>(w);
  auto *sp = static_cast<uint4*>(sum), *op = static_cast<uint4*>(out);
  return d ? launch_norm<DT, true>(xp, dp, wp, sp, op, rows, chunks, eps, inv_dim, s)
           : launch_norm<DT, false>(xp, dp, wp, sp, op, rows, chunks, eps, inv_dim, s);
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace
}  // namespace mip

using namespace mip;

extern "C" int mip_add_rms_norm(void* out, void* sum, const void* x, const void* delta, const void* weight, int32_t rows,
                                int32_t dim, float eps, int32_t dtype, void* stream) {
  if (dtype != MIP_F32 && dtype != MIP_F16 && dtype != MIP_BF16) return MIP_EINVAL;
  if (rows < 0 || dim <= 0 || (delta != nullptr) != (sum != nullptr)) return MIP_EINVAL;
  if (rows == 0) return MIP_OK;
  if (!out || !x || !weight) return MIP_EINVAL;
  const int es = dtype == MIP_F32 ? 4 : 2;
  const int64_t row_bytes = static_cast<int64_t>(dim) * es;
  if (row_bytes % 16 || row_bytes > 16 * 2048) return MIP_EUNSUPPORTED;
  if (!aligned16(out) || !aligned16(sum) || !aligned16(x) || !aligned16(delta) || !aligned16(weight)) return MIP_EUNSUPPORTED;
  const int chunks = static_cast<int>(row_bytes / 16);
  const float inv_dim = 1.f / static_cast<float>(dim);
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case MIP_F32: return norm_dtype<MIP_F32>(x, delta, weight, sum, out, rows, chunks, eps, inv_dim, s);
    case MIP_F16: return norm_dtype<MIP_F16>(x, delta, weight, sum, out, rows, chunks, eps, inv_dim, s);
    default:      return norm_dtype<MIP_BF16>(x, delta, weight, sum, out, rows, chunks, eps, inv_dim, s);
  }
}

extern "C" int mip_silu_mul(void* out, const void* gate_up, int32_t rows, int32_t inter, int32_t dtype, void* stream) {
  if (dtype != MIP_F32 && dtype != MIP_F16 && dtype != MIP_BF16) return MIP_EINVAL;
  if (rows < 0 || inter <= 0) return MIP_EINVAL;
  if (rows == 0) return MIP_OK;
  if (!out || !gate_up) return MIP_EINVAL;
  const int es = dtype == MIP_F32 ? 4 : 2;
  const int64_t row_bytes = static_cast<int64_t>(inter) * es;
  if (row_bytes % 16 || !aligned16(out) || !aligned16(gate_up)) return MIP_EUNSUPPORTED;
  const int64_t total = rows * (row_bytes / 16);
  if (total >= (int64_t{1} << 31)) return MIP_EUNSUPPORTED;
  const uint32_t chunks = static_cast<uint32_t>(row_bytes / 16);
  const int64_t want = (total + 255) / 256;
  const dim3 grid(static_cast<uint32_t>(want < 65536 ? want : 65536)), b(256);
  const auto* src = static_cast<const uint4*>(gate_up);
  auto* dst = static_cast<uint4*>(out);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const uint32_t n = static_cast<uint32_t>(total);
  switch (dtype) {
    case MIP_F32: hipLaunchKernelGGL((silu_mul_kernel<MIP_F32>), grid, b, 0, s, src, dst, n, chunks); break;
    case MIP_F16: hipLaunchKernelGGL((silu_mul_kernel<MIP_F16>), grid, b, 0, s, src, dst, n, chunks); break;
    default:      hipLaunchKernelGGL((silu_mul_kernel<MIP_BF16>), grid, b, 0, s, src, dst, n, chunks); break;
  }
  return status_from_hip(hipGetLastError());
}
