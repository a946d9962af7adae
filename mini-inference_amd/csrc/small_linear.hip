// Linear layers of a decode step (few rows), with the work around them fused in:
//     y = A W^T                      A: the input rows, or their RMS norm computed on the fly
//     out = y (+ bias), its q and k heads rotated (rotary embedding) where asked,
//           or  residual + y,  or  silu(y[:, :I]) * y[:, I:]
//
// Reference semantics: engine/model.py's qkv_proj(input_norm(x)), x + o_proj(..),
// silu * up of gate_up_proj(post_attn_norm(x)), x + down_proj(..). Products accumulate in fp32;
// the normed row, the product (with its bias), the silu and the result are each rounded to the
// dtype, as torch stores them, so the values differ from torch's by the order of the sums only.
//
// What bounds it: at few rows a weight is used once per row, so the layer is a read of its
// weights: 2 to 35 MB, where the launch and the first memory round trip cost as much as the bytes.
// The split follows from that:
//   - one workgroup owns a TM*16 x TN*16 tile of the output and its NW wavefronts split K, with no
//     second launch to sum the parts; the parts meet in LDS once, at the end. K is not split over
//     workgroups, so at up to 16 rows N = 896 gives 56 workgroups and N = 1152 72 for 256 CUs: the down
//     product of the 0.5B layer (896 x 4864, 8.7 MB) takes 10.5 us, 0.84 TB/s, on a fifth of the chip;
//   - wavefronts share nothing until then, so both operands go from global memory straight into
//     registers in the MFMA layout (16 rows x 64 contiguous bytes per load) with no barrier in the
//     loop, U k-steps in flight and the next U requested before the current are multiplied;
//   - the tiles of the same weight rows sit on one XCD (workgroup b runs on XCD b mod 8), so its
//     L2 reads them from memory once.
// W is the first MFMA operand, so a lane ends up with 4 consecutive output columns of one row.
//
// Measured (bf16, weights cold, graph replay, the fused call against the library product and the
// separate kernels it takes the place of), 0.5B shapes at 8 rows: norm + qkv 4.5 against 8.6 us,
// norm + gate + up + silu 9.3 / 14.6 (17.4 MB, 1.9 TB/s; a bare read of the weights in this split
// takes 6.1), o + residual 3.8 / 8.5, down + residual 10.5 / 20.3; at 64 rows 5.7 / 11.2,
// 16.3 / 18.3, 4.2 / 10.0, 12.0 / 19.1. The rotation at the end of the q, k, v projection costs 0.7 us
// and saves the 3.2 to 5 us kernel that rotates and appends (the decode's merge appends instead). With more rows every workgroup's reads of A (L2 to
// registers) take over: gate + up 27 / 18 us at 65 rows, which is left to the library.
#include "mip_common.h"

namespace mip {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

template <int DT> struct Mfma;
template <> struct Mfma<MIP_BF16> {
  using E = __bf16;
  static __device__ __forceinline__ f32x4 mac(const uint4& a, const uint4& b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
template <> struct Mfma<MIP_F16> {
  using E = _Float16;
  static __device__ __forceinline__ f32x4 mac(const uint4& a, const uint4& b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};

struct LinearArgs {
  const char* a;         // [m, k]
  const char* w;         // [n, k] (silu: gate rows, then as many up rows)
  const char* bias;      // [n] or null
  const char* residual;  // [m, n] or null
  const char* norm;      // [k] or null
  char* out;             // [m, n] (silu: n / 2 columns)
  const char* cos;       // rope: [m, head_dim] rows, cs_st bytes apart
  const char* sin;
  int64_t cs_st;
  int m, n, k, m_tiles, n_tiles;
  int head_dim, rot_heads;  // rope: the first rot_heads heads of the n columns are rotated
  float eps, inv_k;
};

enum Epilogue { kPlain = 0, kResidual = 1, kSilu = 2, kRope = 3 };

// First column of rope tile n0 / 16: its head, and 8 columns of that head's first half.
__device__ __forceinline__ int pair_column(int n0, int head_dim) {
  const int head = n0 / head_dim;
  return head * head_dim + ((n0 - head * head_dim) >> 1);
}

// Tiles of 16 x 16: TM over rows, TN over weight rows. A silu tile's 16 weight rows are 8 gate rows
// and the 8 up rows of the same output columns, so its output is 8 wide; a rope tile's are 8 rows
// of a head's first half and the 8 that rotate with them.
template <int DT, int TM, int TN, int NW, int U, bool NORM, int EPI>
__global__ __launch_bounds__(NW * 64) void small_linear_kernel(LinearArgs p) {
  using E = typename Mfma<DT>::E;
  constexpr int kCols = EPI == kSilu ? 8 : 16;  // output columns of a tile
  __shared__ f32x4 part[NW][TM * TN][64];
  __shared__ float sums[NORM ? NW : 1][TM * 16];
  // The wavefront's index as a scalar: the matrix instructions below stand under tests of its k-range,
  // and they ignore the lane mask, so those tests have to be branches.
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = lane & 15, quad = lane >> 4;

  // Workgroup b: XCD b & 7 takes the column tiles congruent to it, every row tile of one in turn.
  const int xcd = blockIdx.x & 7, seq = blockIdx.x >> 3;
  const int tile_n = (seq / p.m_tiles) * 8 + xcd, tile_m = seq % p.m_tiles;
  if (tile_n >= p.n_tiles) return;
  const int m0 = tile_m * TM * 16, n0 = tile_n * TN * kCols;

  const int steps = p.k >> 5;
  const int begin = steps * wave / NW, end = steps * (wave + 1) / NW;
  const char* wp[TN];
  const char* ap[TM];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    int r = n0 + j * kCols + row;
    if (EPI == kSilu && row >= 8) r += (p.n >> 1) - 8;
    if (EPI == kRope) r = pair_column(n0 + j * 16, p.head_dim) + (row < 8 ? row : (p.head_dim >> 1) + row - 8);
    wp[j] = p.w + (static_cast<int64_t>(r) * p.k + quad * 8) * 2;
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int r = m0 + i * 16 + row;
    ap[i] = p.a + (static_cast<int64_t>(r < p.m ? r : p.m - 1) * p.k + quad * 8) * 2;
  }
  // What the epilogue adds, requested ahead of everything: output o = threadIdx.x (one each at most).
  const int half = EPI == kRope ? p.head_dim >> 1 : 0;
  constexpr int kLanes = 4 * kCols / (EPI == kRope ? 2 : 1);  // outputs of 4 (rope: 2 x 4) columns in a tile
  static_assert(TM * TN * kLanes <= NW * 64, "one output per thread");
  const int tile = threadIdx.x / kLanes, l = threadIdx.x % kLanes, ti = tile / TN, tj = tile % TN;
  const int m = m0 + ti * 16 + (l & 15);
  const int n = (EPI == kRope ? pair_column(n0 + tj * 16, p.head_dim) : n0 + tj * kCols) + (l >> 4) * 4;
  const int ldc = EPI == kSilu ? p.n >> 1 : p.n;
  const bool writes = tile < TM * TN && m < p.m;
  const int64_t at_out = (static_cast<int64_t>(m) * ldc + n) * 2;
  E add0[4], add1[4], c0[4], c1[4], s0[4], s1[4];
  bool rotate = false;
  if (writes) {
    if (EPI == kResidual) __builtin_memcpy(add0, p.residual + at_out, 8);
    if ((EPI == kPlain || EPI == kRope) && p.bias) __builtin_memcpy(add0, p.bias + n * 2, 8);
    if (EPI == kRope) {
      if (p.bias) __builtin_memcpy(add1, p.bias + (n + half) * 2, 8);
      const int head = n / p.head_dim, d = n - head * p.head_dim;
      rotate = head < p.rot_heads;
      if (rotate) {
        const char* cs = p.cos + m * p.cs_st + d * 2;
        const char* sn = p.sin + m * p.cs_st + d * 2;
        __builtin_memcpy(c0, cs, 8);
        __builtin_memcpy(c1, cs + half * 2, 8);
        __builtin_memcpy(s0, sn, 8);
        __builtin_memcpy(s1, sn + half * 2, 8);
      }
    }
  }
  const char* np = NORM ? p.norm + quad * 16 : nullptr;

  uint4 wf[U][TN], af[U][TM], nf[NORM ? U : 1];
  // Steps past the wavefront's range read its last one (in bounds) and are not multiplied.
  auto at = [&](int s) { return static_cast<int64_t>(s < end ? s : (end > begin ? end - 1 : 0)) * 64; };
  auto load = [&](int s, uint4 (&w)[TN], uint4 (&a)[TM], uint4& n) {
    const int64_t off = at(s);
#pragma unroll
    for (int i = 0; i < TM; ++i) a[i] = *reinterpret_cast<const uint4*>(ap[i] + off);
    if (NORM) n = *reinterpret_cast<const uint4*>(np + off);
#pragma unroll
    for (int j = 0; j < TN; ++j) w[j] = *reinterpret_cast<const uint4*>(wp[j] + off);
  };
  if (NORM) {
    // Loads return in order: the rows first, so their sums run while the weights are on their way.
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < TM; ++i) af[u][i] = *reinterpret_cast<const uint4*>(ap[i] + at(begin + u));
#pragma unroll
    for (int u = 0; u < U; ++u) {
      nf[u] = *reinterpret_cast<const uint4*>(np + at(begin + u));
#pragma unroll
      for (int j = 0; j < TN; ++j) wf[u][j] = *reinterpret_cast<const uint4*>(wp[j] + at(begin + u));
    }
    __builtin_amdgcn_sched_barrier(0);
  } else {
#pragma unroll
    for (int u = 0; u < U; ++u) load(begin + u, wf[u], af[u], nf[0]);
  }

  float inv[TM];
  if (NORM) {
    // Row sums of squares: the first steps' rows are in registers already, later ones are read
    // here and again below (from cache), behind the weights' own latency.
    float ss[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) ss[i] = 0.f;
    auto square = [&](const uint4& c, float& acc) {
      E e[8];
      __builtin_memcpy(e, &c, 16);
#pragma unroll
      for (int t = 0; t < 8; ++t) acc += static_cast<float>(e[t]) * static_cast<float>(e[t]);
    };
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (begin + u < end)
#pragma unroll
        for (int i = 0; i < TM; ++i) square(af[u][i], ss[i]);
    for (int s = begin + U; s < end; ++s)
#pragma unroll
      for (int i = 0; i < TM; ++i) square(*reinterpret_cast<const uint4*>(ap[i] + at(s)), ss[i]);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      ss[i] += __shfl_xor(ss[i], 16);
      ss[i] += __shfl_xor(ss[i], 32);
      if (quad == 0) sums[wave][i * 16 + row] = ss[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      float t = 0.f;
#pragma unroll
      for (int v = 0; v < NW; ++v) t += sums[v][i * 16 + row];
      inv[i] = rsqrtf(t * p.inv_k + p.eps);
    }
  }

  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int s = begin; s < end; s += U) {
    uint4 wn[U][TN], an[U][TM], nn[NORM ? U : 1];
    const bool more = s + U < end;
    if (more) {
#pragma unroll
      for (int u = 0; u < U; ++u) load(s + U + u, wn[u], an[u], nn[NORM ? u : 0]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (s + u < end) {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          uint4 a = af[u][i];
          if (NORM) {
            E x[8], g[8];
            __builtin_memcpy(x, &a, 16);
            __builtin_memcpy(g, &nf[u], 16);
#pragma unroll
            for (int t = 0; t < 8; ++t) {
              const E h = static_cast<E>(static_cast<float>(x[t]) * inv[i]);
              x[t] = static_cast<E>(static_cast<float>(g[t]) * static_cast<float>(h));
            }
            __builtin_memcpy(&a, x, 16);
          }
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = Mfma<DT>::mac(wf[u][j], a, acc[i][j]);
        }
      }
    }
    if (more) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int j = 0; j < TN; ++j) wf[u][j] = wn[u][j];
#pragma unroll
        for (int i = 0; i < TM; ++i) af[u][i] = an[u][i];
        if (NORM) nf[u] = nn[u];
      }
    }
  }

#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) part[wave][i * TN + j][lane] = acc[i][j];
  __syncthreads();

  if (!writes) return;
  auto total = [&](int at) {
    f32x4 v = part[0][tile][at];
#pragma unroll
    for (int w = 1; w < NW; ++w) v += part[w][tile][at];
    return v;
  };
  auto stored = [](float f) { return static_cast<float>(static_cast<E>(f)); };
  f32x4 v = total(l);
  E e[4];
  if constexpr (EPI == kSilu) {
    const f32x4 up = total(l + 32);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float g = stored(v[c]);
      v[c] = stored(g / (1.f + expf(-g))) * stored(up[c]);
    }
  } else if constexpr (EPI == kResidual) {
#pragma unroll
    for (int c = 0; c < 4; ++c) v[c] = static_cast<float>(add0[c]) + stored(v[c]);
  } else if (p.bias) {
#pragma unroll
    for (int c = 0; c < 4; ++c) v[c] += static_cast<float>(add0[c]);
  }
  if constexpr (EPI == kRope) {
    f32x4 x1 = total(l + 32);
    if (p.bias) {
#pragma unroll
      for (int c = 0; c < 4; ++c) x1[c] += static_cast<float>(add1[c]);
    }
    if (rotate) {
      // The rounding of every product and sum, as rope_append.hip (bit-identical to it).
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const float a = stored(v[c]), b = stored(x1[c]);
        v[c] = stored(a * static_cast<float>(c0[c])) + stored(-b * static_cast<float>(s0[c]));
        x1[c] = stored(b * static_cast<float>(c1[c])) + stored(a * static_cast<float>(s1[c]));
      }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) e[c] = static_cast<E>(x1[c]);
    __builtin_memcpy(p.out + at_out + half * 2, e, 8);
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) e[c] = static_cast<E>(v[c]);
  __builtin_memcpy(p.out + at_out, e, 8);
}

template <int DT, int TM, int TN, int NW, int U, bool NORM, int EPI>
int launch(LinearArgs p, hipStream_t s) {
  constexpr int kCols = EPI == kSilu ? 8 : 16;
  p.m_tiles = (p.m + TM * 16 - 1) / (TM * 16);
  p.n_tiles = (EPI == kSilu ? p.n / 2 : p.n) / (TN * kCols);
  const int grid = (p.n_tiles + 7) / 8 * 8 * p.m_tiles;
  hipLaunchKernelGGL((small_linear_kernel<DT, TM, TN, NW, U, NORM, EPI>), dim3(grid), dim3(NW * 64), 0, s, p);
  return status_from_hip(hipGetLastError());
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

int check(const void* out, const void* a, const void* w, int32_t m, int32_t n, int32_t k, int32_t dtype) {
  if (dtype != MIP_F32 && dtype != MIP_F16 && dtype != MIP_BF16) return MIP_EINVAL;
  if (m < 0 || n <= 0 || k <= 0) return MIP_EINVAL;
  if (m == 0) return MIP_OK;
  if (!out || !a || !w) return MIP_EINVAL;
  if (dtype == MIP_F32 || m > 256 || n % 16 || k % 32 || n > (1 << 24) || k > (1 << 24)) return MIP_EUNSUPPORTED;
  if (!aligned16(out) || !aligned16(a) || !aligned16(w)) return MIP_EUNSUPPORTED;
  return MIP_OK;
}

// The tile by rows: enough workgroups to cover the CUs at N = 896 .. 9728 while each reads as few
// rows of A as that allows (a wavefront's A loads cost as much as its W loads at TM = TN = 1).
template <int DT, bool NORM, int EPI> int plain_linear(const LinearArgs& p, hipStream_t s) {
  if constexpr (NORM) {
    if (p.m > 128 && p.n % 64 == 0) return launch<DT, 2, 4, 8, 2, NORM, EPI>(p, s);
    if (p.m > 64 && p.n % 32 == 0) return launch<DT, 2, 2, 8, 4, NORM, EPI>(p, s);
  } else {
    if (p.m > 192 && p.n % 64 == 0) return launch<DT, 2, 4, 8, 2, NORM, EPI>(p, s);
    if (p.m > 96 && p.n % 32 == 0) return launch<DT, 2, 2, 8, 2, NORM, EPI>(p, s);
  }
  if (p.m > 32 && p.n % 32 == 0) return launch<DT, 1, 2, 4, 7, NORM, EPI>(p, s);
  return p.k <= 1024 ? launch<DT, 1, 1, 4, 8, NORM, EPI>(p, s) : launch<DT, 1, 1, 8, 4, NORM, EPI>(p, s);
}
template <int DT> int norm_linear(const LinearArgs& p, hipStream_t s) {
  if (p.cos) return p.norm ? plain_linear<DT, true, kRope>(p, s) : plain_linear<DT, false, kRope>(p, s);
  return plain_linear<DT, true, kPlain>(p, s);
}
template <int DT> int norm_gate_up(const LinearArgs& p, hipStream_t s) {
  if (p.m > 32 && p.n % 64 == 0) return launch<DT, 4, 4, 8, 1, true, kSilu>(p, s);
  if (p.m > 16 && p.n % 32 == 0) return launch<DT, 1, 2, 4, 7, true, kSilu>(p, s);
  return launch<DT, 1, 1, 4, 8, true, kSilu>(p, s);
}
template <int DT> int linear_residual(const LinearArgs& p, hipStream_t s) {
  if (p.m > 128 && p.n % 32 == 0) return launch<DT, 2, 2, 8, 2, false, kResidual>(p, s);
  if (p.m > 64) return launch<DT, 2, 1, 8, 4, false, kResidual>(p, s);
  if (p.m > 16 && p.n >= 2048 && p.n % 32 == 0) return launch<DT, 2, 2, 4, 4, false, kResidual>(p, s);
  return p.k <= 1024 ? launch<DT, 1, 1, 4, 8, false, kResidual>(p, s) : launch<DT, 1, 1, 8, 4, false, kResidual>(p, s);
}

LinearArgs args(void* out, const void* a, const void* w, int m, int n, int k) {
  LinearArgs p{};
  p.a = static_cast<const char*>(a);
  p.w = static_cast<const char*>(w);
  p.out = static_cast<char*>(out);
  p.m = m;
  p.n = n;
  p.k = k;
  return p;
}

}  // namespace
}  // namespace mip

using namespace mip;

extern "C" int mip_norm_linear(void* out, const void* x, const void* norm, float eps, const void* weight, const void* bias,
                               int32_t m, int32_t n, int32_t k, int32_t gate_up, int32_t dtype, void* stream) {
  const int st = check(out, x, weight, m, n, k, dtype);
  if (st != MIP_OK || m == 0) return st;
  if (!norm || (gate_up && bias)) return MIP_EINVAL;
  if (!aligned16(norm) || !aligned16(bias)) return MIP_EUNSUPPORTED;
  LinearArgs p = args(out, x, weight, m, n, k);
  p.norm = static_cast<const char*>(norm);
  p.bias = static_cast<const char*>(bias);
  p.eps = eps;
  p.inv_k = 1.f / static_cast<float>(k);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == MIP_F16) return gate_up ? norm_gate_up<MIP_F16>(p, s) : norm_linear<MIP_F16>(p, s);
  return gate_up ? norm_gate_up<MIP_BF16>(p, s) : norm_linear<MIP_BF16>(p, s);
}

extern "C" int mip_qkv_linear(void* out, const void* x, const void* norm, float eps, const void* weight, const void* bias,
                              const void* cos, const void* sin, int64_t cs_stride_tok, int32_t m, int32_t n, int32_t k,
                              int32_t head_dim, int32_t rot_heads, int32_t dtype, void* stream) {
  const int st = check(out, x, weight, m, n, k, dtype);
  if (st != MIP_OK || m == 0) return st;
  if (!cos || !sin || head_dim <= 0 || rot_heads < 0 || n % head_dim || rot_heads > n / head_dim) return MIP_EINVAL;
  if (head_dim % 16 || !aligned16(norm) || !aligned16(bias)) return MIP_EUNSUPPORTED;
  if ((reinterpret_cast<uintptr_t>(cos) | reinterpret_cast<uintptr_t>(sin) | static_cast<uint64_t>(cs_stride_tok * 2)) & 7)
    return MIP_EUNSUPPORTED;  // read 4 elements at a time
  LinearArgs p = args(out, x, weight, m, n, k);
  p.norm = static_cast<const char*>(norm);
  p.bias = static_cast<const char*>(bias);
  p.cos = static_cast<const char*>(cos);
  p.sin = static_cast<const char*>(sin);
  p.cs_st = cs_stride_tok * 2;
  p.head_dim = head_dim;
  p.rot_heads = rot_heads;
  p.eps = eps;
  p.inv_k = 1.f / static_cast<float>(k);
  hipStream_t s = static_cast<hipStream_t>(stream);
  return dtype == MIP_F16 ? norm_linear<MIP_F16>(p, s) : norm_linear<MIP_BF16>(p, s);
}

extern "C" int mip_linear_residual(void* out, const void* a, const void* weight, const void* residual, int32_t m, int32_t n,
                                   int32_t k, int32_t dtype, void* stream) {
  const int st = check(out, a, weight, m, n, k, dtype);
  if (st != MIP_OK || m == 0) return st;
  if (!residual) return MIP_EINVAL;
  if (!aligned16(residual)) return MIP_EUNSUPPORTED;
  LinearArgs p = args(out, a, weight, m, n, k);
  p.residual = static_cast<const char*>(residual);
  hipStream_t s = static_cast<hipStream_t>(stream);
  return dtype == MIP_F16 ? linear_residual<MIP_F16>(p, s) : linear_residual<MIP_BF16>(p, s);
}
