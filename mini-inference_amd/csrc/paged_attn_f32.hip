// Paged attention in fp32 on the matrix cores (gfx950): decode partitions and packed prefill, at
// head_dim 64 or 128 and up to 16 query heads per kv head.
//
// Reference semantics: engine/kv_cache.py:615-620 (decode) and :268-294 (packed prefill), fp32
// throughout: v_mfma_f32_16x16x4_f32 multiplies and accumulates in fp32, the softmax is fp32.
//
// A wavefront's tile is 16 keys x 16 query rows; a row is one (token, head of the group) pair, so
// a decode workgroup holds the G heads of one token and a prefill workgroup 16 consecutive pairs
// of one sequence, token-major. K, V and Q go from global memory straight into the MFMA layout:
//   S^T[key][row] = K . Q^T   lane (c = lane & 15, g = lane >> 4) holds key c's dims g*D/4 ..,
//                             i.e. MFMA step s multiplies dims {s, s + D/4, ..} (their order does
//                             not matter as long as Q uses the same);
//   O^T[d][row] += V^T . P^T  step i multiplies keys {4g + i}: exactly the S^T output layout, so
//                             the weights stay where they are.
// The 4 wavefronts of a workgroup take the key tiles in turn and meet once in LDS; a key tile is
// used by one wavefront, so nothing is staged.
//
// What bounds it: at the short contexts that fp32 runs have, the chain of memory round trips
// (lengths, table, keys, merge) and each wavefront's steps; at long prefills the fp32 matrix rate
// (157 TFLOP/s). Against the VALU kernel, which reduced every score across lanes, took 8 keys a
// step and gave each new token a workgroup of its own (graph replay, 14q/2kv d64 | 28q/4kv d128; the
// rules that choose between the two lie in paged_decode.hip, with the other group sizes):
//   decode, 8 sequences of 16-256 keys 16.5 -> 8.4 | 21.7 -> 12.9 us; 64 of 2,000 44.4 -> 37.1 | 130 -> 130
//   prefill, 8 prompts of 16-256       38.5 -> 20.0 | 104 -> 58.3;   8 of 1,024 740 -> 245 | 2811 -> 961
// The sums are kept at least as exact as the VALU kernel's: a score in chains of 8 products, a tile's
// values pairwise. Decode, relative error against 64 bits at both head sizes, 64 sequences x 8 seeds:
// 7.9-8.0e-8 over 1-16 keys (0.99 of the VALU kernel's), 1.3e-7 over 16-64 (0.97), 1.4e-7 over 16-256 (0.89),
// 1.7e-7 over 500-1,024 (0.80), 1.9e-7 over 1,000-4,096 (0.83). That costs 5-15 %: single chains took 7.4 and 18.8 us on the two 14q/2kv mixes, at 2.9e-7.
// 8 wavefronts per workgroup: 7.2 / 39.5 us (decode), 25.0 / 302 (prefill); two row tiles per
// wavefront: 20.8 / 231 | 79.1 / 996 (prefill; a workgroup's steps get twice as long), single chains.
#include "paged_decode_common.h"

namespace mip {
namespace decode {
namespace {

constexpr int kRows = 16;

__device__ __forceinline__ f32x4_t mfma_f32(float a, float b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Where a tile of 16 keys lies: this lane's key row c and value rows 4g + i, and which keys are
// real (bit j: key base + j lies below t1 in a block of the pool). Keys past t1 stand for the
// tile's first key and block ids outside the pool for block 0, both flagged invalid, so every
// address stays inside the pool.
struct F32Rows {
  int k, v[4];
  uint32_t valid;
};

__device__ __forceinline__ F32Rows f32_rows(const DecodeArgs& a, const int32_t* table, int kvh, int base, int t1, int c,
                                            int g) {
  F32Rows r;
  const int left = t1 - base;  // base < t1, a multiple of 16
  const uint32_t in = left >= 16 ? 0xffffu : (1u << left) - 1u;
  if (a.bs >= 16) {  // the whole tile lies in one block
    const int blk = load_uniform_i32(table + (base >> a.log2_bs));
    const bool ok = blk >= 0 && blk < a.ncb;
    const int first = ((ok ? blk : 0) * a.hkv + kvh) * a.bs + (base & (a.bs - 1));
    r.valid = ok ? in : 0u;
    r.k = first + (c < left ? c : 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) r.v[i] = first + (4 * g + i < left ? 4 * g + i : 0);
  } else {
    bool ok;
    auto row_of = [&](int j) {
      const int tok = base + (j < left ? j : 0);
      const int blk = table[tok >> a.log2_bs];
      ok = blk >= 0 && blk < a.ncb;
      return ((ok ? blk : 0) * a.hkv + kvh) * a.bs + (tok & (a.bs - 1));
    };
    r.k = row_of(c);
    r.valid = static_cast<uint32_t>(__ballot(ok)) & in;  // lanes 0 .. 15 hold keys 0 .. 15
#pragma unroll
    for (int i = 0; i < 4; ++i) r.v[i] = row_of(4 * g + i);
  }
  return r;
}

// This lane's share of a tile: dims g * D/4 .. of key c; dims 16 t + c of keys 4g + i.
template <int D> __device__ __forceinline__ void f32_load_k(float (&k)[D / 4], const DecodeArgs& a, const F32Rows& r, int g) {
  const float4* p = reinterpret_cast<const float4*>(a.k) + (static_cast<int64_t>(r.k) * D + g * (D / 4)) / 4;
#pragma unroll
  for (int t = 0; t < D / 16; ++t) {
    const float4 x = p[t];
    k[4 * t] = x.x; k[4 * t + 1] = x.y; k[4 * t + 2] = x.z; k[4 * t + 3] = x.w;
  }
}
template <int D>
__device__ __forceinline__ void f32_load_v(float (&v)[4][D / 16], const DecodeArgs& a, const F32Rows& r, int c) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float* p = reinterpret_cast<const float*>(a.v) + static_cast<int64_t>(r.v[i]) * D + c;
#pragma unroll
    for (int t = 0; t < D / 16; ++t) v[i][t] = p[16 * t];
  }
}

template <int D>
__global__ __launch_bounds__(kNW * kWave) void paged_attn_f32(DecodeArgs a) {
  constexpr int T = D / 16;  // dim tiles
  __shared__ float sh_acc[kNW][kRows][D + 4];  // + 4: the 16 rows of a store spread over the banks
  __shared__ float sh_m[kNW][kRows], sh_l[kNW][kRows];
  const int lane = threadIdx.x & (kWave - 1), c = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int kvh = blockIdx.y;

  // The workgroup's rows: row r is query row q0 + r / group of q, head kvh * group + r % group,
  // from row r0 on; it sees keys below first + r / group (decode: one token, the whole context).
  int part = 0, q0, r0, rows, trow, first;
  if (a.cu_q) {
    const int tiles = (a.max_q_len * a.group + kRows - 1) / kRows;
    const int s = blockIdx.x / tiles;
    q0 = a.cu_q[s];
    rows = (a.cu_q[s + 1] - q0) * a.group;
    r0 = (blockIdx.x - s * tiles) * kRows;
    if (r0 >= rows) return;
    trow = s;
    first = a.ctx_start[s] + 1;
  } else {
    part = blockIdx.x;
    q0 = trow = blockIdx.z;
    rows = a.group;
    r0 = 0;
    first = a.lens[q0];
  }
  const int cap = a.max_blocks * a.bs;
  const int last_row = r0 + kRows < rows ? r0 + kRows - 1 : rows - 1;
  const int ctx = min(first + last_row / a.group, cap);  // keys of the row that sees most
  const int np_b = !a.cu_q && ctx > 0 ? (ctx + a.part_tokens - 1) / a.part_tokens : 1;
  if (part >= np_b) return;
  const int t0 = part * a.part_tokens;
  const int t1 = a.cu_q ? ctx : min(t0 + a.part_tokens, ctx);

  const int row = min(r0 + c, last_row);  // rows past the end shadow the last one
  const int row_tok = row / a.group;
  const int lim = min(first + row_tok, cap);
  const float* qp = reinterpret_cast<const float*>(a.q) + (q0 + row_tok) * a.q_sb +
                    (kvh * a.group + row - row_tok * a.group) * a.q_sh + g * (D / 4);
  float qf[D / 4];
#pragma unroll
  for (int i = 0; i < D / 4; ++i) qf[i] = qp[i];
  // Keys below this are seen by every row.
  const int all_see = min(first + r0 / a.group, cap);

  float m = kNoScore, l = 0.f;
  f32x4_t acc[T];
#pragma unroll
  for (int t = 0; t < T; ++t) acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const int32_t* table = a.bt + static_cast<int64_t>(trow) * a.bt_stride;
  // A step: the tile's values are requested first and the next tile's keys as soon as the scores
  // have used this one's, so each load has at least half a step to arrive and no operand is
  // held twice.
  constexpr int kStep = kNW * 16;
  int base = t0 + w * 16;
  F32Rows at{};
  float kf[D / 4];
  if (base < t1) {
    at = f32_rows(a, table, kvh, base, t1, c, g);
    f32_load_k<D>(kf, a, at, g);
  }
  for (; base < t1; base += kStep) {
    float v[4][T];
    f32_load_v<D>(v, a, at, c);
    const uint32_t valid = at.valid;
    const int next = base + kStep;
    at = f32_rows(a, table, kvh, next < t1 ? next : base, t1, c, g);
    // A score is the sum of many short chains, added pairwise (the VALU kernel's depth: 8 products
    // each), so that few roundings fall on a sum that has already grown; and no product waits
    // for the one before it.
    f32x4_t s{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int h = 0; h < D / 64; ++h) {
      f32x4_t sq[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) sq[j] = mfma_f32(kf[16 * h + j], qf[16 * h + j], f32x4_t{0.f, 0.f, 0.f, 0.f});
#pragma unroll
      for (int j = 0; j < 8; ++j) sq[j] = mfma_f32(kf[16 * h + 8 + j], qf[16 * h + 8 + j], sq[j]);
      s += ((sq[0] + sq[1]) + (sq[2] + sq[3])) + ((sq[4] + sq[5]) + (sq[6] + sq[7]));
    }
    f32_load_k<D>(kf, a, at, g);
    bool need = false;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = 4 * g + i;
      s[i] = ((valid >> key) & 1u) && base + key < lim ? s[i] * a.scale_log2 : -INFINITY;
      need |= s[i] > m + kRescaleLog2;
    }
    if (__any(need)) {
      float mx = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
      mx = fmaxf(mx, __shfl_xor(mx, 16));
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      const float mn = fmaxf(m, mx);
      const float alpha = fast_exp2(m - mn);
      l *= alpha;
#pragma unroll
      for (int t = 0; t < T; ++t) acc[t] *= alpha;
      m = mn;
    }
    float p[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      p[i] = fast_exp2(s[i] - m);  // 0 for a key that is not seen, or scores -inf: m is finite
      l += p[i];
    }
    bool odd = false;  // an infinity or NaN in a value that not every row sees
    const bool ragged = base + 16 > all_see;
    if (ragged || valid != 0xffffu) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool ok = (valid >> (4 * g + i)) & 1u;
#pragma unroll
        for (int t = 0; t < T; ++t) {
          v[i][t] = ok ? v[i][t] : 0.f;
          odd |= !(fabsf(v[i][t]) < INFINITY);
        }
      }
    }
    if (ragged && __any(odd)) {
      // 0 * inf would reach the rows that do not see the key: such values leave the products and
      // are added one key at a time to the rows that do.
#pragma unroll 1
      for (int key = 0; key < 16; ++key) {
        // Values of this key are held by lanes of group key / 4, dim 16 t + c; row c's
        // accumulator holds dims 16 t + 4 g + i.
#pragma unroll
        for (int t = 0; t < T; ++t) {
          const float vk = key % 4 == 0 ? v[0][t] : key % 4 == 1 ? v[1][t] : key % 4 == 2 ? v[2][t] : v[3][t];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float x = __shfl(vk, (key / 4) * 16 + 4 * g + i);
            const bool wild = !(fabsf(x) < INFINITY);
            const float pk = key % 4 == 0 ? p[0] : key % 4 == 1 ? p[1] : key % 4 == 2 ? p[2] : p[3];
            const float pr = __shfl(pk, (key / 4) * 16 + c);
            if (wild && base + key < lim) acc[t][i] += pr * x;
          }
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < T; ++t) v[i][t] = fabsf(v[i][t]) < INFINITY ? v[i][t] : 0.f;
    }
    // The tile's 16 keys are summed pairwise before they meet the running sum.
#pragma unroll
    for (int t = 0; t < T; ++t) {
      f32x4_t o[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = mfma_f32(v[i][t], p[i], f32x4_t{0.f, 0.f, 0.f, 0.f});
      acc[t] += (o[0] + o[1]) + (o[2] + o[3]);
    }
  }

  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);
#pragma unroll
  for (int t = 0; t < T; ++t)
    *reinterpret_cast<f32x4_t*>(&sh_acc[w][c][16 * t + 4 * g]) = acc[t];
  if (g == 0) {
    sh_m[w][c] = m;
    sh_l[w][c] = l;
  }
  __syncthreads();

  float* out = reinterpret_cast<float*>(a.out);
  for (int i = threadIdx.x; i < (last_row - r0 + 1) * D; i += kNW * kWave) {
    const int r = i / D, d = i - r * D;
    float mx = -INFINITY;
#pragma unroll
    for (int ww = 0; ww < kNW; ++ww) mx = fmaxf(mx, sh_m[ww][r]);
    float A = 0.f, Ls = 0.f;
#pragma unroll
    for (int ww = 0; ww < kNW; ++ww) {
      const float wt = fast_exp2(sh_m[ww][r] - mx);  // a wavefront without keys for the row has sums of 0
      A = fmaf(wt, sh_acc[ww][r][d], A);
      Ls = fmaf(wt, sh_l[ww][r], Ls);
    }
    const int tok = (r0 + r) / a.group, head = kvh * a.group + (r0 + r) - tok * a.group;
    if (np_b == 1) {
      out[(q0 + tok) * a.out_sb + head * a.out_sh + d] = Ls > 0.f ? A / Ls : 0.f;
    } else {
      const int64_t slot = (static_cast<int64_t>(q0) * a.hq + head) * a.nparts + part;
      a.ws_acc[slot * D + d] = A;
      if (d == 0) {
        a.ws_ml[slot * 2] = mx;
        a.ws_ml[slot * 2 + 1] = Ls;
      }
    }
  }
}

}  // namespace

KernelFn f32_decode_kernel(int d) { return d == 64 ? paged_attn_f32<64> : paged_attn_f32<128>; }

int f32_prefill_launch(const DecodeArgs& a, int num_seqs, int d, hipStream_t stream) {
  // At most max_q_len tiles per sequence (group <= 16), so the grid fits where one per token did.
  const int64_t tiles = (static_cast<int64_t>(a.max_q_len) * a.group + kRows - 1) / kRows;
  hipLaunchKernelGGL(f32_decode_kernel(d), dim3(static_cast<unsigned>(tiles * num_seqs), a.hkv), dim3(kNW * kWave), 0,
                     stream, a);
  return status_from_hip(hipGetLastError());
}

}  // namespace decode
}  // namespace mip
