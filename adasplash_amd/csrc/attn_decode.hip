// Entmax attention of a few new queries against a cache of keys (a decoding step): any alpha > 1, ALiBi slopes, left or
// right padding, causal mask aligned to the bottom right.  Two kernels; the semantics are those of examples/attention.py:34-91.
//
// 1. decode_scores_kernel reads K once and writes z = (alpha - 1) (q k / sqrt(D) + bias) in fp32, [B, H, q_len, k_pad].  It is
//    bound by HBM: a wave takes 64 keys, all of their rows under way together (D = 64 in 16 bits: 8 KB per wave), and the
//    products run on 16 x 16 matrix tiles whose other side is the up to 16 queries -- 16 keys a tile, so that the split over
//    the keys alone fills the chip whatever the batch.
// 2. decode_output_kernel, a workgroup per query row: the row's scores come back from L2, the few that can be in the
//    support (z >= max - 1) go to a list in LDS, the threshold is solved on the list as in the rows kernels, and only the V rows
//    of the support are read.  The list's order, and with it that of every sum over it, is the order of the threads (a prefix sum
//    over their counts), so a call returns the same bits every time.
// A step of 16 x 16 heads against caches of up to 4096 keys (D = 64, bf16, 84 MB of K in use): 265 us as fp32 copies of q and
// K, a library product, ten elementwise launches, the rows kernel and a second product; 27 us now (20 us = 4.2 TB/s and 6.9 us).
#include "entmax_rows_kernel.h"
#include "../../include/adasplash_hip.h"
#include <math.h>

namespace adsp {
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

struct DecodeParams {
  const void *q, *k, *v;
  void* out;
  float* z;
  const void* varlen;
  const float* slopes;
  long long k_sb, k_sh, k_sn, v_sb, v_sh, v_sn;  // strides of K and V in elements: batch, head, key
  int varlen_bits, left, causal;
  int H, q_len, k_len, k_pad;
  float sm_scale, alpha_m1;
  RowsParams rows;  // (the solver's constants)
};
constexpr int kDecodeKeys = 256;  // keys per workgroup of the first kernel
constexpr int kDecodeCap = 1024;  // candidates of a row that fit its list

__device__ __forceinline__ void decode_span(const DecodeParams& p, int b, int& first, int& last) {
  long long len = p.k_len;
  if (p.varlen) {
    len = p.varlen_bits == 64 ? ((const long long*)p.varlen)[b] : (long long)((const int*)p.varlen)[b];
    len = len < 0 ? 0 : (len > p.k_len ? p.k_len : len);
  }
  first = p.left ? p.k_len - (int)len : 0;
  last = first + (int)len;
}

template <typename T> __device__ __forceinline__ f32x4 decode_mfma(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (elem_traits<T>::kVec == 4) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t x = a[e], y = b[e];
      c = __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(float, x), __builtin_bit_cast(float, y), c, 0, 0, 0);
    }
    return c;
  } else if constexpr (elem_traits<T>::kIsBf16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
}

// Operand layout: lane l holds row l % 16 of its matrix, the 16-byte chunk l / 16 of every 64 bytes (the four floats of a
// chunk are four contraction steps; both sides use the same order, so which step takes which column does not matter); of the
// result query l % 16 and keys 4 (l / 16) + 0 .. 3.
template <typename T, int D> __global__ __launch_bounds__(256) void decode_scores_kernel(DecodeParams p) {
  constexpr int kSteps = D * elem_traits<T>::kBytes / 64;
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int bh = blockIdx.y, b = bh / p.H, h = bh % p.H;
  int first, last;
  decode_span(p, b, first, last);
  const int key0 = blockIdx.x * kDecodeKeys + (threadIdx.x >> 6) * 64;
  if (key0 >= last || key0 + 64 <= first) return;
  const char* const kbase = (const char*)p.k + (b * p.k_sb + h * p.k_sh) * elem_traits<T>::kBytes;
  u32x4 kf[4][kSteps], qf[kSteps];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    int key = key0 + j * 16 + r;
    key = key < p.k_len ? key : p.k_len - 1;
    const u32x4* src = reinterpret_cast<const u32x4*>(kbase + key * p.k_sn * elem_traits<T>::kBytes) + g;
#pragma unroll
    for (int s = 0; s < kSteps; ++s) kf[j][s] = src[s * 4];
  }
  {
    const int qi = r < p.q_len ? r : p.q_len - 1;
    const u32x4* src = reinterpret_cast<const u32x4*>((const char*)p.q + ((size_t)bh * p.q_len + qi) * D * elem_traits<T>::kBytes) + g;
#pragma unroll
    for (int s = 0; s < kSteps; ++s) qf[s] = src[s * 4];
  }
  const float slope = p.slopes ? p.slopes[h] : 0.f;
  // (one new query sits on the last key; with several the bias counts from the query's own index: a constant per row either way)
  const int zero_at = (p.q_len == 1 && p.k_len > 1) ? p.k_len - 1 : r;
  const int limit = p.causal ? p.k_len - p.q_len + r : p.k_len - 1;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < kSteps; ++s) acc = decode_mfma<T>(kf[j][s], qf[s], acc);
    const int key = key0 + j * 16 + g * 4;
    f32x4 z;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int at = key + i;
      const float s = acc[i] * p.sm_scale + slope * (float)(at - zero_at);
      z[i] = (at >= first && at < last && at <= limit) ? s * p.alpha_m1 : -INFINITY;
    }
    if (r < p.q_len) *reinterpret_cast<f32x4*>(p.z + ((size_t)bh * p.q_len + r) * p.k_pad + key) = z;
  }
}

template <typename T, int D, int AM> __global__ __launch_bounds__(256) void decode_output_kernel(DecodeParams p) {
  constexpr int kVec = elem_traits<T>::kVec;
  constexpr int kLanes = D / kVec;        // lanes per V row, 16 bytes each
  constexpr int kGroups = 256 / kLanes;   // V rows read side by side
  __shared__ float sm[32];
  __shared__ float list_z[kDecodeCap];
  __shared__ int list_key[kDecodeCap];
  __shared__ int counts[2][4];
  __shared__ float red[4][D];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // Where this thread's `count` entries start in a list that the 256 threads fill in turn, behind the `n` that it holds; `n` becomes
  // the new length.  One barrier: two calls in a row use the two halves of `counts`.
  auto place = [&](int count, int half, int& n) {
    const int upto = wave_prefix_sum(count);
    if (lane == 63) counts[half][wave] = upto;
    __syncthreads();
    const int c0 = counts[half][0], c1 = counts[half][1], c2 = counts[half][2], c3 = counts[half][3];
    const int at = n + upto - count + (wave > 0 ? c0 : 0) + (wave > 1 ? c1 : 0) + (wave > 2 ? c2 : 0);
    n += (c0 + c1) + (c2 + c3);
    return at;
  };
  const int row = blockIdx.x, bh = row / p.q_len, b = bh / p.H, h = bh % p.H;
  int first, last;
  decode_span(p, b, first, last);
  const float* const zrow = p.z + (size_t)row * p.k_pad;
  // whole groups of four keys around [first, last): the scores kernel has written -inf at the keys outside the span
  const int c0 = first >> 2, c1 = first < last ? (last + 3) >> 2 : c0;
  const f32x4* const z4 = reinterpret_cast<const f32x4*>(zrow);
  // eight loads of a thread under way together; a row of up to 8192 keys is then in registers for the second look as well
  constexpr int kHold = 8;
  f32x4 held[kHold];
  const f32x4 none = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
  auto load_held = [&](int from) {
#pragma unroll
    for (int i = 0; i < kHold; ++i) {
      const int c = from + i * 256 + tid;
      held[i] = c < c1 ? z4[c] : none;
    }
  };
  float m = -INFINITY;
  for (int from = c0; from < c1; from += kHold * 256) {
    load_held(from);
#pragma unroll
    for (int i = 0; i < kHold; ++i) m = fmaxf(m, fmaxf(fmaxf(held[i][0], held[i][1]), fmaxf(held[i][2], held[i][3])));
  }
  m = row_max<256>(m, sm);
  float acc[kVec];
#pragma unroll
  for (int e = 0; e < kVec; ++e) acc[e] = 0.f;
  if (m > -INFINITY) {  // (a query that sees no key at all is a row of zeros)
    const float thr = m - 1.f;
    int n = 0, half = 0;
    for (int from = c0; from < c1; from += kHold * 256) {
      if (c1 - c0 > kHold * 256) load_held(from);
      int count = 0;
#pragma unroll
      for (int i = 0; i < kHold; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) count += held[i][e] >= thr ? 1 : 0;
      int at = place(count, half, n);
      half ^= 1;
#pragma unroll
      for (int i = 0; i < kHold; ++i) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float z = held[i][e];
          if (z >= thr) {
            if (at < kDecodeCap) {
              list_z[at] = z;
              list_key[at] = (from + i * 256 + tid) * 4 + e;
            }
            ++at;
          }
        }
      }
    }
    __syncthreads();
    const int grp = tid / kLanes, col = tid % kLanes;
    const char* const vbase = (const char*)p.v + ((size_t)(b * p.v_sb + h * p.v_sh) + col * kVec) * elem_traits<T>::kBytes;
    auto row_of = [&](int key) { return *reinterpret_cast<const u32x4*>(vbase + key * p.v_sn * elem_traits<T>::kBytes); };
    auto add_row = [&](float w, u32x4 raw) {
#pragma unroll
      for (int e = 0; e < kVec; ++e) acc[e] = fmaf(w, chunk_elem<T>(raw, e), acc[e]);
    };
    if (n <= kDecodeCap) {
      float tau;
      if (n <= 64) {
        ListRow<1> lr;
        lr.load(list_z, n, lane);
        tau = solve_row<AM, 64>(lr, m, p.rows, sm);
      } else {
        ListRow<kDecodeCap / 64> lr;
        lr.load(list_z, n, lane);
        tau = solve_row<AM, 64>(lr, m, p.rows, sm);
      }
      // the support, in the list's place: every entry is in a register before the first is written back
      float w[kDecodeCap / 256];
      int key[kDecodeCap / 256];
#pragma unroll
      for (int c = 0; c < kDecodeCap / 256; ++c) {
        const int i = c * 256 + tid;
        w[c] = i < n ? prob<AM>(list_z[i] - tau, p.rows.c0) : 0.f;
        key[c] = i < n ? list_key[i] : 0;
      }
      int count = 0, members = 0;
#pragma unroll
      for (int c = 0; c < kDecodeCap / 256; ++c) count += w[c] > 0.f ? 1 : 0;
      int at = place(count, half, members);  // (its barrier: every thread has read its part of the list)
#pragma unroll
      for (int c = 0; c < kDecodeCap / 256; ++c) {
        if (w[c] > 0.f) {
          list_z[at] = w[c];
          list_key[at] = key[c];
          ++at;
        }
      }
      __syncthreads();
      // four rows of a group under way together; a slot past the end takes the first member's row with weight zero
      for (int i = grp; i < members; i += 4 * kGroups) {
        u32x4 raw[4];
        float wt[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int at = i + u * kGroups;
          wt[u] = at < members ? list_z[at] : 0.f;
          raw[u] = row_of(list_key[at < members ? at : 0]);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) add_row(wt[u], raw[u]);
      }
    } else {
      // a flat row: more candidates than the list holds; solved on the scores in memory, and every key is looked at
      StreamRow<float, 256> sr{zrow + first, 0, (long long)(last - first), 1.f, tid};
      const float tau = solve_row<AM, 256>(sr, m, p.rows, sm);
#pragma unroll 4
      for (int key = first + grp; key < last; key += kGroups) {
        const float w = prob<AM>(zrow[key] - tau, p.rows.c0);
        if (w > 0.f) add_row(w, row_of(key));
      }
    }
  }
  // the groups' sums: within a wave over the lanes of equal column, then over the four waves
#pragma unroll
  for (int o = kLanes; o < 64; o <<= 1)
#pragma unroll
    for (int e = 0; e < kVec; ++e) acc[e] += __shfl_xor(acc[e], o, 64);
  if (lane < kLanes) {
#pragma unroll
    for (int e = 0; e < kVec; ++e) red[tid >> 6][lane * kVec + e] = acc[e];
  }
  __syncthreads();
  for (int d = tid; d < D; d += 256) store_elem<T>(p.out, (size_t)row * D + d, red[0][d] + red[1][d] + red[2][d] + red[3][d]);
}

template <typename T, int D> static void launch_decode(const DecodeParams& p, int B, double alpha, hipStream_t s) {
  const dim3 grid((unsigned)(p.k_pad / kDecodeKeys), (unsigned)(B * p.H)), rows((unsigned)(B * p.H * p.q_len)), block(256);
  hipLaunchKernelGGL((decode_scores_kernel<T, D>), grid, block, 0, s, p);
  if (alpha == 1.5) hipLaunchKernelGGL((decode_output_kernel<T, D, AM_15>), rows, block, 0, s, p);
  else if (alpha == 2.0) hipLaunchKernelGGL((decode_output_kernel<T, D, AM_2>), rows, block, 0, s, p);
  else hipLaunchKernelGGL((decode_output_kernel<T, D, AM_GEN>), rows, block, 0, s, p);
}
template <typename T> static bool launch_decode_d(const DecodeParams& p, int B, int D, double alpha, hipStream_t s) {
  switch (D) {
    case 32: return launch_decode<T, 32>(p, B, alpha, s), true;
    case 64: return launch_decode<T, 64>(p, B, alpha, s), true;
    case 128: return launch_decode<T, 128>(p, B, alpha, s), true;
    case 256: return launch_decode<T, 256>(p, B, alpha, s), true;
  }
  return false;
}
static int decode_pad(int k_len) { return (k_len + kDecodeKeys - 1) / kDecodeKeys * kDecodeKeys; }
}  // namespace adsp

extern "C" size_t adsp_attn_decode_workspace_bytes(int B, int H, int q_len, int k_len) {
  if (B <= 0 || H <= 0 || q_len <= 0 || k_len <= 0) return 0;
  return (size_t)B * H * q_len * adsp::decode_pad(k_len) * 4;
}

extern "C" int adsp_attn_decode_fwd(const void* q, const void* k, const void* v, void* out, const void* varlen, int varlen_bits,
                                    int left_padding, const float* alibi_slopes, int B, int H, int q_len, int k_len, int D,
                                    int64_t k_stride_b, int64_t k_stride_h, int64_t k_stride_n, int64_t v_stride_b,
                                    int64_t v_stride_h, int64_t v_stride_n, int dtype, double alpha, int is_causal, void* workspace,
                                    size_t workspace_bytes, void* stream) {
  using namespace adsp;
  if (!q || !k || !v || !out) return ADSP_ERR_NULL;
  if (dtype != ADSP_F32 && dtype != ADSP_BF16 && dtype != ADSP_F16) return ADSP_ERR_DTYPE;
  if (B <= 0 || H <= 0 || q_len <= 0 || q_len > 16 || k_len <= 0 || k_len > (1 << 24)) return ADSP_ERR_SHAPE;
  if (D != 32 && D != 64 && D != 128 && D != 256) return ADSP_ERR_SHAPE;
  if ((long long)B * H > 65535 || is_causal < 0) return ADSP_ERR_SHAPE;  // (the grid's second dimension)
  if (!(alpha > 1.0)) return ADSP_ERR_UNSUPPORTED;
  if (varlen && varlen_bits != 32 && varlen_bits != 64) return ADSP_ERR_UNSUPPORTED;
  const int es = dtype == ADSP_F32 ? 4 : 2;
  if ((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out) & 15) != 0) return ADSP_ERR_ALIGN;
  if (((k_stride_b | k_stride_h | k_stride_n | v_stride_b | v_stride_h | v_stride_n) * es & 15) != 0) return ADSP_ERR_ALIGN;
  if (!workspace || workspace_bytes < adsp_attn_decode_workspace_bytes(B, H, q_len, k_len) || ((uintptr_t)workspace & 15) != 0)
    return ADSP_ERR_WORKSPACE;
  DecodeParams p;
  p.q = q;
  p.k = k;
  p.v = v;
  p.out = out;
  p.z = (float*)workspace;
  p.varlen = varlen;
  p.varlen_bits = varlen_bits;
  p.left = left_padding ? 1 : 0;
  p.causal = is_causal ? 1 : 0;
  p.slopes = alibi_slopes;
  p.k_sb = k_stride_b;
  p.k_sh = k_stride_h;
  p.k_sn = k_stride_n;
  p.v_sb = v_stride_b;
  p.v_sh = v_stride_h;
  p.v_sn = v_stride_n;
  p.H = H;
  p.q_len = q_len;
  p.k_len = k_len;
  p.k_pad = decode_pad(k_len);
  p.sm_scale = (float)(1.0 / sqrt((double)D));
  p.alpha_m1 = (float)(alpha - 1.0);
  p.rows = RowsParams{};
  p.rows.scale = (float)(alpha - 1.0);
  p.rows.c0 = (float)(1.0 / (alpha - 1.0));
  p.rows.inv_c0 = (float)(alpha - 1.0);
  hipStream_t s = (hipStream_t)stream;
  (void)hipGetLastError();
  if (dtype == ADSP_F32) launch_decode_d<float>(p, B, D, alpha, s);
  else if (dtype == ADSP_BF16) launch_decode_d<bf16_t>(p, B, D, alpha, s);
  else launch_decode_d<f16_t>(p, B, D, alpha, s);
  return hipGetLastError() == hipSuccess ? ADSP_OK : ADSP_ERR_LAUNCH;
}
