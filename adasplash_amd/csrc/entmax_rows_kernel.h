// Row-wise alpha-entmax forward / backward for gfx950: the kernels and their dispatch for one element type.
//
// Forward: y[r, j] = [(alpha-1) x[r, j] - tau_r]_+^(1/(alpha-1)).  The kernel is HBM-bound: a row is read
// from HBM exactly once (16-byte loads, the whole row then lives in registers), the threshold is solved on the
// few entries that can be in the support, and the result is written once.  A row that does not start or end on a
// 16-byte boundary (an odd number of columns) keeps aligned 16-byte accesses for its inner part; the up to
// fifteen bytes at either end are an extra register slot of the row's first sixteen lanes, an element each, and the chunks are dealt out from a 128-byte line on
// (fp32 [2048, 32001] forward and backward: 665 us when such rows took the streaming kernels, which re-read the row per
// pass with 4-byte accesses, 196 us with the edges in two lanes, 183 us = 5.7 TB/s now; [1024, 65536]: 1003 and 195 us).  Rows longer than the registers of
// 1024 threads hold take a streaming variant that re-reads the row (from L2) per pass.  Semantics follow
// adasplash/triton_entmax_v2.py:363-536.
#pragma once
#include "common.h"
#include "solver.h"

namespace adsp {

enum AlphaMode { AM_15 = 0, AM_2 = 1, AM_GEN = 2 };

struct RowsParams {
  const void* x;
  void* y;
  long long rows, cols;
  float scale;   // alpha - 1
  float c0;      // 1 / (alpha - 1)
  float inv_c0;  // alpha - 1
};

// ---- reductions across the TPR threads that share a row ---------------------------------------------
template <int TPR> __device__ __forceinline__ float row_max(float v, float* sm) {
  if constexpr (TPR == 16) return group16_max(v);
  v = wave_max(v);
  if constexpr (TPR > 64) {
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = v;
    __syncthreads();
    v = sm[0];
#pragma unroll
    for (int w = 1; w < TPR / 64; ++w) v = fmaxf(v, sm[w]);
  }
  return v;
}
template <int TPR, int K> __device__ __forceinline__ void row_sum(float (&v)[K], float* sm) {
  if constexpr (TPR == 16) {
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = group16_sum(v[k]);
    return;
  }
#pragma unroll
  for (int k = 0; k < K; ++k) v[k] = wave_sum(v[k]);
  if constexpr (TPR > 64) {
    __syncthreads();
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
      for (int k = 0; k < K; ++k) sm[(threadIdx.x >> 6) * K + k] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
      float s = sm[k];
#pragma unroll
      for (int w = 1; w < TPR / 64; ++w) s += sm[w * K + k];
      v[k] = s;
    }
  }
}

template <int AM> __device__ __forceinline__ float prob(float u, float c0) {
  // u = z - tau (may be <= 0)
  if constexpr (AM == AM_2) return fmaxf(u, 0.f);
  if constexpr (AM == AM_15) {
    float r = fmaxf(u, 0.f);
    return r * r;
  }
  return u > 0.f ? fast_exp2(fast_log2(u) * c0) : 0.f;
}

template <int AM> __device__ __forceinline__ void accum_stats(float u, float c0, float (&a)[2]) {
  if constexpr (AM == AM_2) {
    a[0] += fmaxf(u, 0.f);
    a[1] += u > 0.f ? 1.f : 0.f;
  } else if constexpr (AM == AM_15) {
    float r = fmaxf(u, 0.f);
    a[0] = fmaf(r, r, a[0]);
    a[1] += r;
  } else {
    if (u > 0.f) {
      float uc = fmaxf(u, 1e-6f);  // same clamp as the reference's masked power (triton_entmax_v2.py:35-39)
      float lg = fast_log2(uc);
      a[0] += fast_exp2(lg * c0);
      a[1] += fast_exp2(lg * (c0 - 1.f));
    }
  }
}

// The threshold of a row whose largest scaled element is `m`, generic over how the elements z are visited:
// `Row::for_each(f)` calls f(z) for every element this thread owns (invalid slots yield -inf).
//
// Newton's method from t = m - 1 on h(t) = (sum_j [z_j - t]_+^c0)^(1/c0) - 1, c0 = 1/(alpha - 1) >= 1.  h is a c0-norm of the
// positive parts, hence convex and decreasing, and h(m - 1) >= 0: the iteration rises to the root without passing it.
// While the support does not change h is nearly a straight line (sum_j [z_j - t]_+^c0 itself is a power of it), so four to
// six steps do, each with two sums, where the reference's Halley steps from a histogram bracket (triton_entmax_v2.py:43-110,
// 415-447) need the histogram, three sums per step and as many steps again for the last digits.  The number of steps the
// caller asks for (`n_iter`) bounds an iteration that stops short; this one runs until the sum is 1 to rounding level, or
// (at large |tau|, where the spacing of floats keeps the sum above any fixed bound) until a step no longer moves t.
template <int AM, int TPR, typename Row>
__device__ __forceinline__ float solve_row(const Row& row, float m, const RowsParams& p, float* sm) {
  float t = m - 1.f;
  if (AM == AM_GEN && p.c0 < 1.f) {
    // alpha > 2: the sum is not convex; bisection on [m - 1, m] to the spacing of floats
    float lo = t, hi = m;
    for (int it = 0; it < 40; ++it) {
      const float mid = 0.5f * (lo + hi);
      float a[2] = {0.f, 0.f};
      row.for_each([&](float z) { accum_stats<AM>(z - mid, p.c0, a); });
      row_sum<TPR, 2>(a, sm);
      if (a[0] > 1.f) lo = mid;
      else hi = mid;
      if (!(hi - lo > 6e-8f * fmaxf(fabsf(lo), 1.f))) break;
    }
    return 0.5f * (lo + hi);
  }
  for (int it = 0; it < 64; ++it) {
    float a[2] = {0.f, 0.f};
    row.for_each([&](float z) { accum_stats<AM>(z - t, p.c0, a); });
    row_sum<TPR, 2>(a, sm);
    float step;
    if constexpr (AM == AM_2) step = a[0] - 1.f;
    else if constexpr (AM == AM_15) step = a[0] - __builtin_amdgcn_sqrtf(a[0]);
    else step = a[0] - fast_exp2(fast_log2(a[0]) * (1.f - p.inv_c0));
    step = a[1] > 0.f ? step * fast_rcp(a[1]) : 0.f;
    t += step;
    if (fabsf(a[0] - 1.f) <= 2e-6f || !(fabsf(step) > 1.2e-7f * fabsf(t))) break;
  }
  return t;
}

// ---- streaming rows (any length / alignment): one 256-thread block per row, scalar accesses --------
template <typename T> __device__ __forceinline__ float load_elem(const void* base, size_t i);
template <> __device__ __forceinline__ float load_elem<float>(const void* b, size_t i) { return ((const float*)b)[i]; }
template <> __device__ __forceinline__ float load_elem<bf16_t>(const void* b, size_t i) {
  return bf16_bits_to_float(((const uint16_t*)b)[i]);
}
template <> __device__ __forceinline__ float load_elem<f16_t>(const void* b, size_t i) {
  return f16_bits_to_float(((const uint16_t*)b)[i]);
}
template <typename T> __device__ __forceinline__ void store_elem(void* base, size_t i, float v);
template <> __device__ __forceinline__ void store_elem<float>(void* b, size_t i, float v) { ((float*)b)[i] = v; }
template <> __device__ __forceinline__ void store_elem<bf16_t>(void* b, size_t i, float v) {
  ((uint16_t*)b)[i] = (uint16_t)float_to_bf16_bits(v);
}
template <> __device__ __forceinline__ void store_elem<f16_t>(void* b, size_t i, float v) {
  ((uint16_t*)b)[i] = (uint16_t)float_to_f16_bits(v);
}

template <typename T, int TPR> struct StreamRow {
  const void* x;
  size_t base;
  long long cols;
  float scale;
  int t_in_row;
  template <typename F> __device__ __forceinline__ void for_each(F f) const {
    for (long long j = t_in_row; j < cols; j += TPR) f(load_elem<T>(x, base + j) * scale);
  }
};

// ---- register-resident rows ------------------------------------------------------------------------
// The row stays in registers as loaded (raw 16-byte chunks).  Only entries with z >= max - 1 can be in the
// support (tau >= max - 1 for every alpha), so after the max pass those candidates are compacted into a
// short LDS list and the whole threshold solve runs on that list inside one wave; the other entries are
// touched twice more at most: one compare against the candidate threshold and one against tau, both
// done per 16-byte chunk on the chunk's maximum.  Rows with more candidates than the list holds fall
// back to solving on the full register copy.
constexpr int kCandPerLane = 16;
constexpr int kCandCap = 64 * kCandPerLane;  // list capacity per row

template <typename T> __device__ __forceinline__ float chunk_elem(u32x4 raw, int e) {
  // the element is copied to a scalar first: bit-casting a vector-element expression directly makes this
  // compiler read element 0 whatever the index
  if constexpr (elem_traits<T>::kVec == 4) {
    const uint32_t w = raw[e];
    return __builtin_bit_cast(float, w);
  } else {
    const uint32_t w = raw[e >> 1];
    return (e & 1) ? unpack_hi<T>(w) : unpack_lo<T>(w);
  }
}

template <int K> struct ListRow {
  float z[K];
  template <typename F> __device__ __forceinline__ void for_each(F f) const {
#pragma unroll
    for (int i = 0; i < K; ++i) f(z[i]);
  }
  // thread t of the `stride` threads that solve the list takes entries t, t + stride, ...
  __device__ __forceinline__ void load(const float* list, int n, int t, int stride = 64) {
#pragma unroll
    for (int i = 0; i < K; ++i) {
      const int idx = i * stride + t;
      z[i] = idx < n ? list[idx] : -INFINITY;
    }
  }
};

// (Register budget: everything is compiled for four waves per SIMD, 128 registers: a block of 1024 threads needs it, and so do
// the shorter rows to keep enough loads in flight.)
template <int TPR> constexpr int rows_threads() { return TPR > 256 ? TPR : 256; }

// A row as the threads that share it see it: `nvec` aligned 16-byte chunks from element `head` on, and with EDGE the elements
// in front of and behind them, one to a lane: the row's first lanes hold the front ones, those from the ninth on the ones at the end (two lanes with up to seven
// each took a load and a store an element: of the figures below, bf16, 16384 x 8191 104.5 -> 91.4).  With EDGE the lanes' places start
// `lead` chunks in front of the first, on a 128-byte line: a wave's load or store then takes whole lines, where one that starts and ends inside a line
// costs that line twice.  `places`: how many the row's lanes have.  us, forward and backward, chunk 0 in the first lane and two lanes with all edge
// elements -> this: fp32, 2048 x 32001: 97.8, 96.4 -> 89.4, 93.5; 32768 x 2047: 95.5, 98 -> 86.8, 95; bf16, 16384 x 8191: 104.2, 112 -> 87.9, 94.7; 2048 x 50000: 75.3, 78.2 -> 71.2,
// 73.3; 32768 x 1000: 31, 36.6 -> 24.5, 26.6.
template <typename T, bool EDGE> struct RowSpan {
  size_t base;       // index of the row's first element
  long long nvec;
  int lead;          // (0 without EDGE, and where the row has no place to spare)
  int head;          // elements in front of the chunks (0 without EDGE)
  long long e0;      // this lane's edge element: index in the row
  bool edge;         // whether it has one
  __device__ __forceinline__ RowSpan(const void* x, long long row, long long cols, int t_in_row, int places) {
    constexpr int kVec = elem_traits<T>::kVec;
    base = (size_t)row * cols;
    head = 0;
    lead = 0;
    e0 = 0;
    edge = false;
    if constexpr (EDGE) {
      const uint32_t addr = (uint32_t)(uintptr_t)x + (uint32_t)base * elem_traits<T>::kBytes;
      head = (int)((0u - addr) & 15u) / elem_traits<T>::kBytes;
      nvec = (cols - head) / kVec;  // (at least one: the dispatch asks for 2 kVec - 1 columns and more)
      const int tail = (int)(cols - head - nvec * kVec);
      e0 = t_in_row < 8 ? t_in_row : cols - tail + (t_in_row - 8);
      edge = t_in_row < head || (t_in_row >= 8 && t_in_row < 8 + tail);
      lead = (int)((addr + (uint32_t)head * elem_traits<T>::kBytes) >> 4) & 7;
      lead = nvec + lead <= places ? lead : 0;
    } else {
      nvec = cols / kVec;
    }
  }
  __device__ __forceinline__ const u32x4* chunks(const void* x) const {
    return reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(x) + (base + head) * elem_traits<T>::kBytes);
  }
  __device__ __forceinline__ u32x4* chunks(void* y) const {
    return reinterpret_cast<u32x4*>(reinterpret_cast<char*>(y) + (base + head) * elem_traits<T>::kBytes);
  }
  // the lane's edge element of `x`, `fill` where it has none
  __device__ __forceinline__ float load_edge(const void* x, float fill) const { return edge ? load_elem<T>(x, base + e0) : fill; }
};

template <typename T, int AM, int NCHUNK, int TPR, bool EDGE>
__global__ __launch_bounds__(rows_threads<TPR>()) __attribute__((amdgpu_waves_per_eu(4))) void entmax_rows_reg_kernel(RowsParams p) {
  constexpr int kVec = elem_traits<T>::kVec;
  constexpr int kRowsPerBlock = rows_threads<TPR>() / TPR;
  __shared__ float sm[32];
  // Short rows (16 threads each, four to a wave): the row's own 16 lanes solve its list.
  constexpr int kCap = TPR == 16 ? (NCHUNK * TPR * kVec < 512 ? NCHUNK * TPR * kVec : 512) : kCandCap;
  __shared__ float cand[kRowsPerBlock][kCap];
  __shared__ int cand_n[kRowsPerBlock];
  const int tid = threadIdx.x;
  const int t_in_row = tid % TPR, r_in_blk = tid / TPR, lane = tid & 63;
  long long row = (long long)blockIdx.x * kRowsPerBlock + r_in_blk;
  // TPR >= 256: one row per block, every thread is active.  TPR == 64: a wave owns a row, and a wave
  // past the last row simply leaves (no block-level barrier is used in that configuration).
  if (row >= p.rows) return;

  const RowSpan<T, EDGE> span(p.x, row, p.cols, t_in_row, NCHUNK * TPR);
  const long long nvec = span.nvec;
  const int t_place = t_in_row - span.lead;
  const u32x4* xrow = span.chunks(p.x);
  u32x4* yrow = span.chunks(p.y);

  struct {
    u32x4 raw[NCHUNK];
    bool valid[NCHUNK];
  } r;
#pragma unroll
  for (int c = 0; c < NCHUNK; ++c) {
    long long vi = (long long)c * TPR + t_place;
    r.valid[c] = EDGE ? (unsigned long long)vi < (unsigned long long)nvec : vi < nvec;
    // a lane outside the row re-reads the row's last chunk and ignores it: no branch between the loads
    r.raw[c] = __builtin_nontemporal_load(xrow + (r.valid[c] ? vi : nvec - 1));
  }
  float ev = -INFINITY;
  if constexpr (EDGE) ev = span.load_edge(p.x, -INFINITY);
  if (t_in_row == 0) cand_n[r_in_blk] = 0;

  // pass 1: per-chunk and row maxima, in the input's own units
  float cmax[NCHUNK];
  float xm = -INFINITY;
#pragma unroll
  for (int c = 0; c < NCHUNK; ++c) {
    float cm = -INFINITY;
    if constexpr (kVec == 4) {
#pragma unroll
      for (int e = 0; e < 4; ++e) cm = fmaxf(cm, chunk_elem<T>(r.raw[c], e));
    } else if constexpr (sizeof(T) == 2 && elem_traits<T>::kIsBf16) {
      // bf16: the upper element of a dword is compared as the dword itself (the lower element only adds
      // mantissa bits below one bf16 ulp), so a chunk maximum may exceed the true one by less than an
      // ulp -- harmless for the two "can this chunk matter" tests, and removed from the row maximum below
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t w = r.raw[c][e];
        cm = fmaxf(cm, fmaxf(__builtin_bit_cast(float, w), __builtin_bit_cast(float, w << 16)));
      }
    } else {
      // f16: packed maxima of the words (unpacking all of them here leaves the compiler two registers per word to keep)
      typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
      uint32_t w[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = r.raw[c][e];
      const f16x2 a = __builtin_elementwise_max(__builtin_bit_cast(f16x2, w[0]), __builtin_bit_cast(f16x2, w[1]));
      const f16x2 b = __builtin_elementwise_max(__builtin_bit_cast(f16x2, w[2]), __builtin_bit_cast(f16x2, w[3]));
      const f16x2 m2 = __builtin_elementwise_max(a, b);
      cm = fmaxf((float)m2[0], (float)m2[1]);
    }
    cmax[c] = r.valid[c] ? cm : -INFINITY;
    xm = fmaxf(xm, cmax[c]);
  }
  if constexpr (EDGE) xm = fmaxf(xm, ev);
  xm = row_max<TPR>(xm, sm);  // (TPR >= 256: its barriers also publish cand_n = 0)
  if constexpr (elem_traits<T>::kIsBf16) xm = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, xm) & 0xffff0000u);

  // pass 2: compact the candidates z >= max - 1 into the row's LDS list
  const float x_thr = xm - p.c0;  // (alpha-1) x >= (alpha-1) xm - 1
#pragma unroll
  for (int c = 0; c < NCHUNK; ++c) {
    if (cmax[c] >= x_thr) {
#pragma unroll
      for (int e = 0; e < kVec; ++e) {
        const float x = chunk_elem<T>(r.raw[c], e);
        if (x >= x_thr) {
          const int idx = atomicAdd(&cand_n[r_in_blk], 1);
          if (idx < kCap) cand[r_in_blk][idx] = x * p.scale;
        }
      }
    }
  }
  if constexpr (EDGE) {
    if (span.edge && ev >= x_thr) {
      const int idx = atomicAdd(&cand_n[r_in_blk], 1);
      if (idx < kCap) cand[r_in_blk][idx] = ev * p.scale;
    }
  }
  if constexpr (TPR > 64) __syncthreads();
  const int n_cand = cand_n[r_in_blk];

  float tau;
  if constexpr (TPR == 16) {
    if (n_cand <= 16) {
      ListRow<1> lr;
      lr.load(cand[r_in_blk], n_cand, t_in_row, 16);
      tau = solve_row<AM, 16>(lr, xm * p.scale, p, sm);
    } else if (n_cand <= kCap) {
      ListRow<kCap / 16> lr;
      lr.load(cand[r_in_blk], n_cand, t_in_row, 16);
      tau = solve_row<AM, 16>(lr, xm * p.scale, p, sm);
    } else {
      StreamRow<T, 16> sr{p.x, (size_t)row * p.cols, p.cols, p.scale, t_in_row};
      tau = solve_row<AM, 16>(sr, xm * p.scale, p, sm);
    }
  } else if (n_cand <= 64) {
    // every wave of the row solves the same short list redundantly: wave-level reductions only.  The
    // usual case (a peaked row) has at most one candidate per lane.
    ListRow<1> lr;
    lr.load(cand[r_in_blk], n_cand, lane);
    tau = solve_row<AM, 64>(lr, xm * p.scale, p, sm);
  } else if (n_cand <= kCandCap) {
    ListRow<kCandPerLane> lr;
    lr.load(cand[r_in_blk], n_cand, lane);
    tau = solve_row<AM, 64>(lr, xm * p.scale, p, sm);
  } else {
    // too many candidates for the list: solve on the whole row, re-read (from L2) pass by pass
    StreamRow<T, TPR> sr{p.x, (size_t)row * p.cols, p.cols, p.scale, t_in_row};
    tau = solve_row<AM, TPR>(sr, xm * p.scale, p, sm);
  }

  // pass 3: outputs; a chunk whose maximum is not above tau is all zeros
#pragma unroll
  for (int c = 0; c < NCHUNK; ++c) {
    if (r.valid[c]) {
      long long vi = (long long)c * TPR + t_place;
      u32x4 o = {0u, 0u, 0u, 0u};
      if (cmax[c] * p.scale > tau) {
        if constexpr (kVec == 4) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            o[e] = __builtin_bit_cast(uint32_t, prob<AM>(chunk_elem<T>(r.raw[c], e) * p.scale - tau, p.c0));
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            o[e] = pack2<T>(prob<AM>(chunk_elem<T>(r.raw[c], 2 * e) * p.scale - tau, p.c0),
                            prob<AM>(chunk_elem<T>(r.raw[c], 2 * e + 1) * p.scale - tau, p.c0));
        }
      }
      __builtin_nontemporal_store(o, yrow + vi);
    }
  }
  if constexpr (EDGE) {
    if (span.edge) store_elem<T>(p.y, span.base + span.e0, prob<AM>(ev * p.scale - tau, p.c0));
  }
}

template <typename T, int AM> __global__ __launch_bounds__(256) void entmax_rows_stream_kernel(RowsParams p) {
  __shared__ float sm[32];
  for (long long row = blockIdx.x; row < p.rows; row += gridDim.x) {
    StreamRow<T, 256> r{p.x, (size_t)row * p.cols, p.cols, p.scale, (int)threadIdx.x};
    float m = -INFINITY;
    r.for_each([&](float z) { m = fmaxf(m, z); });
    const float tau = solve_row<AM, 256>(r, row_max<256>(m, sm), p, sm);
    for (long long j = threadIdx.x; j < p.cols; j += 256) {
      float z = load_elem<T>(p.x, r.base + j) * p.scale;
      store_elem<T>(p.y, r.base + j, prob<AM>(z - tau, p.c0));
    }
  }
}

// ---- backward: dx = u*dy - (sum u*dy / sum u) * u, u = y^(2-alpha) on y > 0 (triton_entmax_v2.py:541-617)
template <typename T, int AM> __global__ __launch_bounds__(256) void entmax_rows_bwd_kernel(
    const void* y, const void* dy, void* dx, long long rows, long long cols, float cf) {
  __shared__ float sm[32];
  for (long long row = blockIdx.x; row < rows; row += gridDim.x) {
    const size_t base = (size_t)row * cols;
    float s[2] = {0.f, 0.f};
    for (long long j = threadIdx.x; j < cols; j += 256) {
      float yy = load_elem<T>(y, base + j);
      float g = load_elem<T>(dy, base + j);
      float u = 0.f;
      if (yy > 0.f) u = (AM == AM_2) ? 1.f : (AM == AM_15 ? sqrtf(yy) : fast_exp2(fast_log2(fmaxf(yy, 1e-6f)) * cf));
      s[0] = fmaf(u, g, s[0]);
      s[1] += u;
    }
    row_sum<256, 2>(s, sm);
    const float q = s[1] > 0.f ? s[0] / s[1] : 0.f;
    for (long long j = threadIdx.x; j < cols; j += 256) {
      float yy = load_elem<T>(y, base + j);
      float g = load_elem<T>(dy, base + j);
      float u = 0.f;
      if (yy > 0.f) u = (AM == AM_2) ? 1.f : (AM == AM_15 ? sqrtf(yy) : fast_exp2(fast_log2(fmaxf(yy, 1e-6f)) * cf));
      store_elem<T>(dx, base + j, u * g - q * u);
    }
    __syncthreads();
  }
}

// Register-resident backward: y and dy are read from HBM once (16-byte non-temporal loads), dx is written
// once.  The support of an entmax row is small, so most 16-byte chunks of y are all zeros: their dy is never
// loaded and their dx is stored as zeros without arithmetic.
template <int AM> __device__ __forceinline__ float bwd_u(float yy, float cf) {
  if (!(yy > 0.f)) return 0.f;
  if constexpr (AM == AM_2) return 1.f;
  if constexpr (AM == AM_15) return __builtin_amdgcn_sqrtf(yy);  // one instruction, 1 ulp
  return fast_exp2(fast_log2(fmaxf(yy, 1e-6f)) * cf);
}

// Rows of more than 8 chunks per lane that are shared by more than 256 threads do not keep dy in registers between the sums
// and the result: it is read a second time (a chunk or two of a lane, from L2).
template <typename T, int AM, int NCHUNK, int TPR, bool EDGE>
__global__ __launch_bounds__(rows_threads<TPR>()) void entmax_rows_bwd_reg_kernel(const void* y, const void* dy, void* dx,
                                                                     long long rows, long long cols, float cf) {
  constexpr int kVec = elem_traits<T>::kVec;
  constexpr int kRowsPerBlock = rows_threads<TPR>() / TPR;
  constexpr bool kKeepDy = NCHUNK <= 8 || TPR <= 256;
  __shared__ float sm[32];
  const int tid = threadIdx.x;
  const int t_in_row = tid % TPR, r_in_blk = tid / TPR;
  const long long row = (long long)blockIdx.x * kRowsPerBlock + r_in_blk;
  if (row >= rows) return;  // TPR >= 256: the whole block; TPR == 64: a wave, and no block barrier is used
  const RowSpan<T, EDGE> span(y, row, cols, t_in_row, NCHUNK * TPR);
  const long long nvec = span.nvec;
  const int t_place = t_in_row - span.lead;
  const u32x4* yrow = span.chunks(y);
  const u32x4* grow = span.chunks(dy);
  u32x4* xrow = span.chunks(dx);

  u32x4 yr[NCHUNK], gr[kKeepDy ? NCHUNK : 1];
  bool valid[NCHUNK], live[NCHUNK];
  // every lane loads (a lane past the row end re-reads the row's last chunk and ignores it): no branches, so
  // all the loads of a row are in flight together
#pragma unroll
  for (int c = 0; c < NCHUNK; ++c) {
    const long long vi = (long long)c * TPR + t_place;
    valid[c] = EDGE ? (unsigned long long)vi < (unsigned long long)nvec : vi < nvec;
    yr[c] = __builtin_nontemporal_load(yrow + (valid[c] ? vi : nvec - 1));
  }
#pragma unroll
  for (int c = 0; c < NCHUNK; ++c) live[c] = valid[c] && (yr[c][0] | yr[c][1] | yr[c][2] | yr[c][3]) != 0u;
  // dy matters only where y has a non-zero element: the other lanes re-read the row's first chunk (one cached
  // line per wave instead of a kilobyte of HBM traffic) so that these loads need no branch either
  if constexpr (kKeepDy) {
#pragma unroll
    for (int c = 0; c < NCHUNK; ++c) gr[c] = __builtin_nontemporal_load(grow + (live[c] ? (long long)c * TPR + t_place : 0ll));
  }
  float ey = 0.f, eg = 0.f;
  if constexpr (EDGE) {
    ey = span.load_edge(y, 0.f);
    eg = span.load_edge(dy, 0.f);
  }
  float s[2] = {0.f, 0.f};
#pragma unroll
  for (int c = 0; c < NCHUNK; ++c) {
    if (live[c]) {
      const u32x4 g = kKeepDy ? gr[kKeepDy ? c : 0] : grow[(long long)c * TPR + t_place];
#pragma unroll
      for (int e = 0; e < kVec; ++e) {
        const float u = bwd_u<AM>(chunk_elem<T>(yr[c], e), cf);
        s[0] = fmaf(u, chunk_elem<T>(g, e), s[0]);
        s[1] += u;
      }
    }
  }
  if constexpr (EDGE) {
    const float u = bwd_u<AM>(ey, cf);
    s[0] = fmaf(u, eg, s[0]);
    s[1] += u;
  }
  row_sum<TPR, 2>(s, sm);
  const float q = s[1] > 0.f ? s[0] / s[1] : 0.f;
#pragma unroll
  for (int c = 0; c < NCHUNK; ++c) {
    if (valid[c]) {
      u32x4 o = {0u, 0u, 0u, 0u};
      if (live[c]) {
        const u32x4 g = kKeepDy ? gr[kKeepDy ? c : 0] : grow[(long long)c * TPR + t_place];
        if constexpr (kVec == 4) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            o[e] = __builtin_bit_cast(uint32_t, bwd_u<AM>(chunk_elem<T>(yr[c], e), cf) * (chunk_elem<T>(g, e) - q));
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            o[e] = pack2<T>(bwd_u<AM>(chunk_elem<T>(yr[c], 2 * e), cf) * (chunk_elem<T>(g, 2 * e) - q),
                            bwd_u<AM>(chunk_elem<T>(yr[c], 2 * e + 1), cf) * (chunk_elem<T>(g, 2 * e + 1) - q));
        }
      }
      __builtin_nontemporal_store(o, xrow + (long long)c * TPR + t_place);
    }
  }
  if constexpr (EDGE) {
    if (span.edge) store_elem<T>(dx, span.base + span.e0, bwd_u<AM>(ey, cf) * (eg - q));
  }
}

// ---- host dispatch ---------------------------------------------------------------------------------
// How a row of `nvec` 16-byte chunks is shared out.  Up to 128 chunks: 16 threads per row, four rows to a wave, so that the
// per-row solve is shared out.  Up to 512: a wave per row (no block barriers).  Beyond that four waves, where more loads in
// flight per row pay more than the barriers cost (2^27-element problems: bf16 4096 columns 74 % of HBM peak with a wave per
// row against 42 %, 8192 columns 66 % against 74-77 %), and from 4096 chunks on eight or sixteen, which keeps a lane at
// 16 chunks.  CALL(NCHUNK, TPR) is expanded for the first entry that holds the row; the edges of a ragged row are extra.
#define ADSP_ROWS_DISPATCH(nvec, CALL)        \
  do {                                        \
    const long long n_ = (nvec);              \
    if (n_ <= 16) CALL(1, 16);                \
    else if (n_ <= 32) CALL(2, 16);           \
    else if (n_ <= 64) CALL(4, 16);           \
    else if (n_ <= 128) CALL(8, 16);          \
    else if (n_ <= 256) CALL(4, 64);          \
    else if (n_ <= 512) CALL(8, 64);          \
    else if (n_ <= 1024) CALL(4, 256);        \
    else if (n_ <= 2048) CALL(8, 256);        \
    else if (n_ <= 4096) CALL(16, 256);       \
    else if (n_ <= 8192) CALL(16, 512);       \
    else CALL(16, 1024);                      \
  } while (0)
constexpr long long kRowsMaxChunks = 16384;

// HIP takes launches of fewer than 2^32 threads: whether `rows` rows of `nvec` chunks stay below it, rounded up to whole blocks.
inline bool rows_fit_grid(long long rows, long long nvec) {
  long long threads = 0;
#define ADSP_ROWS_THREADS(NC, TPR) threads = (rows + rows_threads<TPR>() / TPR - 1) / (rows_threads<TPR>() / TPR) * rows_threads<TPR>()
  ADSP_ROWS_DISPATCH(nvec, ADSP_ROWS_THREADS);
  return threads < (1ll << 32);
}

// The places that rows of `nvec` chunks ask for: where they do not start on a line, up to seven more, in front of the first chunk.  Rows of a few
// hundred bytes do without where they have none to spare (32768 rows, bf16, 249 columns: 13.7 us with, 9.8 without; fp32, 125: 8.6, 7.7; beyond the line bf16,
// 1019: 26.0, 30.1; fp32, 505: 23.6, 27.4).  So do longer ones where the seven would take them to an instance of as many threads and twice the chunks a thread, half of
// them empty, or forward to the one of 1024 threads.  us, 96 MiB in bf16 and as many chunks in fp32, seven
// places always -> so: bf16, 250 chunks 38.5 -> 35.0, and one column more 40.9 -> 36.0; 1018 37.4 -> 34.7; 8186 41.9 -> 36.6; backward fp32, 2042 and one column more 40.4 -> 37.7, bf16
// 42.2 -> 39.0.  At the other lines the next instance has more threads: fp32, 125 chunks 43.3 with none, 34.3 with seven; 509 36.4, 34.4; 4093 40.1, 37.3; backward bf16, 8189 39.9, 37.3.
constexpr long long kRowsShort = 64;
inline long long rows_places(long long rows, long long nvec, int shape, bool backward) {
  if (shape != 1 || nvec <= kRowsShort || !rows_fit_grid(rows, nvec + 7)) return nvec;
  auto over = [nvec](long long line) { return nvec <= line && nvec + 7 > line; };
  if (over(256) || over(1024) || over(2048) || (!backward && over(8192))) return nvec;
  return nvec + 7;
}

// 0: the rows' chunks are aligned and fill them, and the rows start on 128-byte lines or are short; 1: they have edges, or start inside a line; 2: neither (bases that differ in their offset from a 16-byte
// boundary, elements off their own alignment, very short ragged rows, more chunks than the registers hold, more rows than a
// launch of the register kernels holds): stream it
template <typename T> static int rows_shape(uintptr_t a, uintptr_t b, uintptr_t c, long long rows, long long cols) {
  constexpr int kVec = elem_traits<T>::kVec;
  if (cols / kVec > kRowsMaxChunks || rows >= (1ll << 32) || !rows_fit_grid(rows, cols / kVec)) return 2;
  const bool whole = ((a | b | c) & 15) == 0 && cols % kVec == 0;
  if (whole && (cols / kVec <= kRowsShort || (((a | b | c) & 127) == 0 && cols * elem_traits<T>::kBytes % 128 == 0))) return 0;
  if (((a ^ b) & 15) != 0 || ((a ^ c) & 15) != 0 || a % elem_traits<T>::kBytes != 0 || cols < 2 * kVec - 1) return 2;
  return 1;
}

template <typename T, int AM> static void launch_fwd(const RowsParams& p, hipStream_t s) {
  const int shape = rows_shape<T>((uintptr_t)p.x, (uintptr_t)p.y, (uintptr_t)p.x, p.rows, p.cols);
  if (shape == 2) {
    const long long blocks = p.rows < 65536 ? p.rows : 65536;
    hipLaunchKernelGGL((entmax_rows_stream_kernel<T, AM>), dim3((unsigned)blocks), dim3(256), 0, s, p);
    return;
  }
#define ADSP_ROWS_FWD(NC, TPR)                                                                                              \
  do {                                                                                                                      \
    constexpr int rpb = rows_threads<TPR>() / TPR;                                                                          \
    const dim3 grid((unsigned)((p.rows + rpb - 1) / rpb)), block(rows_threads<TPR>());                                      \
    if (shape == 0) hipLaunchKernelGGL((entmax_rows_reg_kernel<T, AM, NC, TPR, false>), grid, block, 0, s, p);              \
    else hipLaunchKernelGGL((entmax_rows_reg_kernel<T, AM, NC, TPR, true>), grid, block, 0, s, p);                          \
  } while (0)
  ADSP_ROWS_DISPATCH(rows_places(p.rows, p.cols / elem_traits<T>::kVec, shape, false), ADSP_ROWS_FWD);
}

template <typename T, int AM>
static void launch_bwd(const void* y, const void* dy, void* dx, long long rows, long long cols, float cf, hipStream_t s) {
  const int shape = rows_shape<T>((uintptr_t)y, (uintptr_t)dy, (uintptr_t)dx, rows, cols);
  if (shape == 2) {
    const long long blocks = rows < 65536 ? rows : 65536;
    hipLaunchKernelGGL((entmax_rows_bwd_kernel<T, AM>), dim3((unsigned)blocks), dim3(256), 0, s, y, dy, dx, rows, cols, cf);
    return;
  }
#define ADSP_ROWS_BWD(NC, TPR)                                                                                                      \
  do {                                                                                                                              \
    constexpr int rpb = rows_threads<TPR>() / TPR;                                                                                  \
    const dim3 grid((unsigned)((rows + rpb - 1) / rpb)), block(rows_threads<TPR>());                                                \
    if (shape == 0) hipLaunchKernelGGL((entmax_rows_bwd_reg_kernel<T, AM, NC, TPR, false>), grid, block, 0, s, y, dy, dx, rows, cols, cf); \
    else hipLaunchKernelGGL((entmax_rows_bwd_reg_kernel<T, AM, NC, TPR, true>), grid, block, 0, s, y, dy, dx, rows, cols, cf);      \
  } while (0)
  ADSP_ROWS_DISPATCH(rows_places(rows, cols / elem_traits<T>::kVec, shape, true), ADSP_ROWS_BWD);
}

}  // namespace adsp
