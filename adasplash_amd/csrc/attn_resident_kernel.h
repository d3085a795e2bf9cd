// Sparse entmax attention forward for gfx950 with a row's scores resident in registers: 16-bit types, head dims 64 and 128, up to
// kResidentMaxKeys keys.
//
// What bounds it: the vector pipe (an iteration of the solver is three instructions a score, 4 cycles each, and there are four to
// six of them; the products are a tenth of that), and on small calls the chain of load, product, solver and output itself.
//
// Split: a workgroup owns 32 rows, its 4, 8 or 16 waves hold up to four blocks of 32 keys each, so that the scores of a row of up to 2048
// keys are formed once and stay in registers: the solver touches no memory but a few numbers a wave and iteration in LDS,
// and neither lists, nor a second product, nor a saved mask is needed whatever the scores are.  Four waves a SIMD, 128 registers:
// the chunks of K and V come through a ring of two 4 KB chunks a wave, in the order of their use.  The weights are multiplied as the sum
// of two 16-bit values, which the idle matrix pipe does for nothing (relative error for bf16: 2.3e-3 -> 1.7e-3, that of the rounded result).
//
// Newton's steps are taken on (sum u^c0)^(1/c0) - 1, which is convex and nearly linear, from the maximum less 1, where u is at most 1.
// They end with one of up to 4e-4, behind which the weights' relative error is below 6e-6 (alpha = 1.5 and below, 64 to 2048 keys, scores of
// spread 1e-4 to 10).  Towards alpha = 2 the sum becomes piecewise linear, a step leaves what the keys that it puts off the support had, and
// u is itself some 5e-4 where 2048 scores are nearly equal; so a step is also asked to be small beside the mean of u: 2e-3 of it at
// alpha = 2, 5e-3 at a generic alpha, which adds nothing up to 1.333 and a quarter of a step at 1.9 (the weights' error at 1.75, 1.9 and 1.99 without it:
// 2.2e-4, 9e-4, 1.8e-2; with it at most 2.7e-5).
//
// Measured, us, the kernels on the supports or on lists -> this one, q of spread 1, 3 and 1/8: 16 x 12 heads, N <= 500, D = 64: 86 -> 35,
// 64 -> 33, 147 -> 34; 32 x 16 heads, N <= 512, D = 128: 256 -> 122, 172 -> 125, 394 -> 127.  A first solver
// stage on pairs of 16-bit scores (v_dot2) was no faster and is not here.
#pragma once
#include "attn_tile16.h"

namespace adsp {
namespace resident {

using tile16::add_powers;
using f32path::kChunk;
using f32path::kRows;
constexpr int kBlocks = 4;       // blocks of 32 keys a wave holds
constexpr int kMaxWaves = 16;
static_assert(kRows * kBlocks * kMaxWaves == kResidentMaxKeys, "a key beyond the registers would be dropped");

// u clamped to [0, 1] in the fma itself: a score is at most 1 above a threshold that is a bound
__device__ __forceinline__ float above(float s, float qs, float minus_t) { return __builtin_amdgcn_fmed3f(fmaf(s, qs, minus_t), 0.f, 1.f); }
template <int AM> __device__ __forceinline__ float power(float u, float c0) {
  if constexpr (AM == ATT_15) return u * u;
  if constexpr (AM == ATT_2) return u;
  return fast_exp2(fast_log2(u) * c0);
}

template <typename T, int D, int AM, int W>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(4, 4))) void attn_resident_fwd_kernel(AttnParams p) {
  constexpr int kStride = D * 2;
  constexpr int NC = D / 64;  // chunks of 64 columns
  __shared__ __align__(4096) unsigned char smem[W * 2 * kChunk];
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  __shared__ f32x2 red[2][W][kRows];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, lq = lane & 31, lh = lane >> 5;
  const int N = p.N, group = p.Hq / p.Hkv, n_rblk = (N + kRows - 1) / kRows;
  int bkv, mi, hg;
  if (!xcd_block_map(p.varlen != nullptr, p.B * p.Hkv, n_rblk, group, p.causal != 0, 2ll * N * kStride, bkv, mi, hg)) return;
  const int b = bkv / p.Hkv, kvh = bkv % p.Hkv, h = kvh * group + hg;
  const int m0 = (n_rblk - 1 - mi) * kRows;
  int L = N;
  if (p.varlen) {
    const long long l = p.varlen_bits == 64 ? ((const long long*)p.varlen)[b] : (long long)((const int*)p.varlen)[b];
    L = (int)(l < 0 ? 0 : (l > N ? N : l));
  }
  const size_t q_row0 = (size_t)(b * p.Hq + h) * N;
  unsigned char* const out = reinterpret_cast<unsigned char*>(p.out) + q_row0 * kStride;
  if (m0 >= L) {
    const int rows = N - m0 < kRows ? N - m0 : kRows;
    for (int i = tid; i < rows * (kStride / 16); i += 64 * W) reinterpret_cast<f32x4*>(out + (size_t)m0 * kStride)[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    return;
  }
  const unsigned char* kg = reinterpret_cast<const unsigned char*>(p.k) + (size_t)bkv * N * kStride;
  const unsigned char* vg = reinterpret_cast<const unsigned char*>(p.v) + (size_t)bkv * N * kStride;
  const int qi = m0 + lq;
  const bool live = qi < L;
  const int lim = p.causal ? (qi < L - 1 ? qi : L - 1) : L - 1;  // last key of the lane's row
  const int key_hi = p.causal ? (m0 + kRows < L ? m0 + kRows : L) : L;
  const int n_kblk = (key_hi + kRows - 1) / kRows;
  const float qs = p.qscale, c0 = p.c0;

  // A wave holds up to kBlocks blocks, block `wave` and every W-th behind it; each count has code of its own, so that what a
  // wave keeps has its place in registers and no block is worked on for nothing.  (The numbers differ by one at most
  // between the waves, and every count passes the same barriers.)
  const int nb = wave < n_kblk ? (n_kblk - wave + W - 1) / W : 0;
  const int n_w = n_kblk < W ? n_kblk : W;  // waves with a block
  auto run = [&](auto nb_c) {
    constexpr int NB = decltype(nb_c)::value, NB1 = NB > 0 ? NB : 1;
    // ---- the wave's chunks, in the order in which they are used: K block by block, then V 64 columns at a time ----
    f32path::Ring<kStride> ring(smem + wave * (2 * kChunk), lane);
    auto issue = [&](int x) {  // (a constant everywhere)
      if (x < NB * NC) ring.issue(kg, (x / NC * W + wave) * kRows, L, x % NC, x & 1);
      else if (x < 2 * NB * NC) ring.issue_t(vg, ((x - NB * NC) % NB1 * W + wave) * kRows, L, (x - NB * NC) / NB1, x & 1);
    };
    // V's second 64 columns wait until the first are stored: the waves' sums meet in the rings
    auto last_of = [&](int x) { return x < NB * (NC + 1) ? NB * (NC + 1) - 1 : 2 * NB * NC - 1; };
    auto arrive = [&](int x) -> uint32_t {
      if (x < last_of(x)) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      return (uint32_t)(uintptr_t)(smem + wave * (2 * kChunk) + (x & 1) * kChunk);
    };
    auto release = [&](int x) {  // the wave's reads of the chunk are done: its place takes the chunk after next
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (x + 2 <= last_of(x)) issue(x + 2);
      __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (NB > 0) {
      issue(0);
      issue(1);
    }

    // ---- scores ----
    f32x16 s[NB1];
    float mx = -INFINITY;
    {
      const uint32_t rl = f32path::row_lane_of(lq, lh);
      uint32_t qf[16 * NC];
      f32path::load_row<4 * NC>(reinterpret_cast<const unsigned char*>(p.q) + (q_row0 + (live ? qi : L - 1)) * kStride, lh, qf);
#pragma unroll
      for (int kb = 0; kb < NB; ++kb) {
#pragma unroll
        for (int i = 0; i < 16; ++i) s[kb][i] = 0.f;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const uint32_t at = arrive(kb * NC + c) + rl;
          constexpr int kRead = NC == 1 ? 4 : 2;  // operands under way at a time
#pragma unroll
          for (int g0 = 0; g0 < 4; g0 += kRead) {
            u32x4 a[kRead];
#pragma unroll
            for (int g = 0; g < kRead; ++g) a[g] = lds_read16(at ^ ((g0 + g) << 5));
            if (g0 + kRead == 4) release(kb * NC + c);
#pragma unroll
            for (int g = 0; g < kRead; ++g) {
              const int f = 16 * c + 4 * (g0 + g);
              s[kb] = mfma_16bit<T>(a[g], u32x4{qf[f], qf[f + 1], qf[f + 2], qf[f + 3]}, s[kb]);
            }
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        tile16::products_end();
        const int k0 = (kb * W + wave) * kRows;
        if (k0 + kRows > L || (p.causal && k0 + kRows - 1 > m0)) {
          const int jb = k0 + 4 * lh;
#pragma unroll
          for (int i = 0; i < 16; ++i) s[kb][i] = jb + 8 * (i >> 2) + (i & 3) <= lim ? s[kb][i] : -INFINITY;
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[kb][i]);
      }
    }

    // ---- over the waves: each lane adds up (or takes the maximum of) half of the waves' numbers for its row ----
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    if (lh == 0) red[0][wave][lq] = f32x2{mx, 0.f};
    __syncthreads();
#pragma unroll
    for (int w = 0; w < W / 2; ++w) mx = fmaxf(mx, red[0][lh * (W / 2) + w][lq][0]);
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    auto both = [](float x) -> float {  // the two lanes of a row
      const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x), false, false);
      return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
    };
    auto total = [&](int buf, float& a, float& c) {
      a = both(a);
      c = both(c);
      if (lh == 0) red[buf][wave][lq] = f32x2{a, c};
      __syncthreads();
      a = c = 0.f;
#pragma unroll
      for (int w = 0; w < W / 2; ++w) {
        const f32x2 x = red[buf][lh * (W / 2) + w][lq];
        a += x[0];
        c += x[1];
      }
      a = both(a);
      c = both(c);
    };

    // ---- threshold: Newton from the left on the norm ----
    const float t_min = fmaf(mx, qs, -1.f);
    float t = t_min;
    int buf = 1;
    for (int it = 0; it < 48; ++it) {
      float s0 = 0.f, s1 = 0.f;
#pragma unroll
      for (int kb = 0; kb < NB; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i) add_powers<AM>(above(s[kb][i], qs, -t), c0, s0, s1);
      total(buf, s0, s1);
      buf ^= 1;
      const float step = f32path::norm_step<AM>(s0, s1, c0);
      t = fmaxf(t + step, t_min);
      float near = 4e-4f;
      if constexpr (AM != ATT_15) {
        const float beside = (AM == ATT_2 ? 2e-3f : 5e-3f) * s0 * fast_rcp(s1), least = fmaxf(2e-6f, 1.2e-7f * fabsf(t));
        near = fmaxf(AM == ATT_2 ? beside : fminf(beside, 4e-4f), least);
      }
      if (__builtin_amdgcn_ballot_w64(fabsf(step) > near) == 0ull) break;  // (the same sums in every wave)
    }
    if (live && wave == 0 && lh == 0 && p.taus) p.taus[q_row0 + qi] = t;

    // ---- probabilities, each as the sum of two 16-bit values ----
    uint32_t hi[NB1][8], lo[NB1][8];
    float zsum = 0.f, unused = 0.f;
#pragma unroll
    for (int kb = 0; kb < NB; ++kb)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float a = power<AM>(above(s[kb][2 * i], qs, -t), c0), c = power<AM>(above(s[kb][2 * i + 1], qs, -t), c0);
        zsum += a;
        zsum += c;
        hi[kb][i] = pack2<T>(a, c);
        lo[kb][i] = pack2<T>(a - unpack_lo<T>(hi[kb][i]), c - unpack_hi<T>(hi[kb][i]));
      }
    total(buf, zsum, unused);
    const float inv = zsum > 0.f ? 1.f / zsum : 0.f;

    // ---- output, 64 columns at a time ----
    uint32_t ta[2];
    {
      const int a4 = lane & 15, grp = lane >> 4, r = a4 >> 2, c = a4 & 3, dl = grp & 1;
#pragma unroll
      for (int x2 = 0; x2 < 2; ++x2) {
        const int x = 4 * (grp >> 1) + r + 8 * x2;
        ta[x2] = (uint32_t)(x * 128 + (((2 * dl + (c >> 1)) ^ ((2 * x) & 7)) << 4) + (c & 1) * 8);
      }
    }
    using KS = Swz<256>;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if constexpr (NB > 0) {
        f32x16 o[2];
#pragma unroll
        for (int db = 0; db < 2; ++db)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
#pragma unroll
        for (int kb = 0; kb < NB; ++kb) {
          const int ch = NB * NC + c * NB + kb;
          const uint32_t at = arrive(ch);
#pragma unroll
          for (int x = 0; x < 2; ++x) {
            u32x4 a[2];
#pragma unroll
            for (int db = 0; db < 2; ++db) {
              const u32x2_t a0 = lds_read8_tr((at + ta[0]) ^ (db << 6), 16 * x * 128);
              const u32x2_t a1 = lds_read8_tr((at + ta[1]) ^ (db << 6), 16 * x * 128);
              a[db] = u32x4{a0[0], a0[1], a1[0], a1[1]};
            }
            if (x == 1) release(ch);
            const u32x4 ph = {hi[kb][4 * x], hi[kb][4 * x + 1], hi[kb][4 * x + 2], hi[kb][4 * x + 3]};
            const u32x4 pl = {lo[kb][4 * x], lo[kb][4 * x + 1], lo[kb][4 * x + 2], lo[kb][4 * x + 3]};
#pragma unroll
            for (int db = 0; db < 2; ++db) o[db] = mfma_16bit<T>(a[db], ph, o[db]);
#pragma unroll
            for (int db = 0; db < 2; ++db) o[db] = mfma_16bit<T>(a[db], pl, o[db]);
          }
        }
        tile16::products_end();
        unsigned char* const mine = smem + wave * (2 * kChunk);
#pragma unroll
        for (int db = 0; db < 2; ++db)
#pragma unroll
          for (int g = 0; g < 4; ++g)
            *reinterpret_cast<f32x4*>(mine + KS::off(lq, db * 8 + 2 * g + lh)) =
                f32x4{o[db][4 * g] * inv, o[db][4 * g + 1] * inv, o[db][4 * g + 2] * inv, o[db][4 * g + 3] * inv};
      }
      __syncthreads();
      for (int id = tid; id < kRows * 16; id += 64 * W) {
        const int row = id >> 4, c4 = id & 15;
        const int at = KS::off(row, c4);
        f32x4 x = *reinterpret_cast<const f32x4*>(smem + at);
        for (int w = 1; w < n_w; ++w) {
          const f32x4 y = *reinterpret_cast<const f32x4*>(smem + w * (2 * kChunk) + at);
#pragma unroll
          for (int e = 0; e < 4; ++e) x[e] += y[e];
        }
        u32x2 r = {pack2<T>(x[0], x[1]), pack2<T>(x[2], x[3])};
        if (m0 + row >= L) r = u32x2{0u, 0u};
        if (m0 + row < N) *reinterpret_cast<u32x2*>(out + (size_t)(m0 + row) * kStride + c * 128 + c4 * 8) = r;
      }
      if (c + 1 < NC) {
        __syncthreads();
        if constexpr (NB > 0) {
          issue(NB * (NC + 1));
          issue(NB * (NC + 1) + 1);
        }
      }
    }
  };
  switch (nb) {
    case 0: run(std::integral_constant<int, 0>{}); break;
    case 1: run(std::integral_constant<int, 1>{}); break;
    case 2: run(std::integral_constant<int, 2>{}); break;
    case 3: run(std::integral_constant<int, 3>{}); break;
    default: run(std::integral_constant<int, 4>{}); break;
  }
}

}  // namespace resident
}  // namespace adsp
