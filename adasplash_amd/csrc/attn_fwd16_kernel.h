// Forward of the sparse entmax attention on all pairs of a row, 16-bit types, head dims 64 and 128, for gfx950, for the row blocks
// that the kernels on the supports leave over (flat scores).
//
// What bounds it: matrix and vector pipe together, at the 1.8 - 1.9 GHz that their power leaves (a block of 32 x 32 scores takes two to
// four products of 34 cycles a walk and three vector instructions a score).  So the number of walks over the keys is what counts.
//
// A row's threshold starts from a sample of 256 keys held in registers, where Newton's steps cost no memory; one step on every
// second tile corrects the sampling error, and one or two on all tiles finish it (a step squares what is left; flat scores: two and
// a half walks and the output's).  The output walk's own sums take the threshold that a backward reads one step further.
//
// Split: four waves of 32 rows, tiles of K (and V in the output walk) through two stages of LDS, two workgroups a CU; two blocks of a tile go
// together, the sums or weights of one between the products of the other (tile16::stream).  The weights' sum is that of the rounded
// weights, those that the product takes (taken from the unrounded ones the error grows from 2.2e-3 to 2.3e-3).
//
// Measured, us, the kernel with lists (ten solver steps allowed) -> this one: 4 x 16 heads, N = 4096, not causal, alpha = 1.5, D = 64: 2240 -> 760,
// D = 128: 3530 -> 1270; 8 heads, N = 8192, alpha = 1.333: 2860 -> 1020, 3250 -> 1200; 4 x 16, N = 4096, alpha = 2: 2280 -> 1760, 3630 -> 2770 (there
// the sums are piecewise linear and a step halves the support at best: five to eight walks).  Against 64 bits: bf16 2.3e-3 as before, f16 4.5e-4
// -> 2.9e-4 at N = 6000.
#pragma once
#include "attn_tile16.h"

namespace adsp {
namespace fwd16 {
using namespace tile16;

// A walk's Newton step of x times the mean of u leaves about (c0 - 1) / 2 (n sum u^2 / (sum u)^2 - 1) x^2 of it (n members, alpha = 1.5): half of
// that square for flat scores, more where few keys have most of the weight.  The last walk takes steps of up to this: an error of the weights
// below their rounding is left then; the thresholds that a backward reads are taken a step further by the output walk's sums.  bf16,
// alpha = 1.5: with 0.06 a row whose last step was just small enough had an error of 4.2e-3 where rounding alone gives the worst of 256 row
// blocks 3.35e-3 (8 heads, N = 4096, D = 128, q of spread 0.03 to 2); 0.04 has 3.35e-3, 0.03 the same.  us, 0.06 / 0.04 / 0.03, 4 x 16 heads, N = 4096,
// q of spread 1/8: D = 64 699 / 712 / 732, D = 128 1190 / 1213 / 1221; spread 1/2, D = 64: 1081 / 1125 / 1144.
template <typename T, int AM> constexpr float kNear = AM == ATT_15 && elem_traits<T>::kIsBf16 ? 0.04f : 0.02f;
constexpr int kSample = 256;  // keys of the sample that a row's first threshold comes from

template <typename T, int D, int AM, bool kTaus>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void attn_fwd16_kernel(AttnParams p) {
  constexpr int kTR = D == 64 ? 128 : 64;  // two stages of K and V in 64 KB either way: two workgroups a CU
  using TL = Tile<T, D, kTR>;
  constexpr int kRow = TL::kRow, kRows = kMaskRows, kBlk = kTR / 32, G = TL::kG;
  constexpr int kAhead = D == 64 ? 2 : 1;  // (registers)
  constexpr int kSampleTiles = kSample / kTR, NS = kSample / 32;
  __shared__ __align__(1024) unsigned char smem[4 * TL::kBytes];  // two stages of a K and a V tile
  __shared__ uint32_t more_flag[4];
  extern __shared__ uint32_t mask_lds[];  // the tile mask of the row block, where one is asked for
  const LeftOver left(p.block_flags, p.queue);
  if (left.none()) return;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, lq = lane & 31, lh = lane >> 5;
  const int N = p.N, group = p.Hq / p.Hkv, n_blk = (N + kRows - 1) / kRows;
  int bkv, mi, hg;
  if (!xcd_block_map(p.varlen != nullptr, p.B * p.Hkv, n_blk, group, p.causal != 0, 2ll * N * kRow, bkv, mi, hg)) return;
  const BatchItem item = batch_item(p.varlen, p.varlen_bits, p.B, N, bkv / p.Hkv, p.Hkv, n_blk * group, p.causal == 0, 2);
  const int b = item.b, L = item.L, kvh = bkv % p.Hkv, h = kvh * group + hg, bh = b * p.Hq + h;
  bkv = b * p.Hkv + kvh;
  const int mblk = n_blk - 1 - mi, m0 = mblk * kRows;
  if (!left.takes((size_t)bh * p.n_mblk + mblk)) return;
  const size_t q_row0 = (size_t)bh * N;
  unsigned char* const out = reinterpret_cast<unsigned char*>(p.out) + q_row0 * kRow;
  int32_t* const bmask = p.bmask ? p.bmask + ((size_t)bh * p.n_mblk + mblk) * p.mask_words : nullptr;
  if (m0 >= L) {
    zero_rows(out + (size_t)m0 * kRow, (N - m0 < kRows ? N - m0 : kRows) * kRow, tid);
    if (bmask)
      for (int i = tid; i < p.mask_words; i += 256) bmask[i] = 0;
    return;
  }
  const int wave_row0 = m0 + 32 * wave, qi = wave_row0 + lq;
  const bool live = qi < L;
  const float qs = p.qscale, inv_qs = 1.f / p.qscale, c0 = p.c0;
  uint32_t qf[D / 4];
  load_frags<D>(reinterpret_cast<const unsigned char*>(p.q) + (q_row0 + (live ? qi : L - 1)) * kRow, true, lh, qf);
  const int lim = p.causal ? (qi < L - 1 ? qi : L - 1) : L - 1;                     // last key of the lane's row
  const int lim_all = p.causal ? (wave_row0 < L - 1 ? wave_row0 : L - 1) : L - 1;  // the smallest of the wave
  const int key_hi = p.causal ? (m0 + kRows < L ? m0 + kRows : L) : L;
  const int nt = (key_hi + kTR - 1) / kTR;
  const int whole = (p.causal ? m0 : L) / 32;  // blocks of 32 keys that every row of the workgroup sees
  const unsigned char* kg = reinterpret_cast<const unsigned char*>(p.k) + (size_t)bkv * N * kRow;
  const unsigned char* vg = reinterpret_cast<const unsigned char*>(p.v) + (size_t)bkv * N * kRow;
  TL tl((uint32_t)(uintptr_t)smem, wave, lane);

  auto total = [](float x) { return x + __shfl_xor(x, 32, 64); };  // over the two lanes of a row
  auto top = [](float x) { return fmaxf(x, __shfl_xor(x, 32, 64)); };
  auto hide = [&](int k0, f32x16& s) {
    const int jb = k0 + 4 * lh;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = jb + 8 * (i >> 2) + (i & 3) <= lim ? s[i] : -INFINITY;
  };

  // ---- a first threshold from a sample of the keys, or the threshold itself where the sample is all of them ----
  const int n_key_blk = (key_hi + 31) / 32;
  const bool all_sampled = n_key_blk * 32 <= kSample;
  float t;  // in z units
  {
    auto block_of = [&](int x) { return all_sampled ? x : (int)((long long)x * whole / (kSample / 32)); };  // block x of the sample
#pragma unroll
    for (int i = 0; i < kSampleTiles; ++i)
      tl.issue_blocks(kg, [&](int r) {
        const int row = block_of(i * (kTR / 32) + r / 32) * 32 + r % 32;
        return row < L ? row : L - 1;
      }, smem + i * TL::kBytes, wave, lane);
    f32x16 s[NS];
#pragma unroll
    for (int x = 0; x < NS; ++x)
#pragma unroll
      for (int i = 0; i < 16; ++i) s[x][i] = 0.f;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    stream<NS * G, kAhead>([&](int g, u32x4(&a)[4]) { tl.rows(g / G / kBlk, g / G % kBlk, g % G, a); },
                      [&](int g, int k, const u32x4& a) { s[g / G] = mfma_16bit<T>(a, piece<D>(qf, 4 * (g % G) + k), s[g / G]); });
    float mx = -INFINITY;
    if (all_sampled) {
#pragma unroll
      for (int x = 0; x < NS; ++x) hide(x * 32, s[x]);
    }
#pragma unroll
    for (int x = 0; x < NS; ++x)
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[x][i]);
    mx = top(mx);
    // From above its root alpha = 2's sum, of few keys, throws a step far below: its sample aims at three times the sum.
    const float ratio = all_sampled ? 1.f : (float)(lim + 1) * (AM == ATT_2 ? 1.f / (3 * kSample) : 1.f / kSample);
    const float t_min = fmaf(mx, qs, -1.f);
    t = t_min;
    for (int it = 0; it < 16; ++it) {
      float s0 = 0.f, s1 = 0.f;
#pragma unroll
      for (int x = 0; x < NS; ++x)
#pragma unroll
        for (int i = 0; i < 16; ++i) add_powers<AM>(__builtin_amdgcn_fmed3f(fmaf(s[x][i], qs, -t), 0.f, 1.f), c0, s0, s1);
      const float step = f32path::norm_step<AM>(total(s0) * ratio, total(s1) * ratio, c0);
      t = fmaxf(t + step, t_min);
      if (__builtin_amdgcn_ballot_w64(fabsf(step) > (all_sampled ? 2e-4f : 2e-2f)) == 0ull) break;
    }
  }

  // ---- walks over the tiles first, first + step, ... below n ----
  // pair(block) for two of the wave's blocks of a tile that all of its rows see in full, else one(block, its first key)
  auto walk = [&](int first, int step, int n, bool with_v, auto&& one, auto&& pair) {
    __syncthreads();
    int st = 0;
    auto issue = [&](int s, int x) {
      tl.issue(kg, x * kTR, L, smem + s * 2 * TL::kBytes, wave, lane);
      if (with_v) tl.issue(vg, x * kTR, L, smem + s * 2 * TL::kBytes + TL::kBytes, wave, lane);
    };
    if (first < n) issue(0, first);
    for (int cur = first; cur < n; cur += step) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (cur + step < n) issue(st ^ 1, cur + step);
#pragma unroll
      for (int x = 0; x < kBlk; x += 2) {
        const int k0 = cur * kTR + x * 32;
        if (k0 + 63 <= lim_all) {
          asm volatile("; two blocks" ::: "memory");
          pair(x, k0);
          asm volatile("; end of two blocks" ::: "memory");
        } else {
#pragma unroll
          for (int y = 0; y < 2; ++y) {
            const int k1 = k0 + 32 * y;
            if (k1 >= L || (p.causal && k1 > wave_row0 + 31)) continue;
            asm volatile("; one block" ::: "memory");
            one(x + y, k1);
          }
        }
      }
      tl.move(st ? -2u * TL::kBytes : 2u * TL::kBytes);
      st ^= 1;
    }
    if (st) tl.move(-2u * TL::kBytes);
  };
  auto mul = [&](int g, int k, const u32x4& a, f32x16& s) { s = mfma_16bit<T>(a, piece<D>(qf, 4 * (g % G) + k), s); };

  // sums of u^c0 and u^(c0 - 1) above t, and the maximum less t, over the tiles; in raw units of u for alpha = 1.5 and 2
  float s0, s1, mx;
  auto sums_walk = [&](int first, int step, int n) {
    s0 = s1 = 0.f;
    mx = -INFINITY;
    const f32x16 from_t = splat(-t * inv_qs);
    f32x16 late = splat(-INFINITY);
    auto add = [&](float x) {
      mx = fmaxf(mx, x);
      if constexpr (AM == ATT_15) {
        const float u = __builtin_amdgcn_fmed3f(x, 0.f, INFINITY);
        s0 = fmaf(u, u, s0);
        s1 += u;
      } else if constexpr (AM == ATT_2) {
        s0 += __builtin_amdgcn_fmed3f(x, 0.f, INFINITY);
        s1 += x > 0.f ? 1.f : 0.f;
      } else {
        add_powers<AM>(__builtin_amdgcn_fmed3f(x, 0.f, INFINITY) * qs, c0, s0, s1);
      }
    };
    constexpr int kPer = 4 / G;  // values of a block per product of another
    walk(
        first, step, n, false,
        [&](int blk, int k0) {
          f32x16 s = from_t;
          stream<G, 2>([&](int g, u32x4(&a)[4]) { tl.rows(0, blk, g, a); }, [&](int g, int k, const u32x4& a) { mul(g, k, a, s); });
          if (k0 + 31 > lim_all) hide(k0, s);
#pragma unroll
          for (int i = 0; i < 16; ++i) add(s[i]);
        },
        [&](int blk, int) {
          f32x16 x0 = from_t, x1 = from_t;
          stream<2 * G, 2>([&](int g, u32x4(&a)[4]) { tl.rows(0, blk + g / G, g % G, a); },
                           [&](int g, int k, const u32x4& a) {
                             const int n4 = (g % G) * 4 + k;
                             if (g < G) mul(g, k, a, x0);
                             else mul(g, k, a, x1);
#pragma unroll
                             for (int i = 0; i < kPer; ++i) add(g < G ? late[n4 * kPer + i] : x0[n4 * kPer + i]);
                           });
          late = x1;
        });
#pragma unroll
    for (int i = 0; i < 16; ++i) add(late[i]);
    s0 = total(s0);
    s1 = total(s1);
    mx = top(mx);
    if constexpr (AM == ATT_15) {
      s0 *= qs * qs;
      s1 *= qs;
    } else if constexpr (AM == ATT_2) {
      s0 *= qs;
    }
  };
  // whether Newton's step stays in fp32 (it multiplies s0 by up to itself): not with a score far above the threshold, which an
  // unsampled key may have; the maximum less 1 is the next threshold then
  auto in_range = [&]() -> bool { return s0 > 0.f && s0 < 1e18f && s1 > 0.f && s1 < 1e18f; };
  if (!all_sampled) {
    // a step on every second tile, where that is much more than the sample
    const int half = whole * 32 / kTR / 2;
    if (half * kTR >= 2 * kSample) {
      sums_walk(1, 2, half * 2);
      const float ratio = (float)(lim + 1) / (float)(half * kTR) * (AM == ATT_2 ? 0.9f : 1.f);
      if (in_range()) t += fmaxf(mx * qs - 1.f, f32path::norm_step<AM>(s0 * ratio, s1 * ratio, c0));
      else t += fmaxf(mx * qs - 1.f, 0.f);
    }
    for (int it = 0; it < 32; ++it) {
      sums_walk(0, 1, nt);
      // never below the row maximum less 1
      float step = mx * qs - 1.f, near = 0.f;
      if (in_range()) {
        step = fmaxf(step, f32path::norm_step<AM>(s0, s1, c0));
        near = kNear<T, AM> * s0 * fast_rcp(s1);
      }
      if (live) t += step;
      const bool more = __builtin_amdgcn_ballot_w64(live && fabsf(step) > fmaxf(near, 2e-6f)) != 0ull;
      if (lane == 0) more_flag[wave] = more ? 1u : 0u;
      __syncthreads();
      const uint32_t any = more_flag[0] | more_flag[1] | more_flag[2] | more_flag[3];
      if (any == 0u) break;
    }
  }

  // ---- output ----
  if (bmask)
    for (int i = tid; i < p.mask_words; i += 256) mask_lds[i] = 0u;
  f32x16 o[TL::kDB];
#pragma unroll
  for (int db = 0; db < TL::kDB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
  f32x4_t zacc = {0.f, 0.f, 0.f, 0.f};  // the sum of the rounded weights, those that the product takes
  f32x16 zero;
#pragma unroll
  for (int i = 0; i < 16; ++i) zero[i] = 0.f;
  float q0 = 0.f, q1 = 0.f;  // the sums at t, for the threshold that is kept
  auto prob = [&](float x) -> float {
    // (within 1 but for the last step's remainder)
    const float u = __builtin_amdgcn_fmed3f(fmaf(x, qs, -t), 0.f, 1.f);
    float pr, e1;
    if constexpr (AM == ATT_15) {
      e1 = u;
      pr = u * u;
    } else if constexpr (AM == ATT_2) {
      pr = u;
      e1 = u > 0.f ? 1.f : 0.f;
    } else {
      e1 = fast_exp2(fast_log2(u) * (c0 - 1.f));  // (0 at 0)
      pr = e1 * u;
    }
    if constexpr (kTaus) {
      q0 += pr;
      q1 += e1;
      asm volatile("" : "+v"(q0), "+v"(q1));  // (else the compiler gathers the terms of a block, in 36 registers)
    }
    return pr;
  };
  auto operand = [&](const f32x16& s, uint32_t (&w)[8], int i) {
    const float x = prob(s[2 * i]);
    w[i] = pack2<T>(x, prob(s[2 * i + 1]));
  };
  auto add_weights = [&](const uint32_t (&w)[8], int i) { zacc = lane_sum4<T>(u32x2_t{w[2 * i], w[2 * i + 1]}, zacc); };
  auto mul_v = [&](int g, int k, const u32x4& a, const uint32_t (&w)[8]) {
    const int n = 4 * (g % G) + k, s = n / TL::kDB, db = n % TL::kDB;
    o[db] = mfma_16bit<T>(a, u32x4{w[4 * s], w[4 * s + 1], w[4 * s + 2], w[4 * s + 3]}, o[db]);
  };
  // (from the weights themselves: one below 6e-8 of the row's sum does not show in it)
  auto any_of = [](const uint32_t (&w)[8]) -> uint32_t { return ((w[0] | w[1]) | (w[2] | w[3])) | ((w[4] | w[5]) | (w[6] | w[7])); };
  auto mark = [&](uint32_t weights, int k0) {
    if (bmask && __builtin_amdgcn_ballot_w64(weights != 0u) != 0ull && lane == 0) atomicOr(&mask_lds[k0 >> 11], 1u << ((k0 >> 6) & 31));
  };
  walk(
      0, 1, nt, true,
      [&](int blk, int k0) {
        f32x16 s = zero;
        stream<G, 2>([&](int g, u32x4(&a)[4]) { tl.rows(0, blk, g, a); }, [&](int g, int k, const u32x4& a) { mul(g, k, a, s); });
        if (k0 + 31 > lim_all) hide(k0, s);
        uint32_t w[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) operand(s, w, i);
#pragma unroll
        for (int i = 0; i < 4; ++i) add_weights(w, i);
        stream<G, 2>([&](int g, u32x4(&a)[4]) { tl.columns(1, blk, g, a); }, [&](int g, int k, const u32x4& a) { mul_v(g, k, a, w); });
        mark(any_of(w), k0);
      },
      [&](int blk, int k0) {
        f32x16 x0 = zero, x1 = zero;
        uint32_t w0[8], w1[8], any = 0u;
        constexpr int kPer = 2 / G;
        stream<4 * G, kAhead>(
            [&](int g, u32x4(&a)[4]) {
              if (g < 2 * G) tl.rows(0, blk + g / G, g % G, a);
              else tl.columns(1, blk + g / G - 2, g % G, a);
            },
            [&](int g, int k, const u32x4& a) {
              const int n4 = (g % G) * 4 + k;
              if (g < G) {
                mul(g, k, a, x0);
              } else if (g < 2 * G) {
                mul(g, k, a, x1);
#pragma unroll
                for (int i = 0; i < kPer; ++i) operand(x0, w0, n4 * kPer + i);
              } else if (g < 3 * G) {
                mul_v(g, k, a, w0);
#pragma unroll
                for (int i = 0; i < kPer; ++i) operand(x1, w1, n4 * kPer + i);
              } else {
                mul_v(g, k, a, w1);  // (nothing is left for the vector pipe)
                if (n4 < 4) add_weights(w0, n4);
                if (n4 >= 4 * G - 4) add_weights(w1, n4 - (4 * G - 4));
                if (n4 == 0) any = any_of(w0) | any_of(w1);
              }
            });
        mark(any, k0);
      });
  if constexpr (kTaus) {
    q0 = total(q0);
    q1 = total(q1);
    if (!all_sampled && q0 > 0.f && q1 > 0.f) t += f32path::norm_step<AM>(q0, q1, c0);
    if (live && lh == 0) p.taus[q_row0 + qi] = t;
  }
  const float zsum = total(zacc[0]);
  const float inv = live && zsum > 0.f ? 1.f / zsum : 0.f;
  __syncthreads();  // the tiles become the sums' scratch
  BwdTiles<T, D>::store_rows(o, inv, smem + wave * 32 * kRow, out, wave_row0, N, lane);
  if (bmask)
    for (int i = tid; i < p.mask_words; i += 256) bmask[i] = (int32_t)mask_lds[i];
}

}  // namespace fwd16
}  // namespace adsp
