// Backward of the sparse entmax attention on all pairs of a row, 16-bit types, head dims 64 and 128, for gfx950: dQ and dK/dV.
// They serve the row and key blocks that the kernels on the supports leave over (flat scores), and whole problems too short for those.
//
// What bounds them: the matrix pipe, by way of power (on random operands the clock falls to 1.8 - 1.9 GHz), and the vector pipe
// beside it: a product of 32 x 32 x 16 takes 34 cycles of a wave's matrix pipe, and one value's weight, sums and packing 6 to 10
// vector instructions of 4 cycles each.  A wave that does first one, then the other leaves both pipes idle half of the time, and with the
// operands in its registers a CU holds eight waves (D = 64) or four (D = 128), too few to fill the gaps for one another.
//
// Split: a workgroup is four waves of 32 rows (queries; keys in the dK/dV kernel) with their operands in registers, and walks tiles of
// 128 rows of the other side through two stages of LDS; where that leaves CUs idle, P = 2 or 4 waves share the rows, take a half
// or a quarter of each tile's blocks each and add up their sums in LDS.  Two blocks of a tile go together: while the products of one are
// in the matrix pipe, the wave forms the other's weights (tile16::stream).  The accumulators start at -tau and -delta, so that the
// threshold costs no instruction, and one swizzle of a tile serves row reads and transposing reads, so that a tile is loaded once.
// dQ takes two walks, because a row's weights need delta = (sum u dP) / (sum u) first: 10 products of 7.  dK/dV takes one.
// kSplit: dQ's fp32 weights as two 16-bit operands, for f16 behind a power of two per row, where a problem is short enough for that.
//
// Measured, us, the kernels before (128 rows a workgroup, products and weights in turn; 32 rows where kSplit) -> these, dQ and dK/dV: D = 64,
// 4 x 16 heads, N = 4096, causal: 372 -> 365, 471 -> 340; not causal, alpha = 1.333: 1160 -> 909, 1104 -> 705.  D = 128: the same, causal: 788 -> 800,
// 944 -> 780, not causal: 1540 -> 1410, 1760 -> 1380, alpha = 1.333: 1793 -> 1794, 1957 -> 1531; few workgroups: 4 of 6000: 381 -> 237,
// 553 -> 313, alpha = 1.333: 469 -> 304, 618 -> 387.  kSplit, forward included: one head, N = 3000, D = 64: 144 -> 133, N = 4096: 239 -> 225.
#pragma once
#include "attn_tile16.h"

namespace adsp {
namespace bwd16 {
using namespace tile16;

// p and u = p^(2 - alpha) of a score above the threshold, up to the factors prob_scale and u_scale: s in raw units
template <int AM> __device__ __forceinline__ void weights(float s, float qs, float c0, float& pr, float& u) {
  if constexpr (AM == ATT_15) {
    u = __builtin_amdgcn_fmed3f(s, 0.f, INFINITY);
    pr = u * u;
  } else if constexpr (AM == ATT_2) {
    pr = __builtin_amdgcn_fmed3f(s, 0.f, INFINITY);
    u = s > 0.f ? 1.f : 0.f;
  } else {
    const float x = __builtin_amdgcn_fmed3f(s, 0.f, INFINITY) * qs;
    u = fast_exp2(fast_log2(x) * (c0 - 1.f));  // (0 at 0)
    pr = u * x;
  }
}
template <int AM> __device__ __forceinline__ float prob_scale(float qs) { return AM == ATT_15 ? qs * qs : (AM == ATT_2 ? qs : 1.f); }
template <int AM> __device__ __forceinline__ float u_scale(float qs) { return AM == ATT_15 ? qs : 1.f; }
// Whether u (dP - delta) takes u_scale in front of a product instead of behind it: raw u goes up to 1 / qs (16 at D = 64, 22.6 at
// D = 128), and f16 ends at 65504, which gradients of a few hundred reached then.  (bf16 has fp32's range.)
template <typename T, int AM> constexpr bool kScaleFirst = AM == ATT_15 && !elem_traits<T>::kIsBf16;

// ---------------------------------------------------------------------------------------------------------
// dQ
// ---------------------------------------------------------------------------------------------------------
template <typename T, int D, int AM, int P, bool kSplit>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D == 64 ? 2 : 1, D == 64 ? 2 : 1))) void attn_bwd16_dq_kernel(AttnBwdParams p) {
  using TL = Tile<T, D>;
  constexpr int kRow = TL::kRow, kTR = TL::kTR, kRG = 4 / P, kRows = 32 * kRG, kBlk = kTR / 32 / P, G = TL::kG;
  constexpr bool kScaled = kSplit && !elem_traits<T>::kIsBf16;
  __shared__ __align__(1024) unsigned char smem[4 * TL::kBytes];  // two stages of a K and a V tile
  __shared__ float red[P > 1 ? 4 : 1][4][32];
  const LeftOver left(p.block_flags, p.queue);
  if (left.none()) return;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, lq = lane & 31, lh = lane >> 5;
  const int rg = wave % kRG, part = wave / kRG;
  const int N = p.N, group = p.Hq / p.Hkv, n_blk = (N + kRows - 1) / kRows;
  int bkv, mi, hg;
  if (!xcd_block_map(p.varlen != nullptr, p.B * p.Hkv, n_blk, group, p.causal != 0, 2ll * N * kRow, bkv, mi, hg)) return;
  const BatchItem item = batch_item(p.varlen, p.varlen_bits, p.B, N, bkv / p.Hkv, p.Hkv, n_blk * group, p.causal == 0, D == 64 ? 2 : 1);
  const int b = item.b, L = item.L, kvh = bkv % p.Hkv, h = kvh * group + hg, bh = b * p.Hq + h;
  bkv = b * p.Hkv + kvh;
  const int m0 = (n_blk - 1 - mi) * kRows, mblk = m0 / kMaskRows;
  if (!left.takes((size_t)bh * p.n_mblk + mblk)) return;
  const size_t q_row0 = (size_t)bh * N;
  unsigned char* const dq = reinterpret_cast<unsigned char*>(p.dq) + q_row0 * kRow;
  if (m0 >= L) {
    zero_rows(dq + (size_t)m0 * kRow, (N - m0 < kRows ? N - m0 : kRows) * kRow, tid);
    return;
  }
  const int wave_row0 = m0 + 32 * rg, qi = wave_row0 + lq;
  const bool live = qi < L;
  const float qs = p.qscale;
  uint32_t qf[D / 4], dof[D / 4];
  {
    const size_t at = (q_row0 + (live ? qi : L - 1)) * kRow;
    load_frags<D>(reinterpret_cast<const unsigned char*>(p.q) + at, live, lh, qf);
    load_frags<D>(reinterpret_cast<const unsigned char*>(p.dout) + at, live, lh, dof);
  }
  const f32x16 from_tau = splat(live ? -p.taus[q_row0 + qi] / qs : -INFINITY);
  const int lim = p.causal ? (qi < L - 1 ? qi : L - 1) : L - 1;                     // last key of the lane's row
  const int lim_all = p.causal ? (wave_row0 < L - 1 ? wave_row0 : L - 1) : L - 1;  // the smallest of the wave
  const int key_hi = p.causal ? (m0 + kRows < L ? m0 + kRows : L) : L;
  const int nt = (key_hi + kTR - 1) / kTR;
  const int32_t* mrow = p.bmask ? p.bmask + ((size_t)bh * p.n_mblk + mblk) * p.mask_words : nullptr;
  const unsigned char* kg = reinterpret_cast<const unsigned char*>(p.k) + (size_t)bkv * N * kRow;
  const unsigned char* vg = reinterpret_cast<const unsigned char*>(p.v) + (size_t)bkv * N * kRow;
  TL tl((uint32_t)(uintptr_t)smem + part * kBlk * 32 * kRow, wave, lane);

  auto next_tile = [&](int cur) -> int {
    int t = cur + 1;
    if (mrow)
      while (t < nt && !(((uint32_t)mrow[t >> 4] >> (2 * (t & 15))) & 3u)) ++t;
    return t < nt ? t : -1;
  };
  auto issue = [&](int st, int t) {
    tl.issue(kg, t * kTR, L, smem + st * 2 * TL::kBytes, wave, lane);
    tl.issue(vg, t * kTR, L, smem + st * 2 * TL::kBytes + TL::kBytes, wave, lane);
  };
  // pair(block) for two of the wave's blocks of a tile that all of its rows see in full, else one(block, its first key)
  auto walk = [&](auto&& one, auto&& pair) {
    __syncthreads();
    int cur = next_tile(-1), st = 0;
    if (cur >= 0) issue(0, cur);
    while (cur >= 0) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      const int nxt = next_tile(cur);
      if (nxt >= 0) issue(st ^ 1, nxt);
#pragma unroll
      for (int x = 0; x < kBlk; x += 2) {
        const int k0 = cur * kTR + (part * kBlk + x) * 32;
        if (kBlk > 1 && k0 + 63 <= lim_all) {
          asm volatile("; two blocks" ::: "memory");
          pair(x);
          asm volatile("; end of two blocks" ::: "memory");
        } else {
#pragma unroll
          for (int y = 0; y < (kBlk > 1 ? 2 : 1); ++y) {
            const int k1 = k0 + 32 * y;
            if (k1 >= L || (p.causal && k1 > wave_row0 + 31)) continue;
            asm volatile("; masked" ::: "memory");
            one(x + y, k1);
          }
        }
      }
      cur = nxt;
      tl.move(st ? -2u * TL::kBytes : 2u * TL::kBytes);
      st ^= 1;
    }
    if (st) tl.move(-2u * TL::kBytes);
  };
  auto hide = [&](int k0, f32x16& s, f32x16& d) {  // (a value that the row may not see can be anything)
    const int jb = k0 + 4 * lh;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const bool see = jb + 8 * (i >> 2) + (i & 3) <= lim;
      s[i] = see ? s[i] : -INFINITY;
      d[i] = see ? d[i] : 0.f;
    }
  };
  // operands of the scores and dP: group g of K's rows of block 0, V's, K's of block 1, ...
  auto load_rows = [&](int blk, int g, u32x4 (&a)[4]) { tl.rows(g / G & 1, blk + (g / G >> 1), g % G, a); };
  auto mul_rows = [&](int g, int k, const u32x4& a, f32x16& s, f32x16& d) {
    if (g / G & 1) d = mfma_16bit<T>(a, piece<D>(dof, 4 * (g % G) + k), d);
    else s = mfma_16bit<T>(a, piece<D>(qf, 4 * (g % G) + k), s);
  };

  // ---- sums of p, u and u dP ----
  float zsum = 0.f, usum = 0.f, udp = 0.f, dmax = 0.f;
  const f32x16 zero = splat(0.f);
  auto sums = [&](const f32x16& s, const f32x16& dp, int i) {
    float pr, u;
    weights<AM>(s[i], qs, p.c0, pr, u);
    if constexpr (AM == ATT_15) zsum = fmaf(u, u, zsum);
    else zsum += pr;
    usum += u;
    udp = fmaf(u, dp[i], udp);
    if constexpr (kScaled) dmax = fmaxf(dmax, u > 0.f ? fabsf(dp[i]) : 0.f);
  };
  constexpr int kPer = 16 / (8 * G);  // values of a block per product of another
  f32x16 late_s = splat(-INFINITY), late_d = zero;  // a pair's second block is added up beside the products of the next pair
  walk(
      [&](int blk, int k0) {
        f32x16 s = from_tau, d = zero;
        stream<2 * G, 2>([&](int g, u32x4(&a)[4]) { load_rows(blk, g, a); }, [&](int g, int k, const u32x4& a) { mul_rows(g, k, a, s, d); });
        hide(k0, s, d);
#pragma unroll
        for (int i = 0; i < 16; ++i) sums(s, d, i);
      },
      [&](int blk) {
        f32x16 s0 = from_tau, d0 = zero, s1 = from_tau, d1 = zero;
        stream<4 * G, 2>([&](int g, u32x4(&a)[4]) { load_rows(blk, g, a); },
                      [&](int g, int k, const u32x4& a) {
                        const int x = g * 4 + k;
                        if (g < 2 * G) mul_rows(g, k, a, s0, d0);
                        else mul_rows(g, k, a, s1, d1);
#pragma unroll
                        for (int i = 0; i < kPer; ++i) {
                          if (g < 2 * G) sums(late_s, late_d, x * kPer + i);
                          else sums(s0, d0, x * kPer + i - 16);
                        }
                      });
        late_s = s1;
        late_d = d1;
      });
#pragma unroll
  for (int i = 0; i < 16; ++i) sums(late_s, late_d, i);
  zsum += __shfl_xor(zsum, 32, 64);
  usum += __shfl_xor(usum, 32, 64);
  udp += __shfl_xor(udp, 32, 64);
  if constexpr (kScaled) dmax = fmaxf(dmax, __shfl_xor(dmax, 32, 64));
  if constexpr (P > 1) {
    if (lh == 0) {
      red[wave][0][lq] = zsum;
      red[wave][1][lq] = usum;
      red[wave][2][lq] = udp;
      if constexpr (kScaled) red[wave][3][lq] = dmax;
    }
    __syncthreads();
    zsum = usum = udp = 0.f;
#pragma unroll
    for (int w = 0; w < P; ++w) {
      zsum += red[w * kRG + rg][0][lq];
      usum += red[w * kRG + rg][1][lq];
      udp += red[w * kRG + rg][2][lq];
      if constexpr (kScaled) dmax = fmaxf(dmax, red[w * kRG + rg][3][lq]);
    }
  }
  const float delta = usum > 0.f ? udp / usum : 0.f;
  if (live && part == 0 && lh == 0) {
    p.delta[q_row0 + qi] = delta;
    p.zinv[q_row0 + qi] = zsum > 0.f ? 1.f / (zsum * prob_scale<AM>(qs)) : 0.f;
  }
  int up = 0;
  if constexpr (kScaled) {
    const int e = (int)(__builtin_bit_cast(uint32_t, dmax / u_scale<AM>(qs)) >> 23) - 126;
    up = 13 - e;
    up = up > 60 ? 60 : (up < -60 ? -60 : up);
  }

  // ---- dX = u (dP - delta), dQ^T += K^T dX^T ----
  f32x16 o[TL::kDB];
#pragma unroll
  for (int db = 0; db < TL::kDB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
  const f32x16 from_delta = splat(-delta);
  constexpr int kParts = kSplit ? 2 : 1;
  auto dx = [&](const f32x16& s, const f32x16& dp, uint32_t (&w)[kParts][8], int i) {
    float pr, u0, u1;
    weights<AM>(s[2 * i], qs, p.c0, pr, u0);
    weights<AM>(s[2 * i + 1], qs, p.c0, pr, u1);
    float x0 = u0 * dp[2 * i], x1 = u1 * dp[2 * i + 1];
    if constexpr (kScaled) {
      x0 = __builtin_amdgcn_ldexpf(x0, up);
      x1 = __builtin_amdgcn_ldexpf(x1, up);
    } else if constexpr (kScaleFirst<T, AM>) {
      x0 *= qs;
      x1 *= qs;
    }
    w[0][i] = pack2<T>(x0, x1);
    if constexpr (kSplit) w[1][i] = pack2<T>(x0 - unpack_lo<T>(w[0][i]), x1 - unpack_hi<T>(w[0][i]));
  };
  auto mul_columns = [&](int g, int k, const u32x4& a, const uint32_t (&w)[kParts][8]) {
    const int n = 4 * g + k, s = n / TL::kDB, db = n % TL::kDB;
#pragma unroll
    for (int x = 0; x < kParts; ++x) o[db] = mfma_16bit<T>(a, u32x4{w[x][4 * s], w[x][4 * s + 1], w[x][4 * s + 2], w[x][4 * s + 3]}, o[db]);
  };
  walk(
      [&](int blk, int k0) {
        f32x16 s = from_tau, d = from_delta;
        stream<2 * G, 2>([&](int g, u32x4(&a)[4]) { load_rows(blk, g, a); }, [&](int g, int k, const u32x4& a) { mul_rows(g, k, a, s, d); });
        hide(k0, s, d);
        uint32_t w[kParts][8];
#pragma unroll
        for (int i = 0; i < 8; ++i) dx(s, d, w, i);
        stream<G, 2>([&](int g, u32x4(&a)[4]) { tl.columns(0, blk, g, a); }, [&](int g, int k, const u32x4& a) { mul_columns(g, k, a, w); });
      },
      [&](int blk) {
        f32x16 s0 = from_tau, d0 = from_delta, s1 = from_tau, d1 = from_delta;
        uint32_t w0[kParts][8], w1[kParts][8];
        stream<6 * G, 2>(
            [&](int g, u32x4(&a)[4]) {
              if (g < 4 * G) load_rows(blk, g, a);
              else tl.columns(0, blk + (g - 4 * G) / G, g % G, a);
            },
            [&](int g, int k, const u32x4& a) {
              const int x = g * 4 + k;
              if (g < 2 * G) {
                mul_rows(g, k, a, s0, d0);
              } else if (g < 4 * G) {
                mul_rows(g, k, a, s1, d1);
                if (x % G == 0) dx(s0, d0, w0, x / G - 8);
              } else if (g < 5 * G) {
                mul_columns(g - 4 * G, k, a, w0);
#pragma unroll
                for (int i = 0; i < 2 / G; ++i) dx(s1, d1, w1, (x - 16 * G) * (2 / G) + i);
              } else {
                mul_columns(g - 5 * G, k, a, w1);
              }
            });
      });
  __syncthreads();  // the tiles become the sums' scratch
  float scale = p.sm_scale;
  if constexpr (kScaled || !kScaleFirst<T, AM>) scale *= u_scale<AM>(qs);
  if constexpr (kScaled) scale = __builtin_amdgcn_ldexpf(scale, -up);
  if constexpr (P == 1) BwdTiles<T, D>::store_rows(o, scale, smem + wave * 32 * kRow, dq, wave_row0, N, lane);
  else store_parts<T, D, P>(o, scale, smem, dq, m0, N, wave, lane);
}

// ---------------------------------------------------------------------------------------------------------
// dK, dV
// ---------------------------------------------------------------------------------------------------------
template <typename T, int D, int AM, int P>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D == 64 ? 2 : 1, D == 64 ? 2 : 1))) void attn_bwd16_dkdv_kernel(AttnBwdParams p) {
  using TL = Tile<T, D>;
  constexpr int kRow = TL::kRow, kTR = TL::kTR, kRG = 4 / P, kRows = 32 * kRG, kBlk = kTR / 32 / P, G = TL::kG;
  __shared__ __align__(1024) unsigned char smem[4 * TL::kBytes];  // two stages of a Q and a dO tile
  __shared__ __align__(16) float scal[2][3][kTR];  // of a tile's queries: -tau, -delta, 1 / sum p, in the units of the products
  const LeftOver left(p.kv_flags, p.queue2);
  if (left.none()) return;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, lq = lane & 31, lh = lane >> 5;
  const int rg = wave % kRG, part = wave / kRG;
  const int N = p.N, group = p.Hq / p.Hkv, n_blk = (N + kRows - 1) / kRows;
  int bkv, nblk, member_unused;
  if (!xcd_block_map(p.varlen != nullptr, p.B * p.Hkv, n_blk, 1, p.causal != 0, 2ll * group * N * kRow, bkv, nblk, member_unused)) return;
  const BatchItem item = batch_item(p.varlen, p.varlen_bits, p.B, N, bkv / p.Hkv, p.Hkv, n_blk, p.causal == 0, D == 64 ? 2 : 1);
  const int b = item.b, L = item.L, kvh = bkv % p.Hkv, n0 = nblk * kRows;
  bkv = b * p.Hkv + kvh;
  if (!left.takes((size_t)bkv * p.n_mblk + n0 / kMaskRows)) return;
  const size_t kv_row0 = (size_t)bkv * N;
  unsigned char* const dk = reinterpret_cast<unsigned char*>(p.dk) + kv_row0 * kRow;
  unsigned char* const dv = reinterpret_cast<unsigned char*>(p.dv) + kv_row0 * kRow;
  if (n0 >= L) {
    const int bytes = (N - n0 < kRows ? N - n0 : kRows) * kRow;
    zero_rows(dk + (size_t)n0 * kRow, bytes, tid);
    zero_rows(dv + (size_t)n0 * kRow, bytes, tid);
    return;
  }
  const int wave_key0 = n0 + 32 * rg, kj = wave_key0 + lq;
  const bool live = kj < L;
  const float qs = p.qscale;
  uint32_t kf[D / 4], vf[D / 4];
  {
    const size_t at = (kv_row0 + (live ? kj : L - 1)) * kRow;
    load_frags<D>(reinterpret_cast<const unsigned char*>(p.k) + at, live, lh, kf);
    load_frags<D>(reinterpret_cast<const unsigned char*>(p.v) + at, live, lh, vf);
  }
  const int t_first = p.causal ? n0 / kTR : 0, nt = (L + kTR - 1) / kTR;
  const size_t q_head0 = (size_t)(b * p.Hq + kvh * group) * N;
  TL tl((uint32_t)(uintptr_t)smem + part * kBlk * 32 * kRow, wave, lane);

  // The walk is over (query tile, query head) pairs, tile major from the last tile down: the key blocks of a K/V head that run
  // side by side are then at the same tile at about the same time and share it in L2.  Step c = tile * group + head.
  auto next_step = [&](int cur) -> int {
    int c = cur - 1;
    const int first = t_first * group;
    if (p.bmask)
      for (; c >= first; --c) {
        const int32_t* mcol = p.bmask + ((size_t)(b * p.Hq + kvh * group + c % group) * p.n_mblk + c / group) * p.mask_words;
        const uint32_t w = (uint32_t)mcol[n0 / 64 / 32] >> (n0 / 64 & 31);  // (a block of 128 keys starts on an even tile of 64)
        if (w & (kRows == 128 ? 3u : 1u)) break;
      }
    return c >= first ? c : -1;
  };
  constexpr int kScal = (3 * kTR + 255) / 256;
  float next_scal[kScal];
  auto issue = [&](int st, int step) {
    const int row0 = step / group * kTR;
    const size_t head = q_head0 + (size_t)(step % group) * N;
    tl.issue(reinterpret_cast<const unsigned char*>(p.q) + head * kRow, row0, L, smem + st * 2 * TL::kBytes, wave, lane);
    tl.issue(reinterpret_cast<const unsigned char*>(p.dout) + head * kRow, row0, L, smem + st * 2 * TL::kBytes + TL::kBytes, wave, lane);
#pragma unroll
    for (int x = 0; x < kScal; ++x) {
      const int id = x * 256 + tid, which = id / kTR;
      int row = row0 + id % kTR;
      row = row < L ? row : L - 1;
      if (which < 3) next_scal[x] = (which == 0 ? p.taus : (which == 1 ? p.delta : p.zinv))[head + row];
    }
  };
  auto put_scalars = [&](int st) {
#pragma unroll
    for (int x = 0; x < kScal; ++x) {
      const int id = x * 256 + tid, which = id / kTR;
      const float f = which == 0 ? -1.f / qs : (which == 1 ? -1.f : prob_scale<AM>(qs));
      if (which < 3) (&scal[st][0][0])[id] = next_scal[x] * f;
    }
  };
  f32x16 ov[TL::kDB], ok[TL::kDB];
#pragma unroll
  for (int db = 0; db < TL::kDB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) ov[db][i] = ok[db][i] = 0.f;
  auto start = [&](const float* sc, f32x16& s) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(sc + 8 * g + 4 * lh);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[4 * g + e] = x[e];
    }
  };
  // operands of the scores and dP: group g of q's rows of block 0, dO's, q's of block 1, ...
  auto load_rows = [&](int blk, int g, u32x4 (&a)[4]) { tl.rows(g / G & 1, blk + (g / G >> 1), g % G, a); };
  auto mul_rows = [&](int g, int k, const u32x4& a, f32x16& s, f32x16& d) {
    if (g / G & 1) d = mfma_16bit<T>(a, piece<D>(vf, 4 * (g % G) + k), d);
    else s = mfma_16bit<T>(a, piece<D>(kf, 4 * (g % G) + k), s);
  };
  // of the gradients: dO's columns of block 0, q's, dO's of block 1, ...
  auto load_columns = [&](int blk, int g, u32x4 (&a)[4]) { tl.columns(g / G & 1 ? 0 : 1, blk + (g / G >> 1), g % G, a); };
  auto mul_columns = [&](int g, int k, const u32x4& a, const uint32_t (&wp)[8], const uint32_t (&wx)[8]) {
    const int n = 4 * (g % G) + k, s = n / TL::kDB, db = n % TL::kDB;
    if (g / G & 1) ok[db] = mfma_16bit<T>(a, u32x4{wx[4 * s], wx[4 * s + 1], wx[4 * s + 2], wx[4 * s + 3]}, ok[db]);
    else ov[db] = mfma_16bit<T>(a, u32x4{wp[4 * s], wp[4 * s + 1], wp[4 * s + 2], wp[4 * s + 3]}, ov[db]);
  };
  auto operands = [&](const f32x16& s, const f32x16& d, const f32x16& z, uint32_t (&wp)[8], uint32_t (&wx)[8], int i) {
    float p0, u0, p1, u1;
    weights<AM>(s[2 * i], qs, p.c0, p0, u0);
    weights<AM>(s[2 * i + 1], qs, p.c0, p1, u1);
    wp[i] = pack2<T>(p0 * z[2 * i], p1 * z[2 * i + 1]);
    float x0 = u0 * d[2 * i], x1 = u1 * d[2 * i + 1];
    if constexpr (kScaleFirst<T, AM>) {
      x0 *= qs;
      x1 *= qs;
    }
    wx[i] = pack2<T>(x0, x1);
  };
  auto one = [&](int blk, const float* sc, int q0) {
    f32x16 s, d, z;
    start(sc, s);
    start(sc + kTR, d);
    start(sc + 2 * kTR, z);
    stream<2 * G, D == 64 ? 1 : 2>([&](int g, u32x4(&a)[4]) { load_rows(blk, g, a); }, [&](int g, int k, const u32x4& a) { mul_rows(g, k, a, s, d); });
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int qrow = q0 + 8 * (i >> 2) + 4 * lh + (i & 3);
      const bool see = live && qrow < L && (!p.causal || kj <= qrow);
      s[i] = see ? s[i] : -INFINITY;
      d[i] = see ? d[i] : 0.f;
    }
    uint32_t wp[8], wx[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) operands(s, d, z, wp, wx, i);
    stream<2 * G, D == 64 ? 1 : 2>([&](int g, u32x4(&a)[4]) { load_columns(blk, g, a); }, [&](int g, int k, const u32x4& a) { mul_columns(g, k, a, wp, wx); });
  };
  auto pair = [&](int blk, const float* sc) {
    f32x16 s0, d0, s1, d1, z;
    uint32_t wp0[8], wx0[8], wp1[8], wx1[8];
    start(sc, s0);
    start(sc + kTR, d0);
    stream<8 * G, D == 64 ? 1 : 2>(
        [&](int g, u32x4(&a)[4]) {
          if (g == G) start(sc + 2 * kTR, z);
          if (g == 2 * G) start(sc + 32, s1);
          if (g == 3 * G) start(sc + kTR + 32, d1);
          if (g < 4 * G) load_rows(blk, g, a);
          else load_columns(blk, g - 4 * G, a);
        },
        [&](int g, int k, const u32x4& a) {
          const int x = g * 4 + k;
          if (g < 2 * G) {
            mul_rows(g, k, a, s0, d0);
          } else if (g < 4 * G) {
            mul_rows(g, k, a, s1, d1);
            if (x % G == 0) operands(s0, d0, z, wp0, wx0, x / G - 8);
            if (x == 16 * G - 1) start(sc + 2 * kTR + 32, z);
          } else if (g < 6 * G) {
            mul_columns(g - 4 * G, k, a, wp0, wx0);
            if (x % G == 0) operands(s1, d1, z, wp1, wx1, x / G - 16);
          } else {
            mul_columns(g - 6 * G, k, a, wp1, wx1);
          }
        });
  };
  {
    int cur = next_step(nt * group), st = 0;
    if (cur >= 0) issue(0, cur);
    while (cur >= 0) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      put_scalars(st);
      __syncthreads();
      const int nxt = next_step(cur);
      if (nxt >= 0) issue(st ^ 1, nxt);
      const int row0 = cur / group * kTR + part * kBlk * 32;
      const float* const sc = &scal[st][0][part * kBlk * 32];
#pragma unroll
      for (int x = 0; x < kBlk; x += 2) {
        const int q0 = row0 + x * 32;
        if (kBlk > 1 && wave_key0 + 31 < L && q0 + 63 < L && (!p.causal || wave_key0 + 31 <= q0)) {
          asm volatile("; two blocks" ::: "memory");
          pair(x, sc + x * 32);
          asm volatile("; end of two blocks" ::: "memory");
        } else {
#pragma unroll
          for (int y = 0; y < (kBlk > 1 ? 2 : 1); ++y) {
            const int q1 = q0 + 32 * y;
            if (q1 >= L || (p.causal && q1 + 31 < wave_key0)) continue;
            asm volatile("; masked" ::: "memory");
            one(x + y, sc + (x + y) * 32, q1);
          }
        }
      }
      cur = nxt;
      tl.move(st ? -2u * TL::kBytes : 2u * TL::kBytes);
      st ^= 1;
    }
  }
  __syncthreads();
  const float scale = kScaleFirst<T, AM> ? p.sm_scale : p.sm_scale * u_scale<AM>(qs);
  if constexpr (P == 1) {
    unsigned char* const stage = smem + wave * 32 * kRow;
    BwdTiles<T, D>::store_rows(ov, 1.f, stage, dv, wave_key0, N, lane);
    __builtin_amdgcn_s_waitcnt(0xc07f);
    BwdTiles<T, D>::store_rows(ok, scale, stage, dk, wave_key0, N, lane);
  } else {
    store_parts<T, D, P>(ov, 1.f, smem, dv, n0, N, wave, lane);
    __syncthreads();
    store_parts<T, D, P>(ok, scale, smem, dk, n0, N, wave, lane);
  }
}

}  // namespace bwd16
}  // namespace adsp
