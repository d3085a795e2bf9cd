// Forward of the sparse entmax attention on all pairs of a row, 16-bit types, head dims 64 and 128, for gfx950, for the row blocks
// that the kernels on the supports leave over (flat scores).
//
// What bounds it: matrix and vector pipe together, at the 1.8 - 1.9 GHz that their power leaves (a block of 32 x 32 scores takes two to
// four products of 34 cycles a walk and three vector instructions a score).  So the number of walks over the keys is what counts.
//
// A row's threshold starts from a sample of 256 keys held in registers.  alpha = 1.5: from the sample's mean and spread, as if the scores were
// normal, unless the sample contradicts it, then from the sample's own solution; the walks' steps know the members' number and the density where they end (set_step), so that one leaves the
// cube of what there was, at the four instructions a score that the sums and the maximum took.  Where a row has hundreds of members, a quarter of the
// tiles corrects the start, the others give a threshold, and the quarter's sums there go together with the others', moved as far
// (move_sums): one and a quarter walks and the output's.  Fewer members: walks over all tiles until a step is small, mostly two; a wave whose rows are done
// no longer takes part.  The output walk checks what the steps left (kOff).  Other alphas: Newton's steps on the sample, one on every second tile, one or two on all tiles (a step squares what is left).
// The output walk's own sums take the threshold that a backward reads one step further.
//
// Split: four waves of 32 rows, tiles of K (and V in the output walk) through two stages of LDS, two workgroups a CU; two blocks of a tile go
// together, the sums or weights of one between the products of the other (tile16::stream).  The weights' sum is that of the rounded
// weights, those that the product takes (taken from the unrounded ones the error grows from 2.2e-3 to 2.3e-3).
//
// Measured, us, the kernel with lists (ten solver steps allowed) -> this one: 4 x 16 heads, N = 4096, not causal, alpha = 1.5, D = 64: 2240 -> 760,
// D = 128: 3530 -> 1270; 8 heads, N = 8192, alpha = 1.333: 2860 -> 1020, 3250 -> 1200; 4 x 16, N = 4096, alpha = 2: 2280 -> 1760, 3630 -> 2770 (there
// the sums are piecewise linear and a step halves the support at best: five to eight walks).  Against 64 bits: bf16 2.3e-3 as before, f16 4.5e-4
// -> 2.9e-4 at N = 6000.
// alpha = 1.5, Newton's steps (sample, half, two and more walks) -> this, 32 heads, N = 4096, not causal, scores (z) of spread 1/16, 1/8 and 1/4: D = 64 normal 379 -> 333, 490 ->
// 403, 624 -> 519, even 374 -> 287, 382 -> 292, 370 -> 303, rising along the keys 359 -> 270, 361 -> 277, 358 -> 372; D = 128, 1/16 and 1/4: normal 662 -> 520, 931 -> 793, even 604 -> 463,
// 599 -> 499.  Slower: a tenth of the keys in a cluster above the others, 1/4: 373 -> 423, log-normal 481 -> 532.  With a first threshold by the normal distribution wherever no key of
// the sample was above it: even, 1/8 and 1/4: 686 and 670, D = 128, 1/4: 1044.  Rows of one key far above thousands of others had errors of up to 3.3e-2 and have 4e-3.
#pragma once
#include "attn_tile16.h"

namespace adsp {
namespace fwd16 {
using namespace tile16;

// The last walk takes steps of up to this times (sum u^2 / sum u) -- alpha = 1.5: times the mean of u, see near_of --: an error of the weights below
// their rounding is left then; the thresholds that a backward reads are taken a step further by the output walk's sums.  A walk's Newton step of x times the mean of u leaves about (c0 - 1) / 2 (n sum u^2 / (sum u)^2 - 1)
// x^2 of it (n members), set_step a twentieth of x^3.  With Newton's steps, bf16, alpha = 1.5, and 0.06 a row whose last step was just
// small enough had an error of 4.2e-3 where rounding alone gives the worst of 256 row blocks 3.35e-3 (8 heads, N = 4096, D = 128, q of spread 0.03 to 2); 0.04 had
// 3.35e-3: some 1e-3 of the mean of u left.  set_step leaves as much behind 0.22 of the mean of u where there are 256 members (f16: a sixth of it behind 0.15); with fewer they are
// further apart, and a member that changes counts for more.  The parts' sums are moved by up to 2.5 times that where
// the sums are as a normal distribution's upper part has them and keys are left to become members, otherwise by 1.5 times (by 2.5 always: rows of two clusters of scores, or of one key far above the others,
// up to 4.7e-3 and 2e-2; by 2: 584 -> 645 us, D = 64).
template <typename T, int AM> constexpr float kNear = AM == ATT_15 ? (elem_traits<T>::kIsBf16 ? 0.22f : 0.15f) : 0.02f;
// What a density misjudges shows in the output walk's own sum of u^2, taken in fp32: where rows of a last step beyond kSure times (sum u^2 / sum u), or of sums that were
// moved, have it kOff and more from 1, Newton's step from there is taken and the output walk done again, twice at most.  Scores of few values, whose members come and go
// by hundreds (600 sets of 4 to 48 values, N = 1100 to 4096, a model of the kernel): the worst row's weights off by 4.0e-3 without this, bf16 1.4e-3 and f16 2.6e-4 with it, 1.5e-3 and 2.3e-4
// with Newton's steps and the smaller limits.  Scores without such steps seldom need it.  32 heads, N = 4096, not causal, us without and with: D = 64 normal scores of spread 1/16 355 and 360, 1/4 481 and 489,
// even 289 and 302, on 25 values 375 and 465; D = 128 normal 522 and 551, 764 and 767; N = 2048, D = 64, 1/16, where all row blocks run at once, 102 and 113.
template <typename T> constexpr float kSure = elem_traits<T>::kIsBf16 ? 0.04f : 0.02f;
template <typename T> constexpr float kOff = elem_traits<T>::kIsBf16 ? 1.5e-3f : 5e-4f;
// alpha = 1.5: steps from the sums of u^2 and u and the members' number.  With the same members the sum of u^2 is a parabola in the threshold; the
// members that change are few, near u = 0, and their density there follows from the three sums (members_density: exact for u distributed evenly
// and exponentially; for a normal distribution above a threshold 0.4 spreads over its mean and more within 2.5 %, at the mean 7 % too high, half a spread below it 18 %, a
// spread below it 44 %: there most keys are members and few change).  What a step of x times the mean of u leaves of it, root of
// mean square and the most of 256 rows of 575 members: x = 0.2: 2e-4 and 6e-4, 0.3: 5e-4 and 2e-3 (Newton's on the norm 9e-3 and 2e-2); of 62 members: 5e-4
// and 2e-3, 1.5e-3 and 4e-3.  Where the parabola has no root nearby Newton's step on the norm is taken.
__device__ __forceinline__ float members_density(float s0, float s1, float n) {
  const float shape = n * s0 * fast_rcp(s1 * s1);
  return n * n * fast_rcp(s1) * __builtin_amdgcn_fmed3f(fmaf(0.75f, shape, -0.5f), 0.f, 1.5f);
}
__device__ __forceinline__ float set_step(float s0, float s1, float n, float c0) {
  const float disc = fmaf(s1, s1, -n * (s0 - 1.f));
  if (!(disc > 0.25f * s1 * s1)) return f32path::norm_step<ATT_15>(s0, s1, c0);
  const float root = __builtin_amdgcn_sqrtf(disc), x = (s0 - 1.f) * fast_rcp(s1 + root);
  return x * (1.f - fminf(members_density(s0, s1, n) * x * x * fast_rcp(6.f * root), 0.4f));  // (far away the density is another)
}
// the sums `by` further up
__device__ __forceinline__ void move_sums(float by, float& s0, float& s1, float& n) {
  const float d = members_density(s0, s1, n);
  s0 = fmaf(by, fmaf(by, fmaf(by, d * (-1.f / 3.f), n), -2.f * s1), s0);
  s1 = fmaf(by, fmaf(by, 0.5f * d, -n), s1);
  n = fmaf(-by, d, n);
}
// Where the threshold of n keys of normally distributed scores lies (alpha = 1.5), in spreads above their mean: n s^2 ((1 + a^2) Q(a) - a phi(a)) = 1,
// within 0.16 from n s^2 = 0.2 to 20000, where the two pieces meet (0.03 from 2 on).
__device__ __forceinline__ float normal_threshold(float ns2) {
  return ns2 < 0.82f ? -__builtin_amdgcn_sqrtf(fmaxf(fast_rcp(ns2) - 1.f, 0.f)) : __builtin_amdgcn_sqrtf(fmaf(1.8f, fast_log2(ns2), 1.7f)) - 1.87f;
}
constexpr int kSample = 256;  // keys of the sample that a row's first threshold comes from

// A row block.  Returns whether it has to be gone through again, from the output walk on (kOff; `turn`: how many times it has been).
template <typename T, int D, int AM, bool kTaus> __device__ __forceinline__ bool row_block(const AttnParams& p, int turn) {
  constexpr int kTR = D == 64 ? 128 : 64;  // two stages of K and V in 64 KB either way: two workgroups a CU
  using TL = Tile<T, D, kTR>;
  constexpr int kRow = TL::kRow, kRows = kMaskRows, kBlk = kTR / 32, G = TL::kG;
  constexpr int kAhead = D == 64 ? 2 : 1;  // (registers)
  constexpr int kSampleTiles = kSample / kTR, NS = kSample / 32;
  constexpr bool kSet = AM == ATT_15;  // steps with the members' number (set_step)
  __shared__ __align__(1024) unsigned char smem[4 * TL::kBytes];  // two stages of a K and a V tile
  __shared__ uint32_t more_flag[4];
  __shared__ float slope_lds[kSet ? 256 : 1], t_lds[kSet ? 256 : 1];  // a lane's sum of u behind its last step, about, and its threshold, for another turn
  extern __shared__ uint32_t mask_lds[];  // the tile mask of the row block, where one is asked for
  const LeftOver left(p.block_flags, p.queue);
  if (left.none()) return false;
  int tid = threadIdx.x;
  if constexpr (kSet) asm volatile("" : "+v"(tid));  // (nothing is kept in registers from turn to turn: D = 128's walks would spill, 10 % of the time)
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, lq = lane & 31, lh = lane >> 5;
  const int N = p.N, group = p.Hq / p.Hkv, n_blk = (N + kRows - 1) / kRows;
  int bkv, mi, hg;
  if (!xcd_block_map(p.varlen != nullptr, p.B * p.Hkv, n_blk, group, p.causal != 0, 2ll * N * kRow, bkv, mi, hg)) return false;
  const BatchItem item = batch_item(p.varlen, p.varlen_bits, p.B, N, bkv / p.Hkv, p.Hkv, n_blk * group, p.causal == 0, 2);
  const int b = item.b, L = item.L, kvh = bkv % p.Hkv, h = kvh * group + hg, bh = b * p.Hq + h;
  bkv = b * p.Hkv + kvh;
  const int mblk = n_blk - 1 - mi, m0 = mblk * kRows;
  if (!left.takes((size_t)bh * p.n_mblk + mblk)) return false;
  const size_t q_row0 = (size_t)bh * N;
  unsigned char* const out = reinterpret_cast<unsigned char*>(p.out) + q_row0 * kRow;
  int32_t* const bmask = p.bmask ? p.bmask + ((size_t)bh * p.n_mblk + mblk) * p.mask_words : nullptr;
  if (m0 >= L) {
    zero_rows(out + (size_t)m0 * kRow, (N - m0 < kRows ? N - m0 : kRows) * kRow, tid);
    if (bmask)
      for (int i = tid; i < p.mask_words; i += 256) bmask[i] = 0;
    return false;
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
  float t = 0.f;  // in z units
  bool flat = false;  // hundreds of members, alpha = 1.5
  if (turn == 0) {
    // block x of the sample (alpha = 1.5: in the middle of its eighth of the keys, for scores that rise or fall along the sequence)
    auto block_of = [&](int x) { return all_sampled ? x : (int)((kSet ? (2ll * x + 1) * whole / 2 : (long long)x * whole) / (kSample / 32)); };
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
    float mx = -INFINITY, m1 = 0.f, m2 = 0.f;
    if (all_sampled) {
#pragma unroll
      for (int x = 0; x < NS; ++x) hide(x * 32, s[x]);
    }
#pragma unroll
    for (int x = 0; x < NS; ++x)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        mx = fmaxf(mx, s[x][i]);
        if constexpr (kSet) {
          m1 += s[x][i];
          m2 = fmaf(s[x][i], s[x][i], m2);
        }
      }
    mx = top(mx);
    // From above its root alpha = 2's sum, of few keys, throws a step far below: its sample aims at three times the sum.
    const float ratio = all_sampled ? 1.f : (float)(lim + 1) * (AM == ATT_2 ? 1.f / (3 * kSample) : 1.f / kSample);
    const float t_min = fmaf(mx, qs, -1.f);
    t = t_min;
    float spread = 0.f;
    bool keep = false, far_out = false;  // some ten members of the sample at most are to be expected
    if constexpr (kSet) {
      if (!all_sampled) {  // (as if the scores were normal: two steps less than from t_min)
        const float mean = total(m1) * (qs / kSample), var = fmaxf(fmaf(-mean, mean, total(m2) * (qs * qs / kSample)), 0.f);
        const float a = normal_threshold(var * (float)(lim + 1)), guess = fmaf(a, spread = __builtin_amdgcn_sqrtf(var), mean);
        far_out = a > 1.7f;
        keep = guess > t_min && guess < t_min + 1.f;  // (below the sample's maximum)
        t = keep ? guess : t_min;
      }
    }
    float many = 0.f;  // members that the sample makes out
    for (int it = 0; it < 16; ++it) {
      float s0 = 0.f, s1 = 0.f, step;
      if constexpr (kSet) {
        // (below the threshold the difference's sign shows; u of up to a sample's rounding above 1 is no harm)
        uint32_t below = 0u, signs = 0u;
#pragma unroll
        for (int x = 0; x < NS; ++x) {
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const float d = fmaf(s[x][i], qs, -t), u = fmaxf(d, 0.f);
            s0 = fmaf(u, u, s0);
            s1 += u;
            signs = __builtin_amdgcn_alignbit(signs, __builtin_bit_cast(uint32_t, d), 31);
          }
          if (x & 1) below += __builtin_popcount(signs);
        }
        s0 = total(s0) * ratio;
        s1 = total(s1) * ratio;
        const float n = total((float)(NS * 16 - (int)below)) * ratio;
        // (the set's steps come from either side of the threshold; Newton's, from below, end in any case)
        step = it < 6 ? set_step(s0, s1, n, c0) : f32path::norm_step<AM>(s0, s1, c0);
        many = n;
        // (the sample's own error is as large as the guess's: one that the sample does not contradict stays.  Far out a guess above the sample's
        // solution, or without a key of the sample above it, may lie where no key is -- scores with an upper end -- and costs walks until it is found: there the
        // sample's own solution is taken.)
        if (it == 0) keep = keep && s1 > 0.f && (far_out ? step >= 0.f && step <= spread : fabsf(step) <= s0 * fast_rcp(s1));
        step = keep ? 0.f : (s1 > 0.f ? step : t_min - t);
      } else {
#pragma unroll
        for (int x = 0; x < NS; ++x)
#pragma unroll
          for (int i = 0; i < 16; ++i) add_powers<AM>(__builtin_amdgcn_fmed3f(fmaf(s[x][i], qs, -t), 0.f, 1.f), c0, s0, s1);
        step = f32path::norm_step<AM>(total(s0) * ratio, total(s1) * ratio, c0);
      }
      t = fmaxf(t + step, t_min);
      if (__builtin_amdgcn_ballot_w64(fabsf(step) > (all_sampled ? 2e-4f : 2e-2f)) == 0ull) break;
    }
    // (f16's last step has to be smaller, and unless a third of the keys are members a quarter's is too far off for it, so that a walk over all follows: 4 x 16 heads, N = 2048, D = 64, not
    // causal, q of spread 1/8 (a quarter of the keys): 225 us with the parts, 188 without; of spread 1/32 (three quarters) 158 and 184; 16 heads, N = 8192, spread 1/32 (two fifths) 526 and 657)
    flat = many >= (elem_traits<T>::kIsBf16 ? 224.f : fmaxf(224.f, 0.3f * (float)(lim + 1)));
  }

  // ---- walks over the tiles next(-1), next of that, ... below n ----
  // pair(block) for two of the wave's blocks of a tile that all of its rows see in full, else one(block, its first key)
  bool idle = false;  // the wave's rows are done: it loads its share of the tiles for the others
  auto walk = [&](auto&& next, int n, bool with_v, auto&& one, auto&& pair) {
    const int first = next(-1);
    __syncthreads();
    int st = 0;
    auto issue = [&](int s, int x) {
      tl.issue(kg, x * kTR, L, smem + s * 2 * TL::kBytes, wave, lane);
      if (with_v) tl.issue(vg, x * kTR, L, smem + s * 2 * TL::kBytes + TL::kBytes, wave, lane);
    };
    if (first < n) issue(0, first);
    for (int cur = first, nxt; cur < n; cur = nxt) {
      nxt = next(cur);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (nxt < n) issue(st ^ 1, nxt);
      if (!idle)
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
  auto every = [](int cur) { return cur + 1; };
  auto mul = [&](int g, int k, const u32x4& a, f32x16& s) { s = mfma_16bit<T>(a, piece<D>(qf, 4 * (g % G) + k), s); };

  // sums of u^c0 and u^(c0 - 1) above t, their number (alpha = 1.5) and the maximum less t (alpha = 1.5: only `with_top`), over the tiles; in raw
  // units of u for alpha = 1.5 and 2.  A score's sign goes into a word with those of the block's others, and the words' ones are counted.
  float s0 = 0.f, s1 = 0.f, mx = -INFINITY, members = 0.f;
  auto sums_walk = [&](auto with_top, auto&& next, int n) {
    constexpr bool kTop = !kSet || decltype(with_top)::value;
    const float k0 = s0, k1 = s1, kn = members;
    s0 = s1 = 0.f;
    mx = -INFINITY;
    uint32_t signs = 0u;
    int count = 0;
    const f32x16 from_t = splat(-t * inv_qs);
    f32x16 late = splat(-INFINITY);
    auto add = [&](float x) {
      if constexpr (kTop) mx = fmaxf(mx, x);
      if constexpr (kSet) {
        const float u = __builtin_amdgcn_fmed3f(x, 0.f, INFINITY);
        s0 = fmaf(u, u, s0);
        s1 += u;
        signs = __builtin_amdgcn_alignbit(signs, __builtin_bit_cast(uint32_t, x), 31);
      } else if constexpr (AM == ATT_2) {
        s0 += __builtin_amdgcn_fmed3f(x, 0.f, INFINITY);
        s1 += x > 0.f ? 1.f : 0.f;
      } else {
        add_powers<AM>(__builtin_amdgcn_fmed3f(x, 0.f, INFINITY) * qs, c0, s0, s1);
      }
    };
    constexpr int kPer = 4 / G;  // values of a block per product of another
    walk(
        next, n, false,
        [&](int blk, int k0) {
          f32x16 s = from_t;
          stream<G, 2>([&](int g, u32x4(&a)[4]) { tl.rows(0, blk, g, a); }, [&](int g, int k, const u32x4& a) { mul(g, k, a, s); });
          if (k0 + 31 > lim_all) hide(k0, s);
#pragma unroll
          for (int i = 0; i < 16; ++i) add(s[i]);
          if constexpr (kSet) count += 16 - __builtin_popcount(signs & 0xffffu);
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
          if constexpr (kSet) count += 32 - __builtin_popcount(signs);
          late = x1;
        });
#pragma unroll
    for (int i = 0; i < 16; ++i) add(late[i]);
    s0 = total(s0);
    s1 = total(s1);
    if constexpr (kSet) members = total((float)(count + 16 - __builtin_popcount(signs & 0xffffu)));
    if constexpr (kTop) mx = top(mx);
    if constexpr (AM == ATT_15) {
      s0 *= qs * qs;
      s1 *= qs;
    } else if constexpr (AM == ATT_2) {
      s0 *= qs;
    }
    if (idle) {
      s0 = k0;
      s1 = k1;
      members = kn;
    }
  };
  // whether a step stays in fp32 (it multiplies s0 by up to itself): not with a score far above the threshold, which an
  // unsampled key may have; the maximum less 1 is the next threshold then
  auto in_range = [&]() -> bool { return s0 > 0.f && s0 < 1e18f && s1 > 0.f && s1 < 1e18f; };
  auto step_of = [&](float ratio, bool set) -> float {
    if constexpr (kSet) return set ? set_step(s0 * ratio, s1 * ratio, members * ratio, c0) : f32path::norm_step<AM>(s0 * ratio, s1 * ratio, c0);
    else return f32path::norm_step<AM>(s0 * ratio, s1 * ratio, c0);
  };
  auto near_of = [&]() -> float {  // (few members have no density to go by, and may have a bulk of keys just below their threshold: limits as wide as Newton's left errors of 1e-2 there)
    if constexpr (kSet) return kNear<T, AM> * s1 * fast_rcp(members) * __builtin_amdgcn_sqrtf(fminf(members * (1.f / 256.f), 1.f));
    else return kNear<T, AM> * s0 * fast_rcp(s1);
  };
  auto any_wave = [&](bool mine) -> bool {  // of a lane of the workgroup
    __syncthreads();
    const bool any = __builtin_amdgcn_ballot_w64(mine) != 0ull;
    if (lane == 0) more_flag[wave] = any ? 1u : 0u;
    __syncthreads();
    return (more_flag[0] | more_flag[1] | more_flag[2] | more_flag[3]) != 0u;
  };
  bool done = false;
  bool far = turn != 0;  // the last step was beyond kSure, or the sums were moved (alpha = 1.5)
  if (kSet && turn != 0) {
    t = t_lds[tid];
  } else if (!all_sampled) {
    if constexpr (kSet) {
      // A step on every fourth tile (the first part), one on the others, and one on all of them: the first part's sums at the threshold
      // that the second part gave, and the second's, which are known for the one before, moved there.  From 1792 keys on (at 1700 the quarter is too
      // few keys and the walk over all follows all the same: 68 us against 64); with fewer than some hundred members likewise (N = 4096, D = 64, q of spread 1/4: 800
      // against 727).
      const int n_first = whole * 32 / kTR / 4 * 4;  // tiles 1, 5, 9, .. below it are the first part
      if (n_first * kTR >= 7 * kSample && !any_wave(live && !flat)) {
        auto first_part = [](int cur) { return cur < 0 ? 1 : cur + 4; };
        auto second_part = [&](int cur) { return cur + 1 + ((cur & 3) == 0 && cur < n_first ? 1 : 0); };
        const int first_keys = n_first / 4 * kTR;
        const float keys = (float)(lim + 1);
        sums_walk(std::false_type{}, first_part, n_first);
        if (in_range()) t += step_of(keys / (float)first_keys, true);
        sums_walk(std::false_type{}, second_part, nt);
        bool ok = in_range();
        if (!any_wave(live && !ok)) {
          const float by = step_of(keys / (float)((lim + 1) - first_keys), true);
          const float shape = members * s0 * fast_rcp(s1 * s1);
          ok = fabsf(by) <= (shape > 1.35f && shape < 2.f && members < 0.9f * (keys - (float)first_keys) ? 2.5f : 1.5f) * near_of();
          float r0 = s0, r1 = s1, rn = members;
          move_sums(by, r0, r1, rn);
          if (live) t += by;
          sums_walk(std::false_type{}, first_part, n_first);
          s0 += r0;
          s1 += r1;
          members += rn;
          ok = ok && in_range();
          if (ok) {
            const float step = step_of(1.f, true);
            ok = fabsf(step) <= near_of();
            if (live) t += step;
            slope_lds[tid] = s1 - members * step;
          }
          done = !any_wave(live && !ok);
          far = true;
        }
      }
    } else {
      // a step on every second tile, where that is much more than the sample
      const int half = whole * 32 / kTR / 2;
      if (half * kTR >= 2 * kSample) {
        sums_walk(std::true_type{}, [](int cur) { return cur + 2; }, half * 2);  // (1, 3, ..)
        const float ratio = (float)(lim + 1) / (float)(half * kTR) * (AM == ATT_2 ? 0.9f : 1.f);
        if (in_range()) t += fmaxf(mx * qs - 1.f, step_of(ratio, false));
        else t += fmaxf(mx * qs - 1.f, 0.f);
      }
    }
    // The first walk over all keys takes the maximum as well (an instruction a score): the threshold is at least that less 1, which is what brings rows of
    // a few keys far above the sample near it, and where a row goes that a step has thrown above all of its keys.
    float low = 0.f;  // that bound, less t
    for (int it = 0; it < 32 && !done; ++it) {
      if constexpr (kSet) {
        if (it == 0) sums_walk(std::true_type{}, every, nt);
        else sums_walk(std::false_type{}, every, nt);
      } else {
        sums_walk(std::true_type{}, every, nt);
      }
      if (!idle) {
        if (!kSet || it == 0) low = mx * qs - 1.f;
        float step = low, near = 0.f;
        if (in_range()) {
          step = fmaxf(step, step_of(1.f, it < 6));
          near = near_of();
          far = kSet && fabsf(step) > kSure<T> * s0 * fast_rcp(s1);
          if constexpr (kSet) slope_lds[tid] = s1 - members * step;
        }
        if (live) t += step;
        low -= step;
        idle = __builtin_amdgcn_ballot_w64(live && fabsf(step) > fmaxf(near, 2e-6f)) == 0ull;
      }
      if (!any_wave(!idle)) break;
    }
    idle = false;
  }

  f32x16 o[TL::kDB];
  f32x4_t zacc;  // the sum of the rounded weights, those that the product takes
  f32x16 zero;
#pragma unroll
  for (int i = 0; i < 16; ++i) zero[i] = 0.f;
  // The sums at t, in fp32, for the threshold that is kept, and alpha = 1.5 for whether t was right (kOff).  (From the rounded weights' sum it would be off by up to 2e-3 of the
  // mean of u in bf16: roundings cancel neither over a few members nor over equal ones.)
  float q0, q1;
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
    if constexpr (kTaus || kSet) {
      q0 += pr;
      if constexpr (kTaus) {
        q1 += e1;
        asm volatile("" : "+v"(q0), "+v"(q1));  // (else the compiler gathers the terms of a block, in 36 registers)
      } else {
        asm volatile("" : "+v"(q0));
      }
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
  // ---- output ----
  if (!live) t = INFINITY;  // rows behind the sequence's end are copies of its last, with thresholds that no walk has moved: no weights and no marks of theirs
  if (bmask)
    for (int i = tid; i < p.mask_words; i += 256) mask_lds[i] = 0u;
#pragma unroll
  for (int db = 0; db < TL::kDB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
  zacc = f32x4_t{0.f, 0.f, 0.f, 0.f};
  q0 = q1 = 0.f;
  walk(
      every, nt, true,
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
  if constexpr (kSet) {
    const float off = total(q0) - 1.f;
    const bool wrong = live && far && fabsf(off) > kOff<T>;
    if (turn < 2 && any_wave(wrong)) {
      t_lds[tid] = wrong ? fmaf(0.5f * off, fast_rcp(slope_lds[tid]), t) : t;
      return true;
    }
  }
  const float zsum = total(zacc[0]);
  if constexpr (kTaus) {
    q0 = total(q0);
    q1 = total(q1);
    if (!all_sampled && q0 > 0.f && q1 > 0.f) t += f32path::norm_step<AM>(q0, q1, c0);
    if (live && lh == 0) p.taus[q_row0 + qi] = t;
  }
  const float inv = live && zsum > 0.f ? 1.f / zsum : 0.f;
  __syncthreads();  // the tiles become the sums' scratch
  BwdTiles<T, D>::store_rows(o, inv, smem + wave * 32 * kRow, out, wave_row0, N, lane);
  if (bmask)
    for (int i = tid; i < p.mask_words; i += 256) bmask[i] = (int32_t)mask_lds[i];
  return false;
}

template <typename T, int D, int AM, bool kTaus>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void attn_fwd16_kernel(AttnParams p) {
  for (int turn = 0; row_block<T, D, AM, kTaus>(p, turn); ++turn) {
  }
}

}  // namespace fwd16
}  // namespace adsp
