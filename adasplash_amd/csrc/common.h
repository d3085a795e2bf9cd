// Shared device helpers for the gfx950 kernels: element types, wave64 reductions, conversions.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace adsp {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));  // a 16-byte global/LDS access

struct bf16_t { uint16_t bits; };  // storage-only tags; arithmetic is always fp32
struct f16_t { uint16_t bits; };

template <typename T> struct elem_traits;
template <> struct elem_traits<float> { static constexpr int kBytes = 4; static constexpr int kVec = 4; static constexpr bool kIsBf16 = false; };
template <> struct elem_traits<bf16_t> { static constexpr int kBytes = 2; static constexpr int kVec = 8; static constexpr bool kIsBf16 = true; };
template <> struct elem_traits<f16_t> { static constexpr int kBytes = 2; static constexpr int kVec = 8; static constexpr bool kIsBf16 = false; };

__device__ __forceinline__ float bf16_bits_to_float(uint32_t b) { return __builtin_bit_cast(float, b << 16); }
__device__ __forceinline__ uint32_t float_to_bf16_bits(float f) {
  return (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)f);  // v_cvt_pk_bf16_f32, round to nearest even
}
__device__ __forceinline__ float f16_bits_to_float(uint32_t b) {
  return (float)__builtin_bit_cast(_Float16, (uint16_t)b);
}
__device__ __forceinline__ uint32_t float_to_f16_bits(float f) {
  return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)f);
}

// Two fp32 -> one dword of packed 16-bit elements (low half = a).
template <typename T> __device__ __forceinline__ uint32_t pack2(float a, float b);
template <> __device__ __forceinline__ uint32_t pack2<bf16_t>(float a, float b) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  f32x2 f = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
}
template <> __device__ __forceinline__ uint32_t pack2<f16_t>(float a, float b) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
  f32x2 f = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, f16x2));
}
// two floats -> two e4m3 bytes in the low (hi = false) or high half of `old`; saturating at the format's largest value
__device__ __forceinline__ uint32_t cvt_e4m3_pair(float a, float b, uint32_t old, bool hi) {
  a = __builtin_amdgcn_fmed3f(a, -448.f, 448.f);
  b = __builtin_amdgcn_fmed3f(b, -448.f, 448.f);
  return hi ? (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(a, b, (int)old, true) : (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(a, b, (int)old, false);
}

template <typename T> __device__ __forceinline__ float unpack_lo(uint32_t w);
template <typename T> __device__ __forceinline__ float unpack_hi(uint32_t w);
template <> __device__ __forceinline__ float unpack_lo<bf16_t>(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
template <> __device__ __forceinline__ float unpack_hi<bf16_t>(uint32_t w) { return __builtin_bit_cast(float, w & 0xffff0000u); }
template <> __device__ __forceinline__ float unpack_lo<f16_t>(uint32_t w) { return f16_bits_to_float(w & 0xffffu); }
template <> __device__ __forceinline__ float unpack_hi<f16_t>(uint32_t w) { return f16_bits_to_float(w >> 16); }

// ---- wave64 butterflies ---------------------------------------------------------------------------
// Wave-wide reductions on the DPP network (row shifts, then the two row broadcasts of this ISA family); the
// result is read from lane 63 into a scalar register, so every lane gets it.  All 64 lanes must be active.
// Six VALU instructions, against six LDS-crossbar round trips for the same reduction written with shuffles.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_move(float old, float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, old), __builtin_bit_cast(int, v), CTRL,
                                                               ROW_MASK, 0xf, false));
}
__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, dpp_move<0x111, 0xf>(-INFINITY, v));  // row_shr:1
  v = fmaxf(v, dpp_move<0x112, 0xf>(-INFINITY, v));  // row_shr:2
  v = fmaxf(v, dpp_move<0x114, 0xf>(-INFINITY, v));  // row_shr:4
  v = fmaxf(v, dpp_move<0x118, 0xf>(-INFINITY, v));  // row_shr:8: lane 15 of a row holds the row's result
  v = fmaxf(v, dpp_move<0x142, 0xa>(-INFINITY, v));  // row_bcast:15 into rows 1 and 3
  v = fmaxf(v, dpp_move<0x143, 0xc>(-INFINITY, v));  // row_bcast:31 into rows 2 and 3
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}
__device__ __forceinline__ float wave_sum(float v) {
  v += dpp_move<0x111, 0xf>(0.f, v);
  v += dpp_move<0x112, 0xf>(0.f, v);
  v += dpp_move<0x114, 0xf>(0.f, v);
  v += dpp_move<0x118, 0xf>(0.f, v);
  v += dpp_move<0x142, 0xa>(0.f, v);
  v += dpp_move<0x143, 0xc>(0.f, v);
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}
// The same within every aligned group of 16 lanes (a DPP row): xor-butterflies over the quad, then the two
// mirrors; every lane of the group ends with the group's result.  Lanes of a group must be active together.
__device__ __forceinline__ float group16_max(float v) {
  v = fmaxf(v, dpp_move<0xb1, 0xf>(v, v));   // quad_perm [1, 0, 3, 2]
  v = fmaxf(v, dpp_move<0x4e, 0xf>(v, v));   // quad_perm [2, 3, 0, 1]
  v = fmaxf(v, dpp_move<0x141, 0xf>(v, v));  // row_half_mirror
  v = fmaxf(v, dpp_move<0x140, 0xf>(v, v));  // row_mirror
  return v;
}
__device__ __forceinline__ float group16_sum(float v) {
  v += dpp_move<0xb1, 0xf>(v, v);
  v += dpp_move<0x4e, 0xf>(v, v);
  v += dpp_move<0x141, 0xf>(v, v);
  v += dpp_move<0x140, 0xf>(v, v);
  return v;
}
__device__ __forceinline__ int wave_sum_i(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Sum over the lanes up to and including this one.
__device__ __forceinline__ int wave_prefix_sum(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // a prefix within every row of 16 lanes
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row 0's total into row 1, row 2's into row 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // the first half's total into rows 2 and 3
  return v;
}

// ---- block numbering of the dense attention kernels -------------------------------------------------------
// Hardware block ids are dealt round-robin to the 8 XCDs (one L2 each): XCD x runs the blocks x, x + 8, ... in
// that order, a new one whenever a slot of its 32 CUs falls free.  The K/V heads (`units`) are dealt round-robin
// to the XCDs -- with right-padded batches a contiguous run of heads is one batch item, and the XCD that drew
// the longest sequence would finish last -- and an XCD works through its heads in sets.  A set is one head when
// the blocks cost the same (`balance` false) or a head alone has several blocks per slot; its K and V then stay
// in that L2.  When the blocks of a head differ in cost (causal: block index 0 is the longest) and a head has
// few of them, a set takes as many heads as give about two blocks per slot and runs them longest block first
// over all its heads: started in that order, the short blocks fill the slots the long ones leave, where head
// after head the last head's longest block would start when the others are almost through.
// `blocks` = blocks per (head, member of its group), `group` = query heads per K/V head, `unit_bytes` = what the
// blocks of one K/V head stream through L2 (they share it while they run side by side): a set never takes more heads
// than bring 8 MB of that, twice an XCD's L2 -- with more, the blocks of a head that are in flight together become
// too few to share their tiles, and on long sequences that costs more than the balance gains (dK/dV kernel on
// B=8, Hkv=8, group 4, N=8192, D=128: 10.1 ms with sets of four heads, 7.5 ms head after head).  Returns false for
// the padding blocks of the grid (xcd_grid workgroups), else the K/V head, the block index and the member.  `padded`: the batch has lengths.
//
// Where the heads do not divide among the XCDs, the last four, two and / or one of them are split over two, four or eight
// XCDs each, which take its blocks in turn, before their whole heads.  (All heads' blocks in one line cut into eight equal runs
// gave one XCD the long blocks of a head and its neighbour the short ones.)  Causal forward and backward: 4 heads in single
// precision, N = 8192: 2925 -> 2135 us; 5 x 16/4 heads, N = 1024, D = 128, bf16, flat scores: 550 -> 498.
inline unsigned xcd_grid(long long units, long long inner) {
  long long per_xcd = units / 8 * inner;
  for (int c = 4; c > 0; c >>= 1)
    if (units & c) per_xcd += (inner + 8 / c - 1) / (8 / c);
  return (unsigned)(per_xcd * 8);
}
__device__ __forceinline__ bool xcd_block_map(bool padded, int units, int blocks, int group, bool balance, long long unit_bytes, int& unit, int& blk,
                                              int& member) {
  const int inner = blocks * group;
  const int x = (int)(blockIdx.x & 7);
  long long seq = (long long)(blockIdx.x >> 3);
  const int upx = units / 8;  // whole heads of this XCD
  int first = upx * 8;
#pragma unroll
  for (int c = 4; c > 0; c >>= 1) {
    if (units & c) {
      const int st = 8 / c, sub = x % st, n = (inner - sub + st - 1) / st;
      if (seq < n) {
        const int idx = (int)seq * st + sub;
        unit = first + x / st;
        blk = idx / group;
        member = idx % group;
        return true;
      }
      seq -= n;
      first += c;
    }
  }
  if (seq >= (long long)upx * inner) return false;
  constexpr int kSetBlocks = 256;  // two blocks for each of 32 CUs x 4 resident blocks
  constexpr long long kSetBytes = 8ll << 20;
  int g = balance ? (kSetBlocks + inner - 1) / inner : 1;
  const long long by_bytes = unit_bytes > 0 ? kSetBytes / unit_bytes : (long long)upx;
  g = g < by_bytes ? g : (int)by_bytes;
  g = g < 1 ? 1 : g;
  g = g < upx ? g : upx;
  const int set = (int)(seq / ((long long)g * inner));
  const int s = (int)(seq - (long long)set * g * inner);
  const int gsize = (upx - set * g) < g ? (upx - set * g) : g;
  const int span = gsize * group;
  blk = s / span;
  // The XCD's 32 CUs take the workgroups of a launch in order, round after round (read from the hardware's id registers), and padding
  // returns at once.  So the heads of a padded batch change places behind each round, or the blocks of one long sequence among
  // short ones all fall to the same few CUs, every second one of a set of two heads.  fp32, 2 x 8 heads, N = 1500 and 375, D = 64,
  // forward and backward: 292 -> 244 us; q of spread 3: 280 -> 228.  (Places changed from block to block fall to half of the CUs as
  // well.)  Without lengths the order stays: changed, training of 4 x 16 heads, N = 2048, D = 128, bf16, flat, took 620 us for 613,
  // prefill of 4 x 16/4, N = 1024, D = 128, fp32, spread 3: 145.2 for 144.0.
  int r = s % span;
  if (padded && gsize > 1) {
    asm volatile("; several heads");  // (a branch: the divisions are a tenth of a microsecond of the smallest calls)
    r += (s - r) / 32 % span;
    r = r < span ? r : r - span;
  }
  unit = (set * g + r / group) * 8 + x;
  member = r % group;
  return true;
}

// The item at place `pos` of a batch, and its length; `longest_first`: the places are in the order of the lengths.  Workgroups start in the
// order of their numbers, and those that find no slot at first start when others end: a long sequence in that place makes a launch longer.
// Head u of a batch runs on XCD u % 8, so with fewer than eight K/V heads an item has some of the XCDs only: every second round of items over the
// XCDs goes backwards, or the same XCDs have the longer items of every round.  us, the items' order (three batches with the same lengths) ->
// plainly longest first -> this: forward of 4 x 4 heads, N <= 1500, D = 64, bf16: 46, 54, 68 -> 55 -> 43 to 46; 5 x 4 of 700, D = 128, f16, alpha = 1.333,
// training: 111, 122, 122 -> 108 to 111 -> 91 to 94; 8 x 4 of 3000, flat, forward: 190, 147, 132 -> 134 -> 116 to 123.
// For kernels whose blocks of a sequence cost the same (not causal) and take long: 16 x 12 heads, N <= 500, D = 64, bf16, training: 113 to 116 -> 107 to 109;
// 8 x 16 heads, N <= 2000, flat, alpha = 1.333: forward 370 -> 346, forward and backward 839 -> 782; 16 x 4 heads: 548 to 589 -> 494; fp32, alpha = 1.333,
// 8 x 8 heads, N <= 700: 291 -> 275; 6 x 8 of 600, D = 128, alpha = 2: 255 -> 237.  Causal launches, whose sets of heads run longest block first, lose
// (8 x 16 heads, N <= 2000, flat, bf16: 320 -> 340), and so do the short workgroups of the resident forward (16 x 12 heads: 40.9 -> 43.0; 32 x 8 of 300: 25.6 -> 29.3).
// And launches of many rounds of workgroups (`blocks` per K/V head, `per_cu` at a time on a CU), where the end is a small part and items of different lengths side by side do better than of
// the same; the more so, the more items: training, D = 128: 32 x 16 heads, N <= 500, bf16 (8 rounds): 489, 505, 499 -> 535; 60 x 8 of 400 (7.5): 365 -> 416; 16 x 16 of 1500, flat
// (12): 1442, 1467, 1431 -> 1464; fp32 32 x 16 of 300 (20): 827 -> 901; at the lines 16 x 8 of 500, fp32 (8): 470, 460, 453 -> 452; 20 x 16 of 300, bf16 (3.75): 164, 157, 166 -> 154;
// 32 x 8 of 500, D = 64 (2): 131, 134, 132 -> 126.  A few heads, which the items' order shares out unevenly, gain in any number: 50 x 2 of 600, fp32: 268, 250, 264 -> 244.
struct BatchItem {
  int b, L;
};
__device__ __forceinline__ BatchItem batch_item(const void* varlen, int varlen_bits, int B, int N, int pos, int Hkv, int blocks, bool longest_first, int per_cu) {
  // (What only padded batches need stands behind the other code, and the number of workgroups is formed here: gridDim would bring 256 bytes of hidden arguments to
  // every launch.  Forward of 8 heads, N = 128, fp32, which starts from cold instruction lines: 12.2 -> 12.05 us; 4 x 16/4 heads, N = 1024, D = 128: 138.2 -> 137.0.)
  if (__builtin_expect(!varlen, 1)) return {pos, N};
  auto length_of = [&](int i) -> int {
    const long long l = varlen_bits == 64 ? ((const long long*)varlen)[i] : (long long)((const int*)varlen)[i];
    return (int)(l < 0 ? 0 : (l > N ? N : l));
  };
  const bool few_rounds = (uint32_t)(B * Hkv) * (uint32_t)blocks <= (B <= 16 ? 8u : B <= 24 ? 4u : 2u) * 256u * (uint32_t)per_cu, few_heads = Hkv % 8 != 0 && B * Hkv <= 128;
  if (!longest_first || B > 64 || !(few_rounds || few_heads)) return {pos, length_of(pos)};
  const int lane = (int)(threadIdx.x & 63);
  const int len = length_of(lane < B ? lane : B - 1);
  const int key = lane < B ? len * 64 + 63 - lane : -1;  // (the length, and of equal ones the earlier; lengths are below 2^24)
  int rank = 0;
  for (int i = 0; i < B; ++i) rank += __builtin_amdgcn_readlane(key, i) > key ? 1 : 0;
  const int c = Hkv & 1 ? 8 : Hkv & 2 ? 4 : Hkv & 4 ? 2 : 1;  // places after which the heads are back at the first XCD
  const int row = pos & -c;
  if ((row & c) != 0 && row + c <= B) pos = 2 * row + c - 1 - pos;
  const int b = __builtin_ctzll(__builtin_amdgcn_ballot_w64(rank == pos));
  return {b, __builtin_amdgcn_readlane(len, b)};
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float fast_log2(float x) { return __builtin_amdgcn_logf(x); }
__device__ __forceinline__ float fast_rcp(float x) { return __builtin_amdgcn_rcpf(x); }

}  // namespace adsp
