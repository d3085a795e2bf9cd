// Sparse entmax attention on workgroups of 32 rows for gfx950, head dims 64 and 128: single-precision forward, dQ and dK/dV
// kernels, and the forward for some 16-bit problems.
//
// What bounds them: vector and matrix pipe together on large problems (per block of 32 x 32 scores and product of 64 columns 24 matrix
// products of 32 cycles and about 110 vector instructions for their operands), and on ordinary ones the length of a workgroup's
// walk over the keys, because a K/V head of N keys has only N / rows workgroups; the forward's solves beside it.
//
// Products: an fp32 operand from 2^-110 on is the sum of three bf16 values exactly (below, the third part is rounded to bf16's smallest number, 2^-133: 2^-18 of
// 2^-116), and six of the nine products of the parts are formed.  The three that are left out are 2^-22 of a product at most, and a small part of fp32's rounding on
// average.  On the bf16 matrix pipe the six take 192 cycles per 16 columns where v_mfma_f32_32x32x2_f32 takes 512, and round less often: relative
// error against 64 bits, fp32 products -> these, of output, dQ, dK, dV: N = 1500, D = 64 4.0e-7, 4.5e-7, 4.5e-7, 4.0e-7 -> 2.7e-7, 3.3e-7, 3.2e-7, 2.8e-7;
// q of spread 3 5.6e-7, 9.4e-7, 9.5e-7, 5.7e-7 -> 3.9e-7, 6.7e-7, 6.9e-7, 4.0e-7; flat 2.1e-7 ... 3.1e-7 -> 1.4e-7 ... 1.9e-7; D = 128
// 3.7e-7, 9.2e-7, 9.2e-7, 8.5e-7 -> 3.4e-7, 3.6e-7, 3.6e-7, 3.5e-7; dQ with a V of mean 10: 1.5e-6 -> 1.1e-6, a K of mean 10: 2.7e-6 -> 1.8e-6.  The small products
// have an accumulator of their own: added to the sum itself, their roundings made these errors 1.2 to 2 times those of fp32 products.
//
// The 16-bit forward: vector issue (its products are a sixteenth as long; about 1400 vector instructions per block of 32 x 32 scores,
// most of them insertions into the lists; matrix pipe 1-2 %, vector pipe about 50 % of the busy SIMD cycles).
//
// Split: a workgroup is four waves and owns 32 rows (queries; keys in the dK/dV kernel); the waves share the rows and
// take the 32-row blocks of the other side in turn, and meet in LDS at the end of a walk.  Against 128 rows per workgroup,
// 32 per wave, a walk is a quarter as long and there are four times as many workgroups.  A wave's operands come through a
// ring of three 4 KB chunks ([32 rows][32 columns]) of LDS of its own, loaded two chunks ahead with direct 16-byte loads:
// a chunk lasts 400 to 900 cycles of matrix and vector work, so the waves need no barrier inside a walk and no tile shared by them.  Each
// operand block is read by one workgroup of 32 rows instead of 128, about 30 bytes per cycle and CU out of L2.  The gradients' own rows
// lie in LDS, split once by all four waves (in registers, 33 to 192 others were spilled).
//
// Forward, one product per (row, key) where supports are short: tau over a subset of the keys is a lower bound of tau over
// all of them, so a wave lists the scores above its row's bound while it walks, and after 1, 2, 4, 8, ... steps the
// workgroup solves the rows on what is listed so far and drops what fell below.  Between two such points about as
// many scores join as a support holds.  Behind the last step the solution is the threshold itself, to fp32 rounding,
// and the output gathers the V rows of the support.  A row whose part of a wave's list overflows (flat scores) sends the
// workgroup to walks: Newton steps on (sum u^c0)^(1/c0) - 1 from the bound the lists gave, until a step is below 2e-5, and
// an output walk.
//
// One such workgroup among hundreds takes the whole launch two to three times as long, and with scores of unit spread it came about by
// chance (a row of 38 members, 14 of them in one wave's list, which 19 scores joined).  Hence the solves come sooner where a row has
// many members (sync(): a solve costs about 1.5 us, so none is added for fewer), and a wave drops what lies below the bound before it
// gives up.  us, q of spread 1: 2 x 8 heads, N = 1500 and 375: 126 -> 66 (65 where no list overflows); N = 2048: 187 -> 101, D = 128, 16/4 heads:
// 288 -> 148; 4 heads, N = 8192: 776 -> 285; bf16, 2 heads, N = 4096, D = 128: 135 -> 75.  Spread 3, where nothing overflows: 82.8 -> 83.2.
//
// Measured (fp32, forward and backward, us; kernels on 128 rows a workgroup -> fp32 products -> these): causal, 2 x 8 heads, N = 1500 and 375,
// D = 64: 1140 -> 241 -> 158 (forward 50, dQ 62, dK/dV 58), flat 316 -> 201; 4 x 16/4 heads, N = 1024, D = 128: 2885 -> 928 -> 700; alpha = 1.333, 8 x 16 heads,
// N = 1024, not causal: 4818 -> 2686 -> 1800; prefill of 8 heads, N = 128: 11.4 -> 11.3.
// Where 16-bit calls come here: rows32_16bit in attn_api.hip.
#pragma once
#include <cfloat>

#include "attn_bwd_kernel.h"

namespace adsp {
namespace f32path {

constexpr int kRows = 32;        // rows per workgroup, and per block of the other side
constexpr int kWaves = 4;
constexpr int kChunk = 4096;     // bytes of a chunk: 32 rows of 128 bytes, 16-byte pieces swizzled
constexpr int kStages = 3;
constexpr int kRing = kWaves * kStages * kChunk;
constexpr int kCap = 32;         // list entries per row and wave
constexpr int kListBytes = kWaves * kCap * kRows * 6;  // a score (fp32) and a key index (16 bits) per entry

// position of 16-byte piece c of chunk row r
__device__ __forceinline__ int piece_sw(int row) { return (row >> 1) & 7; }

// 4-byte global -> LDS copy per lane: lane i writes the i-th word behind the wave-uniform `lds`
__device__ __forceinline__ void dma4(const float* g, float* lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off"
               :
               : "v"(g), "s"(__builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)lds))
               : "memory");
}

// A wave's ring of chunks and its place in it; kStride: bytes per row of the tensors its chunks come from.
template <int kStride> struct Ring {
  unsigned char* base;  // the wave's three chunks
  int lane;
  uint32_t off[2];      // the lane's place in an even / odd group of eight rows, from the group's first row
  int st;               // stage of the next chunk to be consumed
  __device__ __forceinline__ Ring(unsigned char* b, int l) : base(b), lane(l), st(0) {
    const int p0 = (l & 7) ^ (l >> 4);
    off[0] = (uint32_t)((l >> 3) * kStride + p0 * 16);
    off[1] = (uint32_t)((l >> 3) * kStride + (p0 ^ 4) * 16);
  }
  // chunk c (32 columns) of rows [row0, row0 + 32) of a row-major tensor into stage `s`; rows from `limit` on are replaced
  // by the last one in front of it
  __device__ __forceinline__ void issue(const unsigned char* g, int row0, int limit, int c, int s) const {
    unsigned char* l = base + s * kChunk;
    if (row0 + kRows <= limit) {
      const unsigned char* gb = uniform_ptr(g + (size_t)row0 * kStride + c * 128);
#pragma unroll
      for (int j = 0; j < 4; ++j) dma16s(gb + j * (8 * kStride), off[j & 1], l + j * 1024);
    } else {
      const unsigned char* gb = uniform_ptr(g + c * 128);
      const int p0 = (lane & 7) ^ (lane >> 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        int r = row0 + 8 * j + (lane >> 3);
        r = r < limit ? r : limit - 1;
        dma16s(gb, (uint32_t)r * (uint32_t)kStride + (uint32_t)((p0 ^ (4 * (j & 1))) * 16), l + j * 1024);
      }
    }
  }
  // The same in two calls, without a branch: rows() for a block, issue_rows() for each of its chunks
  uint32_t at[4];
  __device__ __forceinline__ void rows(int row0, int limit) {
    const int p0 = (lane & 7) ^ (lane >> 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      int r = row0 + 8 * j + (lane >> 3);
      r = r < limit ? r : limit - 1;
      at[j] = (uint32_t)r * (uint32_t)kStride + (uint32_t)((p0 ^ (4 * (j & 1))) * 16);
    }
  }
  __device__ __forceinline__ void issue_rows(const unsigned char* g, int c, int s) const {
    const unsigned char* gb = uniform_ptr(g + c * 128);
    unsigned char* l = base + s * kChunk;
#pragma unroll
    for (int j = 0; j < 4; ++j) dma16s(gb, at[j], l + j * 1024);
  }
  // the same in the layout of the transposing reads (16-bit V; see BwdTiles::tsw): row r's pieces moved by 2 r
  __device__ __forceinline__ void issue_t(const unsigned char* g, int row0, int limit, int c, int s) const {
    const unsigned char* gb = uniform_ptr(g + c * 128);
    unsigned char* l = base + s * kChunk;
    const int piece = (lane & 7) ^ ((2 * (lane >> 3)) & 7);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      int r = row0 + 8 * j + (lane >> 3);
      r = r < limit ? r : limit - 1;
      dma16s(gb, (uint32_t)r * (uint32_t)kStride + (uint32_t)(piece * 16), l + j * 1024);
    }
  }
  // Waits for the oldest of the two chunks under way and for the wave's own LDS reads (the stage the caller fills next is
  // the one it has just read); returns the LDS address of the chunk.
  __device__ __forceinline__ uint32_t arrive() const {
    asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)" ::: "memory");
    return (uint32_t)(uintptr_t)(base + st * kChunk);
  }
  __device__ __forceinline__ int ahead() const { return st == 0 ? 2 : st - 1; }  // stage of the chunk after next
  __device__ __forceinline__ void advance() { st = st == 2 ? 0 : st + 1; }
  __device__ __forceinline__ void drain() const { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory"); }
};

// A walk takes the blocks first, first + step, ... below n_blk, each SEQ chunks that src(blk, s, stage) issues.  `start` issues
// the first two chunks; `take` waits for chunk s of blk, issues the chunk after next (past the end: one that nothing reads,
// to keep the count) and returns the LDS address.
template <int SEQ, typename Src> __device__ __forceinline__ void start(int first, int n_blk, int step, Src&& src) {
  src(first, 0, 0);
  if constexpr (SEQ == 1) src(first + step < n_blk ? first + step : first, 0, 1);
  else src(first, 1, 1);
}
template <int SEQ, typename R, typename Src> __device__ __forceinline__ uint32_t take(R& ring, int blk, int s, int n_blk, int step, Src&& src) {
  const uint32_t a = ring.arrive();
  const int nb = blk + (s + 2) / SEQ * step;
  src(nb < n_blk ? nb : blk, (s + 2) % SEQ, ring.ahead());
  ring.advance();
  return a;
}
// The whole walk: body(blk, next) consumes a block's chunks by calls of next(0), next(1), ... in order.  kStarted: the caller has issued
// the first two chunks (`start`, where first < n_blk).
template <int SEQ, bool kStarted = false, typename R, typename Src, typename Body>
__device__ __forceinline__ void walk(R& ring, int first, int n_blk, int step, Src&& src, Body&& body) {
  if (first >= n_blk) return;
  ring.st = 0;
  if constexpr (!kStarted) start<SEQ>(first, n_blk, step, src);
  for (int blk = first; blk < n_blk; blk += step) body(blk, [&](int s) -> uint32_t { return take<SEQ>(ring, blk, s, n_blk, step, src); });
  ring.drain();
}

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
// Eight fp32 values as three bf16 parts each, whose sum is the value itself from 2^-110 on (8 + 8 + 8 bits; the first part is cut off instead of rounded, so
// that no finite value becomes infinite): the operand of a product of 32 x 32 x 16.
struct Split {
  u32x4 part[3];
};
// x less the low (high) half of a pair of bf16 values, as a product of pairs with (-1, 0) or (0, -1): one instruction for two.  (The constants
// are kept in scalar registers: as an operand inside the instruction -1 stands in the other half.)
__device__ __forceinline__ float less_half(float x, uint32_t pair, uint32_t minus_one) {
  asm("" : "+s"(minus_one));
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, pair), __builtin_bit_cast(bf16x2_t, minus_one), x, false);
}
__device__ __forceinline__ float less_lo(float x, uint32_t pair) { return less_half(x, pair, 0x0000bf80u); }
__device__ __forceinline__ float less_hi(float x, uint32_t pair) { return less_half(x, pair, 0xbf800000u); }
__device__ __forceinline__ Split split8(const float* x) {
  Split r;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float x0 = x[2 * i], x1 = x[2 * i + 1];
    const uint32_t hi = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, x1), __builtin_bit_cast(uint32_t, x0), 0x07060302u);
    const float r0 = less_lo(x0, hi), r1 = less_hi(x1, hi);
    const uint32_t mid = pack2<bf16_t>(r0, r1);
    r.part[0][i] = hi;
    r.part[1][i] = mid;
    r.part[2][i] = pack2<bf16_t>(less_lo(r0, mid), less_hi(r1, mid));
  }
  return r;
}
// main + small += a b of fp32 operands: the six largest of the nine products of their parts, the largest of them apart from the others (each
// product rounds its accumulator, and the small ones' is 2^-7 of it)
__device__ __forceinline__ void mfma_split(const Split& a, const Split& b, f32x16& main, f32x16& small) {
  small = mfma_16bit<bf16_t>(a.part[2], b.part[0], small);
  small = mfma_16bit<bf16_t>(a.part[0], b.part[2], small);
  small = mfma_16bit<bf16_t>(a.part[1], b.part[1], small);
  small = mfma_16bit<bf16_t>(a.part[1], b.part[0], small);
  small = mfma_16bit<bf16_t>(a.part[0], b.part[1], small);
  main = mfma_16bit<bf16_t>(a.part[0], b.part[0], main);
}

// kPairs pairs of 16-byte pieces of a row, the lane's half of each
template <int kPairs> __device__ __forceinline__ void load_row(const unsigned char* row, int lh, uint32_t (&f)[4 * kPairs]) {
#pragma unroll
  for (int g = 0; g < kPairs; ++g) {
    const u32x4 raw = *reinterpret_cast<const u32x4*>(row + 32 * g + 16 * lh);
#pragma unroll
    for (int e = 0; e < 4; ++e) f[g * 4 + e] = raw[e];
  }
}

// The lane's own row as the operand of products over the columns: of every chunk the pieces 2 g + lh (load_row)
template <typename T, int NC> struct OwnRow {
  static constexpr bool k16 = is16<T>::value;
  uint32_t f[k16 ? 16 * NC : 1];
  Split sp[k16 ? 1 : 2 * NC];
  __device__ __forceinline__ void load(const unsigned char* row, int lh) {
    if constexpr (k16) {
      load_row<4 * NC>(row, lh, f);
    } else {
      uint32_t raw[16 * NC];
      load_row<4 * NC>(row, lh, raw);
#pragma unroll
      for (int s = 0; s < 2 * NC; ++s) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = __builtin_bit_cast(float, raw[8 * s + e]);
        sp[s] = split8(x);
      }
    }
  }
  __device__ __forceinline__ const Split& get(int s) const { return sp[s]; }
};
// The same in LDS, for kernels that have no registers for it (the workgroup's waves have the same rows): 64 lanes x 16 bytes per operand
template <int NC> struct OwnRowLds {
  static constexpr int kBytes = 2 * NC * 3 * 1024;
  uint32_t at;
  // each wave splits its share of the steps; a barrier has to come in front of the first get()
  __device__ __forceinline__ OwnRowLds(const unsigned char* row, unsigned char* lds, int wave, int lane) : at((uint32_t)(uintptr_t)lds + lane * 16) {
    for (int s = wave; s < 2 * NC; s += kWaves) {
      float x[8];
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const f32x4 raw = *reinterpret_cast<const f32x4*>(row + 64 * s + 32 * g + 16 * (lane >> 5));
#pragma unroll
        for (int e = 0; e < 4; ++e) x[4 * g + e] = raw[e];
      }
      const Split sp = split8(x);
#pragma unroll
      for (int i = 0; i < 3; ++i) *reinterpret_cast<u32x4*>(lds + (s * 3 + i) * 1024 + lane * 16) = sp.part[i];
    }
  }
  __device__ __forceinline__ Split get(int s) const { return Split{{lds_read16(at, (s * 3) * 1024), lds_read16(at, (s * 3 + 1) * 1024), lds_read16(at, (s * 3 + 2) * 1024)}}; }
};
// acc (+ small) += (rows of chunk c) . (the lane's own row) over the chunk's columns
template <typename T, typename Own> __device__ __forceinline__ void dot_chunk(f32x16& acc, f32x16& small, uint32_t chunk, uint32_t row_lane, const Own& own, int c) {
  u32x4 a[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) a[g] = lds_read16((chunk + row_lane) ^ (g << 5));
  if constexpr (is16<T>::value) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const uint32_t* f = own.f + 16 * c + 4 * g;
      acc = mfma_16bit<T>(a[g], u32x4{f[0], f[1], f[2], f[3]}, acc);
    }
  } else {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t word = a[2 * s + e / 4][e % 4];  // (a bit cast of a vector's element takes the wrong one)
        x[e] = __builtin_bit_cast(float, word);
      }
      mfma_split(split8(x), own.get(2 * c + s), acc, small);
    }
  }
}
// a block's sixteen weights of the lane's row, in accumulator order, as operands
__device__ __forceinline__ void split16(const float (&w)[16], Split (&sp)[2]) {
  sp[0] = split8(w);
  sp[1] = split8(w + 8);
}
// o[x][column of the chunk][lane's row] += sum over the chunk's rows of chunk[row][column] * (weights x)[row]; kShift: o[0] -= shift o[1] before it; kInf: an infinite
// sum stays what it is, whatever the small products (NaN, where an operand is infinite)
template <bool kShift = false, bool kInf = false, int kN> __device__ __forceinline__ void acc_chunk(f32x16* const (&o)[kN], uint32_t chunk, uint32_t col_lane, const Split (&w)[kN][2], float shift = 0.f) {
  float a[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    // row 8 (i / 4) + 4 lh + i % 4: its swizzle differs from the lane's constant part by an immediate
    const int x = (4 * ((i >> 2) & 1)) ^ ((i >> 1) & 1);
    a[i] = *(const __attribute__((address_space(3))) float*)(((chunk + col_lane) ^ (x << 4)) + (8 * (i >> 2) + (i & 3)) * 128);
  }
  f32x16 part[kN];
#pragma unroll
  for (int n = 0; n < kN; ++n)
#pragma unroll
    for (int i = 0; i < 16; ++i) part[n][i] = kShift && n == 0 ? -shift * (*o[kN - 1])[i] : 0.f;
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const Split as = split8(a + 8 * s);
#pragma unroll
    for (int n = 0; n < kN; ++n) mfma_split(as, w[n][s], *o[n], part[n]);
  }
#pragma unroll
  for (int n = 0; n < kN; ++n)
#pragma unroll
    for (int i = 0; i < 16; ++i) (*o[n])[i] += kInf ? __builtin_amdgcn_fmed3f(part[n][i], -FLT_MAX, FLT_MAX) : part[n][i];
}
// the same for a 16-bit chunk of 64 columns (issue_t): o[0] takes columns 0 .. 31, o[1] the others
template <typename T> __device__ __forceinline__ void acc_chunk_16(f32x16 (&o)[2], uint32_t chunk, int lane, const float (&w)[16]) {
  const int a4 = lane & 15, grp = lane >> 4, r = a4 >> 2, c = a4 & 3, dl = grp & 1;
  uint32_t ta[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int x = 4 * (grp >> 1) + r + 8 * h;
    ta[h] = chunk + (uint32_t)(x * 128 + (((2 * dl + (c >> 1)) ^ ((2 * x) & 7)) << 4) + (c & 1) * 8);
  }
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const u32x4 b = {pack2<T>(w[8 * s], w[8 * s + 1]), pack2<T>(w[8 * s + 2], w[8 * s + 3]), pack2<T>(w[8 * s + 4], w[8 * s + 5]),
                     pack2<T>(w[8 * s + 6], w[8 * s + 7])};
#pragma unroll
    for (int db = 0; db < 2; ++db) {
      const u32x2_t a0 = lds_read8_tr(ta[0] ^ (db << 6), 16 * s * 128);
      const u32x2_t a1 = lds_read8_tr(ta[1] ^ (db << 6), 16 * s * 128);
      o[db] = mfma_16bit<T>(u32x4{a0[0], a0[1], a1[0], a1[1]}, b, o[db]);
    }
  }
}
__device__ __forceinline__ uint32_t row_lane_of(int lq, int lh) { return (uint32_t)(lq * 128 + ((lh ^ piece_sw(lq)) << 4)); }
__device__ __forceinline__ uint32_t col_lane_of(int lq, int lh) {
  return (uint32_t)(4 * lh * 128 + (((lq >> 2) ^ (2 * lh)) << 4) + (lq & 3) * 4);
}

// Adds up the four waves' o (32 columns per block, accumulator layout) in LDS and writes scale[row] * sum to the rows
// [row0, row0 + 32) below n of a row-major tensor.  `smem` holds 4 x 32 x D floats; every wave is done with what it held.
template <int D, typename T, typename Scale>
__device__ __forceinline__ void combine_store(const f32x16 (&o)[D / 32], unsigned char* smem, T* out, int row0, int n, int wave,
                                              int lane, Scale&& scale) {
  using KS = Swz<D * 4>;
  const int lq = lane & 31, lh = lane >> 5, tid = wave * 64 + lane;
  unsigned char* mine = smem + wave * (kRows * D * 4);
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<f32x4*>(mine + KS::off(lq, db * 8 + 2 * g + lh)) =
          f32x4{o[db][4 * g], o[db][4 * g + 1], o[db][4 * g + 2], o[db][4 * g + 3]};
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kRows * D / 4 / 256; ++j) {
    const int id = j * 256 + tid, row = id / (D / 4), c = id % (D / 4);
    const int at = KS::off(row, c);
    f32x4 s = *reinterpret_cast<const f32x4*>(smem + at);
#pragma unroll
    for (int w = 1; w < kWaves; ++w) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(smem + w * (kRows * D * 4) + at);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] += x[e];
    }
    const float k = scale(row);
    if (row0 + row >= n) continue;
    unsigned char* at_out = reinterpret_cast<unsigned char*>(out) + ((size_t)(row0 + row) * D + c * 4) * (is16<T>::value ? 2 : 4);
    if constexpr (is16<T>::value) *reinterpret_cast<u32x2*>(at_out) = u32x2{pack2<T>(s[0] * k, s[1] * k), pack2<T>(s[2] * k, s[3] * k)};
    else *reinterpret_cast<f32x4*>(at_out) = f32x4{s[0] * k, s[1] * k, s[2] * k, s[3] * k};
  }
}

// over the eight lanes of a row: two quad permutations and a mirror of eight lanes, without a trip through LDS
template <int kCtrl> __device__ __forceinline__ float dpp(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), kCtrl, 0xf, 0xf, true));
}
__device__ __forceinline__ float sum8(float x) {
  x += dpp<0xb1>(x);   // quad_perm [1, 0, 3, 2]
  x += dpp<0x4e>(x);   // quad_perm [2, 3, 0, 1]
  return x + dpp<0x141>(x);  // row_half_mirror
}
__device__ __forceinline__ float max8(float x) {
  x = fmaxf(x, dpp<0xb1>(x));
  x = fmaxf(x, dpp<0x4e>(x));
  return fmaxf(x, dpp<0x141>(x));
}

// u^c0 and u^(c0 - 1) of u >= 0
template <int AM> __device__ __forceinline__ void powers(float u, float c0, float& e0, float& e1) {
  if constexpr (AM == ATT_15) {
    e0 = u * u;
    e1 = u;
  } else if constexpr (AM == ATT_2) {
    e0 = u;
    e1 = u > 0.f ? 1.f : 0.f;
  } else {
    e1 = fast_exp2(fast_log2(u) * (c0 - 1.f));  // (0 at 0)
    e0 = e1 * u;
  }
}
// Newton step on (sum u^c0)^(1/c0) - 1: convex and decreasing in the threshold, nearly linear where the support is settled
template <int AM> __device__ __forceinline__ float norm_step(float s0, float s1, float c0) {
  if constexpr (AM == ATT_2) return (s0 - 1.f) * fast_rcp(s1);
  if constexpr (AM == ATT_15) {
    const float g = __builtin_amdgcn_sqrtf(s0);  // g - 1 = (s0 - 1) / (g + 1): exact where it is small
    return (s0 - 1.f) * s0 * fast_rcp((g + 1.f) * g * s1);
  }
  const float g = fast_exp2(fast_log2(s0) / c0);
  return (g - 1.f) * s0 * fast_rcp(g * s1);
}

// Blocks of a causal launch, longest first over all heads of an XCD by what they walk (a padded batch's lengths included; empty blocks come
// last).  `two`: of the kernels of which two workgroups run on a CU at a time, a launch that is under way at once has its second round over the XCD's 32 CUs
// backwards, so that the CU with the longest block of the first has the shortest of the second.  In longer launches blocks go where one ends, and
// every second round backwards costs: 4 x 16/4 heads, N = 1024, D = 128: 717 -> 792 us.
// us, order of xcd_block_map -> this, forward and backward, D = 64: 2 x 8 heads, N = 1500 and 375: 159.0 -> 156.8; 2 x 8 of 1024: 121.6 -> 116.7;
// 8 of 2048: 211 -> 202; with lengths, three batches each: 8 x 8, N <= 700: 151, 152, 134 -> 125; 4 x 16, N <= 1024, forward: 69, 73, 72 -> 62; 8 x 8 of 2000: 613 -> 572; D = 128: 4 x 8,
// N <= 1100: 407, 397, 396 -> 255; 8 x 8 of 1000: 510, 524, 458 -> 411; 4 x 16/4, N <= 1024: 519, 573, 631 -> 507, 544, 612; in long launches of many items it can lose: 32 x 8/2, N <= 900: 1616 -> 1644.
// Without lengths xcd_block_map goes by the same order over sets of heads of 256 blocks.  From two such sets on theirs, whose K and V are fewer, is the faster one:
// this -> theirs, forward and backward, D = 64: 8 x 16/8 heads, N = 1024: 681 -> 667; 8 x 32/8 of 512: 421 -> 415; 8 x 8 of 2048: 1181 -> 1167; below, where a set is
// left that is not whole, this one is: 6 x 8 of 2048, forward: 221, theirs 228.
// For up to 2048 keys and eight heads per XCD, a lane per length and per head, with the heads' operands in 8 MB as in xcd_block_map.
// `keys`: a block of keys is the longer the earlier it is.  False: the launch is not of this kind.
__device__ __forceinline__ bool longest_first(const void* varlen, int varlen_bits, int B, int Hkv, int N, int group, bool causal, long long unit_bytes, bool keys, bool two,
                                              int& bkv, int& rblk, int& member) {
  const int n = (N + kRows - 1) / kRows, heads = B * Hkv / 8, x = (int)(blockIdx.x & 7);
  if (!causal || n > 64 || (B * Hkv) % 8 != 0 || heads > 8 || heads * unit_bytes > (8ll << 20)) return false;
  if (!varlen && heads * n * group >= 512) return false;
  const int lane = (int)(threadIdx.x & 63);
  int len = 0;  // blocks of head `lane` that are not empty; they are as long as 1, 2, ..., len
  if (lane < heads) len = (batch_item(varlen, varlen_bits, B, N, (lane * 8 + x) / Hkv, Hkv, 0, false, 1).L + kRows - 1) / kRows;
  int longer = 0;  // blocks longer than `lane`
  for (int u = 0; u < heads; ++u) {
    const int more = __builtin_amdgcn_readlane(len, u) - lane;
    longer += more > 0 ? more : 0;
  }
  const int total = __builtin_amdgcn_readlane(longer, 0) * group;
  int s = (int)(blockIdx.x >> 3), u = 0;
  if (s < total) {
    if (two && total <= 64 && s >= 32) s = 31 + total - s;
    const int t = 63 - __builtin_clzll(__builtin_amdgcn_ballot_w64(longer * group > s));  // the block is t + 1 long
    const int j = s - (t < 63 ? __builtin_amdgcn_readlane(longer, t < 63 ? t + 1 : 63) * group : 0);
    member = j % group;
    unsigned long long with = __builtin_amdgcn_ballot_w64(len > t);
    for (int k = j / group; k > 0; --k) with &= with - 1;
    u = __builtin_ctzll(with);
    rblk = keys ? __builtin_amdgcn_readlane(len, u) - 1 - t : t;
  } else {
    s -= total;
    member = s % group;
    int k = s / group, have = __builtin_amdgcn_readlane(len, 0);
    while (u < heads - 1 && k >= n - have) {
      k -= n - have;
      have = __builtin_amdgcn_readlane(len, ++u);
    }
    rblk = have + k;
  }
  bkv = u * 8 + x;
  return true;
}

// ---------------------------------------------------------------------------------------------------------
// forward
// ---------------------------------------------------------------------------------------------------------
template <int D> constexpr int fwd_smem() {
  const int a = kRing + kListBytes, b = kWaves * kRows * D * 4;
  return a > b ? a : b;
}

template <typename T, int D, int AM>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void attn_rows32_fwd_kernel(AttnParams p) {
  constexpr bool k16 = is16<T>::value;
  constexpr int kStride = D * (k16 ? 2 : 4);
  constexpr int NC = kStride / 128;  // chunks per block
  __shared__ __align__(4096) unsigned char smem[fwd_smem<D>()];
  __shared__ float t_lds[kRows], est_lds[kRows];
  __shared__ uint8_t n_lds[kWaves][2][kRows];
  __shared__ float red[2][kWaves][3][kRows];
  __shared__ uint32_t over_flag, sync_lds[kWaves];  // sync_lds: how much nearer the next solve has to be
  float* const list_s = reinterpret_cast<float*>(smem + kRing);                                   // [wave][slot][row]
  uint16_t* const list_k = reinterpret_cast<uint16_t*>(smem + kRing + kWaves * kCap * kRows * 4);  // likewise

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, lq = lane & 31, lh = lane >> 5;
  const int N = p.N, group = p.Hq / p.Hkv, n_rblk = (N + kRows - 1) / kRows;
  int bkv, mi, hg, rblk;
  if (!k16 && longest_first(p.varlen, p.varlen_bits, p.B, p.Hkv, N, group, p.causal != 0, 2ll * N * kStride, false, true, bkv, rblk, hg)) mi = n_rblk - 1 - rblk;
  else if (!xcd_block_map(p.varlen != nullptr, p.B * p.Hkv, n_rblk, group, p.causal != 0, 2ll * N * kStride, bkv, mi, hg)) return;
  const BatchItem item = batch_item(p.varlen, p.varlen_bits, p.B, N, bkv / p.Hkv, p.Hkv, n_rblk * group, p.causal == 0, 2);
  const int b = item.b, L = item.L, kvh = bkv % p.Hkv, h = kvh * group + hg;
  bkv = b * p.Hkv + kvh;
  const int m0 = (n_rblk - 1 - mi) * kRows;
  const size_t q_row0 = (size_t)(b * p.Hq + h) * N;
  unsigned char* const out = reinterpret_cast<unsigned char*>(p.out) + q_row0 * kStride;
  if (m0 >= L) {
    const int rows = N - m0 < kRows ? N - m0 : kRows;
    for (int i = tid; i < rows * (kStride / 16); i += 256) reinterpret_cast<f32x4*>(out + (size_t)m0 * kStride)[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    return;
  }
  const unsigned char* kg = reinterpret_cast<const unsigned char*>(p.k) + (size_t)bkv * N * kStride;
  const unsigned char* vg = reinterpret_cast<const unsigned char*>(p.v) + (size_t)bkv * N * kStride;
  const int qi = m0 + lq;
  const bool live = qi < L;
  const int lim = p.causal ? (qi < L - 1 ? qi : L - 1) : L - 1;  // last key of the lane's row
  const int key_hi = p.causal ? (m0 + kRows < L ? m0 + kRows : L) : L;
  const int n_kblk = (key_hi + kRows - 1) / kRows;
  const float qs = p.qscale, inv_qs = 1.f / p.qscale, c0 = p.c0;
  Ring<kStride> ring(smem + wave * (kStages * kChunk), lane);
  const uint32_t rl = row_lane_of(lq, lh), cl = col_lane_of(lq, lh);
  auto src_k = [&](int blk, int s, int st) {
    if (s == 0) ring.rows(blk * kRows, L);
    ring.issue_rows(kg, s, st);
  };
  OwnRow<T, NC> qf;
  // scores of a block plus `init`, -inf on the keys the row may not see, and the largest of the lane's (kTop)
  auto scores = [&](auto kTop, int blk, float init, float& top, auto&& next) -> f32x16 {
    f32x16 acc, small, main;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      acc[i] = init;
      small[i] = 0.f;
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) dot_chunk<T>(acc, small, next(c), rl, qf, c);
    main = acc;
    if constexpr (!k16)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] += small[i];
    const int k0 = blk * kRows;
    if (k0 + kRows > L || (p.causal && k0 + kRows - 1 > m0)) {
      const int jb = k0 + 4 * lh;
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] = jb + 8 * (i >> 2) + (i & 3) <= lim ? acc[i] : -INFINITY;
    }
    if constexpr (kTop) {
      top = acc[0];
#pragma unroll
      for (int i = 1; i < 16; ++i) top = k16 ? fmaxf(top, acc[i]) : __builtin_elementwise_maximum(top, acc[i]);
      // An infinite operand's other parts are NaN, and so are its small products: beside an infinite sum they have no say, or a row with a score of +inf
      // (tau = +inf, output and gradients 0) would lose that key.  (Scores of -inf and NaN drop out of every comparison alike.)  The maximum that is
      // wanted anyway shows NaN (v_maximum3_f32 hands it on); a maximum of the main sums for it, in front of the small ones, cost us, forward: 2 x 8
      // heads, N = 1500 and 375, D = 64: 50.4 against 49.9; of spread 3 34.9, 34.4; alpha = 1.333, 8 x 16 heads, N = 1024: 900, 892 (no test at all: 49.2, 33.9, 884).
      if constexpr (!k16) {
        if (__builtin_amdgcn_ballot_w64(top != top) != 0ull) {
          top = -INFINITY;
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            acc[i] = acc[i] != acc[i] && main[i] == INFINITY ? INFINITY : acc[i];
            top = fmaxf(top, acc[i]);
          }
        }
      }
    }
    return acc;
  };

  // ---- the walk that lists: rows are solved on the lists after 1, 2, 4, ... steps of four blocks and behind the last ----
  if (tid == 0) over_flag = 0u;
  if (tid < kRows) t_lds[tid] = est_lds[tid] = -INFINITY;
  float t_raw = -INFINITY;  // bound of the lane's row, raw score units
  int n_mine = 0;           // entries of this lane: lh = 0 fills the wave's slots of the row from the front, lh = 1 from the back
  bool over = false;
  const int n_steps = (n_kblk + kWaves - 1) / kWaves;
  float* const my_s = list_s + wave * (kCap * kRows) + lq;
  uint16_t* const my_k = list_k + wave * (kCap * kRows) + lq;
  auto slot_of = [&](int e) -> int { return (lh ? kCap - 1 - e : e) * kRows; };
  // solver's view: eight lanes per row, wave w has rows 8 w .. 8 w + 7
  const int srow = wave * 8 + (lane >> 3), sj = lane & 7;
  float sv[16];  // the lane's share of the row's listed scores, relative to their maximum, in z units: kK per wave
  uint32_t sslot[16];
  float s_max = 0.f, s_tau = 0.f, s_members = 0.f;  // s_members: entries above the bound, where a wave has more than 8 of any of the rows
  // kK: the lane's entries per wave's list, enough for the longest of the eight rows' lists
  auto solve_k = [&](auto kc, bool last) {
    constexpr int kK = decltype(kc)::value;
    float x[4 * kK];
    s_max = -INFINITY;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const int n0 = n_lds[w][0][srow], n1 = n_lds[w][1][srow];
#pragma unroll
      for (int k = 0; k < kK; ++k) {
        const int e = sj + 8 * k;  // the wave's entries of the row, those from the front first
        const bool ok = e < n0 + n1;
        const uint32_t at = (uint32_t)(w * (kCap * kRows) + (e < n0 ? e : kCap - 1 - (e - n0)) * kRows + srow);
        sslot[w * kK + k] = ok ? at : (uint32_t)srow;
        const float v = list_s[sslot[w * kK + k]];
        x[w * kK + k] = ok ? v : -INFINITY;
        s_max = fmaxf(s_max, x[w * kK + k]);
      }
    }
    s_max = max8(s_max);
    const float m = s_max > -INFINITY ? s_max : 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) sv[i] = i < 4 * kK ? (x[i < 4 * kK ? i : 0] - m) * qs : -INFINITY;
    // from the bound the row has already; on the way a few steps do, each of which ends on a bound
    s_tau = fmaxf(-1.f, (t_lds[srow] - m) * qs);
    bool go = s_max > -INFINITY;
    const int most = last ? 40 : 4;
    for (int it = 0; it < most && __builtin_amdgcn_ballot_w64(go) != 0ull; ++it) {
      float s0 = 0.f, s1 = 0.f;
#pragma unroll
      for (int i = 0; i < 4 * kK; ++i) {
        float e0, e1;
        powers<AM>(fmaxf(sv[i] - s_tau, 0.f), c0, e0, e1);
        s0 += e0;
        s1 += e1;
      }
      s0 = sum8(s0);
      s1 = sum8(s1);
      const float step = norm_step<AM>(s0, s1, c0);
      if (go) s_tau = fminf(s_tau + step, 0.f);
      go = go && step > (last ? 1e-7f : 1e-3f);
    }
    s_members = 0.f;
    if constexpr (kK > 1) {
      if (!last) {
#pragma unroll
        for (int i = 0; i < 4 * kK; ++i) s_members += sv[i] > s_tau ? 1.f : 0.f;
        s_members = sum8(s_members);
      }
    }
  };
  auto solve = [&](bool last) {
    int most = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const int n = n_lds[w][0][srow] + n_lds[w][1][srow];
      most = n > most ? n : most;
    }
    if (__builtin_amdgcn_ballot_w64(most > 16) != 0ull) solve_k(std::integral_constant<int, 4>{}, last);
    else if (__builtin_amdgcn_ballot_w64(most > 8) != 0ull) solve_k(std::integral_constant<int, 2>{}, last);
    else solve_k(std::integral_constant<int, 1>{}, last);
  };
  bool fallback = false;
  {
    int step_no = 0, next_sync = 1;
    // solves the rows on the lists and keeps what is above the new bound; true when the workgroup gives its lists up
    auto sync = [&]() -> bool {
      n_lds[wave][lh][lq] = (uint8_t)n_mine;
      if (over) over_flag = 1u;
      __syncthreads();
      solve(step_no == n_steps);
      int nearer = 0;
      if (step_no < n_steps && __builtin_amdgcn_ballot_w64(s_members > 28.f) != 0ull) {
        const auto any_above = [&](float m) -> int { return __builtin_amdgcn_ballot_w64(s_members > m) != 0ull ? 1 : 0; };
        // (beyond 90 a list overflows anyway)
        nearer = any_above(90.f) ? 0 : any_above(step_no <= 2 ? 48.f : 28.f) + any_above(step_no <= 2 ? 56.f : 40.f) + any_above(56.f);
        // A list has overflowed, or more than half of the first 128 keys are in a row's support so far and it is about to.  The
        // threshold of a row whose other keys are like these is where the walks then start (a Newton step from beyond tau ends
        // below it).
        if (step_no == 1 ? any_above(64.f) != 0 : (over_flag != 0u && step_no > 2)) {
          const int row = m0 + srow, keys = p.causal ? (row < L - 1 ? row + 1 : L) : L, seen = step_no * (kWaves * kRows);
          const float ratio = (float)keys / (float)seen;
          float e = s_tau;
          for (int it = 0; it < 6; ++it) {
            float s0 = 0.f, s1 = 0.f;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              float e0, e1;
              powers<AM>(fmaxf(sv[i] - e, 0.f), c0, e0, e1);
              s0 += e0;
              s1 += e1;
            }
            s0 = sum8(s0) * ratio;
            s1 = sum8(s1) * ratio;
            const float step = norm_step<AM>(s0, s1, c0);
            if (s0 > 0.f && s1 > 0.f) e += step;
          }
          if (sj == 0 && keys > seen && e < 0.f && e > s_tau) est_lds[srow] = s_max + e * inv_qs;
        }
      }
      if (lane == 0) sync_lds[wave] = (uint32_t)nearer;
      if (sj == 0) {
        // (the margin covers the rounding of the difference and of the product back to raw units)
        t_lds[srow] = s_max > -INFINITY ? (s_max + (s_tau - 1e-6f) * inv_qs) - 4e-7f * fabsf(s_max) : -INFINITY;
      }
      const bool given_up = over_flag != 0u;  // (read in front of the barrier: behind it a faster wave may set it again)
      __syncthreads();
      t_raw = fmaxf(t_raw, t_lds[lq]);
      return given_up;
    };
    // where a wave's list of a row is more than half full, or about to overflow; entries below the bound do no harm otherwise
    auto compact = [&](int more_than) {
      if (__builtin_amdgcn_ballot_w64(n_mine + __shfl_xor(n_mine, 32, 64) > more_than) == 0ull) return;
      int kept = 0;
      for (int e0 = 0; __builtin_amdgcn_ballot_w64(e0 < n_mine) != 0ull; e0 += 8) {
        float s[8];
        uint16_t k[8];
#pragma unroll
        for (int x = 0; x < 8; ++x) {
          s[x] = my_s[slot_of(e0 + x < kCap ? e0 + x : 0)];
          k[x] = my_k[slot_of(e0 + x < kCap ? e0 + x : 0)];
        }
#pragma unroll
        for (int x = 0; x < 8; ++x) {
          if (e0 + x < n_mine && s[x] > t_raw) {
            my_s[slot_of(kept)] = s[x];
            my_k[slot_of(kept)] = k[x];
            ++kept;
          }
        }
      }
      n_mine = kept;
    };
    __syncthreads();  // over_flag is clear
    // (as walk() does it, with the loads of the coming step under way across a solve)
    auto list_block = [&](int blk, auto&& next) {
      float bm;
      const f32x16 s = scores(std::true_type{}, blk, 0.f, bm, next);
      if (over || __builtin_amdgcn_ballot_w64(live && bm > t_raw) == 0ull) return;
      int c = 0;
#pragma unroll
      for (int i = 0; i < 16; ++i) c += s[i] > t_raw ? 1 : 0;
      c = live ? c : 0;
      auto too_many = [&]() -> bool {
        const int need = n_mine + c;
        return __builtin_amdgcn_ballot_w64(need + __shfl_xor(need, 32, 64) > kCap) != 0ull;
      };
      if (too_many()) {
        compact(0);  // (up to half a list may lie below the bound)
        if (too_many()) {
          over = true;  // uniform over the wave
          return;
        }
      }
      const int jb = blk * kRows + 4 * lh;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        if (live && s[i] > t_raw) {
          my_s[slot_of(n_mine)] = s[i];
          my_k[slot_of(n_mine)] = (uint16_t)(jb + 8 * (i >> 2) + (i & 3));
          ++n_mine;
        }
      }
    };
    if (wave < n_kblk) start<NC>(wave, n_kblk, kWaves, src_k);
    qf.load(reinterpret_cast<const unsigned char*>(p.q) + (q_row0 + (live ? qi : L - 1)) * kStride, lh);
    while (true) {
      const int blk = step_no * kWaves + wave;
      if (blk < n_kblk) list_block(blk, [&](int s) -> uint32_t { return take<NC>(ring, blk, s, n_kblk, kWaves, src_k); });
      ++step_no;
      if (step_no == n_steps) ring.drain();  // (the output takes the ring's place behind the solve)
      if (step_no == next_sync || step_no == n_steps) {
        if (sync()) {
          fallback = true;
          break;
        }
        if (step_no == n_steps) break;
        compact(kCap / 2);
        // Between two solves about as many scores join a list as it has members; where a row has so many that it would overflow now
        // and then, the next solve comes sooner.  (sync_lds is written behind the next solve's first barrier at the earliest.)
        const uint32_t nearer = __builtin_elementwise_max(__builtin_elementwise_max(sync_lds[0], sync_lds[1]), __builtin_elementwise_max(sync_lds[2], sync_lds[3]));
        const int gap = step_no >> nearer;
        next_sync = step_no + (gap > 0 ? gap : 1);
      }
    }
    ring.drain();
  }

  if (!fallback) {
    // ---- output from the lists: the solver's lanes hold the row's scores; members to a dense list in the idle ring ----
    float pr[16];
    float psum = 0.f;
    int members = 0;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float e1;
      powers<AM>(fmaxf(sv[i] - s_tau, 0.f), c0, pr[i], e1);
      psum += pr[i];
      members += pr[i] > 0.f ? 1 : 0;
    }
    psum = sum8(psum);
    const float inv = psum > 0.f ? 1.f / psum : 0.f;
    int before = 0, total = members;
#pragma unroll
    for (int d = 1; d < 8; d <<= 1) {
      const int o = __shfl_xor(total, d, 64);
      if (sj & d) before += o;
      total += o;
    }
    float* const mem_p = reinterpret_cast<float*>(smem) + srow * 128;
    uint32_t* const mem_k = reinterpret_cast<uint32_t*>(smem) + kRows * 128 + srow * 128;
    uint32_t bits_done = 0xffffffffu;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      if (pr[i] > 0.f) {
        const uint32_t key = list_k[sslot[i]];
        mem_p[before] = pr[i];
        mem_k[before] = key;
        ++before;
        if (p.bmask && (key >> 6) != bits_done) {
          bits_done = key >> 6;
          atomicOr(reinterpret_cast<uint32_t*>(p.bmask) + ((size_t)(b * p.Hq + h) * p.n_mblk + m0 / kMaskRows) * p.mask_words + (bits_done >> 5),
                   1u << (bits_done & 31));
        }
      }
    }
    // (a row's eight lanes belong to one wave, whose LDS accesses stay in order)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    const int row = m0 + srow;
    if (p.taus && sj == 0 && row < L) p.taus[q_row0 + row] = fmaf(s_max, qs, s_tau);
    constexpr int kPer = k16 ? 8 : 4;  // values per 16-byte piece; a lane has piece sj + 8 c of its row
    float acc[NC][kPer];
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int k = 0; k < kPer; ++k) acc[c][k] = 0.f;
    const u32x4* v4 = reinterpret_cast<const u32x4*>(vg);
    constexpr int kRowsAhead = NC <= 2 ? 8 : 4;  // rows of V under way
    for (int e = 0; __builtin_amdgcn_ballot_w64(e < total) != 0ull; e += kRowsAhead) {
      u32x4 r[kRowsAhead][NC];
      float w[kRowsAhead];
#pragma unroll
      for (int x = 0; x < kRowsAhead; ++x) {
        const bool ok = e + x < total;
        w[x] = ok ? mem_p[e + x] : 0.f;
        const uint32_t key = ok ? mem_k[e + x] : mem_k[0];
        const u32x4* vr = v4 + (size_t)(total > 0 ? key : 0u) * (kStride / 16) + sj;
#pragma unroll
        for (int c = 0; c < NC; ++c) r[x][c] = vr[8 * c];
      }
#pragma unroll
      for (int x = 0; x < kRowsAhead; ++x)
        if (e + x < total)
#pragma unroll
          for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              const uint32_t word = r[x][c][k];
              if constexpr (k16) {
                acc[c][2 * k] = fmaf(w[x], unpack_lo<T>(word), acc[c][2 * k]);
                acc[c][2 * k + 1] = fmaf(w[x], unpack_hi<T>(word), acc[c][2 * k + 1]);
              } else {
                acc[c][k] = fmaf(w[x], __builtin_bit_cast(float, word), acc[c][k]);
              }
            }
    }
    if (row < N) {
      u32x4* o4 = reinterpret_cast<u32x4*>(out + (size_t)row * kStride) + sj;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        u32x4 w;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          if constexpr (k16) w[k] = pack2<T>(acc[c][2 * k] * inv, acc[c][2 * k + 1] * inv);
          else w[k] = __builtin_bit_cast(uint32_t, acc[c][k] * inv);
        }
        o4[8 * c] = w;
      }
    }
    return;
  }

  // ---- walks: t_raw is finite for live rows (every row sees key 0, which the first solve has), a lower bound of tau; the
  // estimate may lie beyond it ----
  float t = live && t_raw > -INFINITY ? fmaxf(t_raw, est_lds[lq]) : 0.f;
  for (int it = 0; it < 24; ++it) {
    float a0 = 0.f, a1 = 0.f, mx = -INFINITY;
    walk<NC>(ring, wave, n_kblk, kWaves, src_k, [&](int blk, auto&& next) {
      float bm;
      const f32x16 s = scores(std::true_type{}, blk, -t, bm, next);
      mx = fmaxf(mx, bm);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        float e0, e1;
        powers<AM>(fmaxf(s[i], 0.f) * qs, c0, e0, e1);
        a0 += e0;
        a1 += e1;
      }
    });
    a0 += __shfl_xor(a0, 32, 64);
    a1 += __shfl_xor(a1, 32, 64);
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    float(*rd)[3][kRows] = red[it & 1];
    if (lh == 0) {
      rd[wave][0][lq] = a0;
      rd[wave][1][lq] = a1;
      rd[wave][2][lq] = mx;
    }
    __syncthreads();
    a0 = (rd[0][0][lq] + rd[1][0][lq]) + (rd[2][0][lq] + rd[3][0][lq]);
    a1 = (rd[0][1][lq] + rd[1][1][lq]) + (rd[2][1][lq] + rd[3][1][lq]);
    mx = fmaxf(fmaxf(rd[0][2][lq], rd[1][2][lq]), fmaxf(rd[2][2][lq], rd[3][2][lq]));
    // never below the row maximum less 1, where the sums of a score far above the bound would also leave fp32
    float step = mx * qs - 1.f;
    if (a0 > 0.f && a0 < 1e30f && a1 > 0.f && a1 < 1e30f) step = fmaxf(step, norm_step<AM>(a0, a1, c0));
    if (live) t += step * inv_qs;
    if (__builtin_amdgcn_ballot_w64(live && fabsf(step) > 2e-5f) == 0ull) break;  // (the same sums in every wave)
  }
  if (live && lh == 0 && wave == 0 && p.taus) p.taus[q_row0 + qi] = t * qs;

  f32x16 o[NC][k16 ? 2 : 1];  // per chunk of V, 32 columns each
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int d = 0; d < (k16 ? 2 : 1); ++d)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[c][d][i] = 0.f;
  float psum = 0.f;
  auto src_kv = [&](int blk, int s, int st) {
    if (s < NC) ring.issue(kg, blk * kRows, L, s, st);
    else if constexpr (k16) ring.issue_t(vg, blk * kRows, L, s - NC, st);
    else ring.issue(vg, blk * kRows, L, s - NC, st);
  };
  walk<2 * NC>(ring, wave, n_kblk, kWaves, src_kv, [&](int blk, auto&& next) {
    float unused;
    const f32x16 s = scores(std::false_type{}, blk, -t, unused, next);  // (a row with a score of +inf has no finite t, and no weights)
    float w[16];
    float bs = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float e1;
      powers<AM>(live ? fmaxf(s[i], 0.f) * qs : 0.f, c0, w[i], e1);
      if constexpr (k16) w[i] = unpack_lo<T>(pack2<T>(w[i], 0.f));  // what the product weighs V with
      bs += w[i];
    }
    psum += bs;
    const bool any = __builtin_amdgcn_ballot_w64(bs > 0.f) != 0ull;
    if (any && p.bmask && lane == 0)
      atomicOr(reinterpret_cast<uint32_t*>(p.bmask) + ((size_t)(b * p.Hq + h) * p.n_mblk + m0 / kMaskRows) * p.mask_words + (blk >> 6),
               1u << ((blk >> 1) & 31));
    Split ws[1][2];
    if constexpr (!k16) split16(w, ws[0]);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const uint32_t a = next(NC + c);
      if constexpr (k16) {
        if (any) acc_chunk_16<T>(o[c], a, lane, w);
      } else {
        f32x16* const to[1] = {&o[c][0]};
        if (any) acc_chunk<false, true>(to, a, cl, ws);
      }
    }
  });
  psum += __shfl_xor(psum, 32, 64);
  __syncthreads();  // the sums of the last step have been read, every wave is done with its ring
  if (lh == 0) red[0][wave][0][lq] = psum;
  combine_store<D>(reinterpret_cast<const f32x16(&)[D / 32]>(o), smem, reinterpret_cast<T*>(out), m0, N, wave, lane, [&](int row) {
    const float z = (red[0][0][0][row] + red[0][1][0][row]) + (red[0][2][0][row] + red[0][3][0][row]);
    return z > 0.f ? 1.f / z : 0.f;
  });
}

// ---------------------------------------------------------------------------------------------------------
// dQ: one walk for sum p, sum u, sum u dP and the products of u (dP - c) and u with K
// ---------------------------------------------------------------------------------------------------------
// x of a row's two lanes, added up
__device__ __forceinline__ float both_lanes(float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return __builtin_bit_cast(float, r[0]) + __builtin_bit_cast(float, r[1]);
}
// u x, 0 where u is 0, whatever x is (one instruction; the intrinsic has no builtin)
__device__ float mul_legacy(float u, float x) __asm("llvm.amdgcn.fmul.legacy");
__device__ __forceinline__ float times(float u, float x) { return mul_legacy(u, x); }

template <int D> constexpr int bwd_smem() { return kRing > kWaves * kRows * D * 4 ? kRing : kWaves * kRows * D * 4; }

template <int D, int AM>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D == 64 ? 2 : 1, D == 64 ? 2 : 1))) void attn_rows32_dq_kernel(AttnBwdParams p) {
  constexpr int kStride = D * 4;
  constexpr int NC = kStride / 128;      // chunks per block
  __shared__ __align__(4096) unsigned char smem[bwd_smem<D>()];
  __shared__ float red[kWaves][3][kRows];
  __shared__ __align__(16) unsigned char own_lds[2][OwnRowLds<NC>::kBytes];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, lq = lane & 31, lh = lane >> 5;
  const int N = p.N, group = p.Hq / p.Hkv, n_rblk = (N + kRows - 1) / kRows;
  int bkv, mi, hg, rblk;
  if (longest_first(p.varlen, p.varlen_bits, p.B, p.Hkv, N, group, p.causal != 0, 2ll * N * kStride, false, D == 64, bkv, rblk, hg)) mi = n_rblk - 1 - rblk;
  else if (!xcd_block_map(p.varlen != nullptr, p.B * p.Hkv, n_rblk, group, p.causal != 0, 2ll * N * kStride, bkv, mi, hg)) return;
  const BatchItem item = batch_item(p.varlen, p.varlen_bits, p.B, N, bkv / p.Hkv, p.Hkv, n_rblk * group, p.causal == 0, D == 64 ? 2 : 1);
  const int b = item.b, L = item.L, kvh = bkv % p.Hkv, h = kvh * group + hg;
  bkv = b * p.Hkv + kvh;
  const int m0 = (n_rblk - 1 - mi) * kRows;
  const size_t q_row0 = (size_t)(b * p.Hq + h) * N;
  unsigned char* const dq = reinterpret_cast<unsigned char*>(p.dq) + q_row0 * kStride;
  if (m0 >= L) {
    const int rows = N - m0 < kRows ? N - m0 : kRows;
    for (int i = tid; i < rows * (kStride / 16); i += 256) reinterpret_cast<f32x4*>(dq + (size_t)m0 * kStride)[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    return;
  }
  const unsigned char* kg = reinterpret_cast<const unsigned char*>(p.k) + (size_t)bkv * N * kStride;
  const unsigned char* vg = reinterpret_cast<const unsigned char*>(p.v) + (size_t)bkv * N * kStride;
  const int qi = m0 + lq;
  const bool live = qi < L;
  const int lim = p.causal ? (qi < L - 1 ? qi : L - 1) : L - 1;
  const int key_hi = p.causal ? (m0 + kRows < L ? m0 + kRows : L) : L;
  const int n_kblk = (key_hi + kRows - 1) / kRows;
  const int lim_all = p.causal ? (m0 < L - 1 ? m0 : L - 1) : L - 1;  // the smallest of the rows
  const float tau = live ? p.taus[q_row0 + qi] : INFINITY;
  Ring<kStride> ring(smem + wave * (kStages * kChunk), lane);
  const uint32_t rl = row_lane_of(lq, lh), cl = col_lane_of(lq, lh);
  // chunks of a block: K, V and K again
  auto src = [&](int blk, int s, int st) {
    if (s == 0) ring.rows(blk * kRows, L);
    ring.issue_rows(s < NC || s >= 2 * NC ? kg : vg, s % NC, st);
  };
  if (wave < n_kblk) start<3 * NC>(wave, n_kblk, kWaves, src);  // (in front of the own rows, whose split waits for their loads)
  const size_t own = (q_row0 + (live ? qi : L - 1)) * kStride;
  const OwnRowLds<NC> qf(reinterpret_cast<const unsigned char*>(p.q) + own, own_lds[0], wave, lane), dof(reinterpret_cast<const unsigned char*>(p.dout) + own, own_lds[1], wave, lane);
  __syncthreads();
  // dX = u (dP - delta) needs delta = (sum u dP) / (sum u) first; instead of a walk for it, the walk adds up u (dP - c) K and u K, of which
  // dQ = the first less (delta - c) of the second.  c is the row's delta over the wave's blocks so far, moved in front of a block that brings as much
  // u as there was when it was last moved: what is added up around one c weighs no more than the keys whose delta c is, and roundings of the size
  // of u |dP - c| stay within a small multiple of those of the terms u (dP - delta) themselves.  (With c kept from a wave's first member, whatever its weight, they
  // do not: a V row of 1000 times the norm with u = 2^-10, 300 members: relative error of dQ 5.7e-5, as here 1.2e-7; K of mean 4: 1.4e-3, 9.7e-7.)
  // The sums so far go over to the new c by o -= shift ou: at head dim 128, where they lie in accumulation registers that the vector pipe does not
  // reach, as the start of the small products' sum.  us, 4 x 16/4 heads, N = 1024, forward and backward: 735 -> 694; D = 64, 2 x 8, N = 1500 and 375: 157.6, that way 160.2.
  constexpr bool kShiftInPart = D != 64;
  float zsum = 0.f, usum = 0.f, udp = 0.f, centre = 0.f;
  float mark = 0x1p-100f;  // sum u when c was last moved (below it, it has no delta worth a division)
  f32x16 o[NC], ou[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[c][i] = ou[c][i] = 0.f;
  walk<3 * NC, true>(ring, wave, n_kblk, kWaves, src, [&](int blk, auto&& next) {
    float r[16], dx[16], u[16];
    f32x16 s, dp, small;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = dp[i] = small[i] = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c) dot_chunk<float>(s, small, next(c), rl, qf, c);
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      r[i] = fmaf(s[i] + small[i], p.qscale, -tau);  // z - tau
      small[i] = 0.f;
    }
    if (blk * kRows + kRows - 1 > lim_all) {
      const int jb = blk * kRows + 4 * lh;
#pragma unroll
      for (int i = 0; i < 16; ++i) r[i] = jb + 8 * (i >> 2) + (i & 3) <= lim ? r[i] : -INFINITY;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) mx = fmaxf(mx, r[i]);
    if (__builtin_amdgcn_ballot_w64(mx > 0.f) == 0ull) {  // no row of the block has a member
#pragma unroll
      for (int c = NC; c < 3 * NC; ++c) next(c);
      return;
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) dot_chunk<float>(dp, small, next(NC + c), rl, dof, c);
    float bu = 0.f, shift = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float pr;
      bwd_prob<AM>(r[i], p.c0, pr, u[i]);
      zsum += pr;
      bu += u[i];
      dp[i] += small[i];
    }
    const float us = both_lanes(usum + bu);
    const bool moves = us >= 2.f * mark;
    if (__builtin_amdgcn_ballot_w64(moves) != 0ull) {
      float bd = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) bd += times(u[i], dp[i] - centre);
      const float ud = both_lanes(udp + bd);
      shift = moves ? ud * fast_rcp(us) : 0.f;
      mark = moves ? us : mark;
      centre += shift;
      udp = fmaf(-shift, usum, udp);
    }
    float bd = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      dx[i] = times(u[i], dp[i] - centre);
      bd += dx[i];
    }
    usum += bu;
    udp += bd;
    if constexpr (!kShiftInPart) {
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[c][i] = fmaf(-shift, ou[c][i], o[c][i]);
    }
    // (alpha = 2: what follows, taken up among the weights, had 23 registers spilled instead of 16.  us, forward and backward, 6 x 8 heads, N <= 600, D = 64: 130.5 ->
    // 127.5; at the other alphas the parts of one block among the weights of it are the faster way: 2 x 8 heads, N = 1500 and 375: 162.2 against 164.7.)
    if constexpr (AM == ATT_2) __builtin_amdgcn_sched_barrier(0);
    Split w[2][2];
    split16(dx, w[0]);
    split16(u, w[1]);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      f32x16* const to[2] = {&o[c], &ou[c]};
      acc_chunk<kShiftInPart>(to, next(2 * NC + c), cl, w, shift);
    }
  });
  zsum += __shfl_xor(zsum, 32, 64);
  usum += __shfl_xor(usum, 32, 64);
  udp += __shfl_xor(udp, 32, 64);
  if (lh == 0) {
    red[wave][0][lq] = zsum;
    red[wave][1][lq] = usum;
    red[wave][2][lq] = fmaf(centre, usum, udp);
  }
  __syncthreads();  // (every wave is done with its ring, too)
  auto all = [&](int k) { return (red[0][k][lq] + red[1][k][lq]) + (red[2][k][lq] + red[3][k][lq]); };
  zsum = all(0);
  usum = all(1);
  const float delta = usum > 0.f ? all(2) / usum : 0.f;
  if (live && wave == 0 && lh == 0) {
    p.delta[q_row0 + qi] = delta;
    p.zinv[q_row0 + qi] = zsum > 0.f ? 1.f / zsum : 0.f;
  }
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[c][i] = fmaf(centre - delta, ou[c][i], o[c][i]);
  const float sm = p.sm_scale;
  combine_store<D>(o, smem, reinterpret_cast<float*>(dq), m0, N, wave, lane,
                   [&](int) { return sm; });
}

// ---------------------------------------------------------------------------------------------------------
// dK, dV: one walk over the (query block, query head) pairs of a K/V head, dV^T += dO^T P and dK^T += Q^T dX
// ---------------------------------------------------------------------------------------------------------
template <int D, int AM>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D == 64 ? 2 : 1, D == 64 ? 2 : 1))) void attn_rows32_dkdv_kernel(AttnBwdParams p) {
  constexpr int kStride = D * 4;
  constexpr int NC = kStride / 128;      // chunks per block
  __shared__ __align__(4096) unsigned char smem[bwd_smem<D>()];
  __shared__ __align__(256) float scal[kWaves][4 * kRows];  // of the wave's block: tau, 1 / sum p, delta (and delta once more)
  __shared__ __align__(16) unsigned char own_lds[2][OwnRowLds<NC>::kBytes];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, lq = lane & 31, lh = lane >> 5;
  const int N = p.N, group = p.Hq / p.Hkv, n_rblk = (N + kRows - 1) / kRows;
  int bkv, kblk, member_unused;
  if (!longest_first(p.varlen, p.varlen_bits, p.B, p.Hkv, N, 1, p.causal != 0, 2ll * group * N * kStride, true, D == 64, bkv, kblk, member_unused) &&
      !xcd_block_map(p.varlen != nullptr, p.B * p.Hkv, n_rblk, 1, p.causal != 0, 2ll * group * N * kStride, bkv, kblk, member_unused)) return;
  const BatchItem item = batch_item(p.varlen, p.varlen_bits, p.B, N, bkv / p.Hkv, p.Hkv, n_rblk, p.causal == 0, D == 64 ? 2 : 1);
  const int b = item.b, L = item.L, kvh = bkv % p.Hkv;
  bkv = b * p.Hkv + kvh;
  const int n0 = kblk * kRows;
  const size_t kv_row0 = (size_t)bkv * N;
  unsigned char* const dk = reinterpret_cast<unsigned char*>(p.dk) + kv_row0 * kStride;
  unsigned char* const dv = reinterpret_cast<unsigned char*>(p.dv) + kv_row0 * kStride;
  if (n0 >= L) {
    const int rows = N - n0 < kRows ? N - n0 : kRows;
    for (int i = tid; i < rows * (kStride / 16); i += 256) {
      reinterpret_cast<f32x4*>(dk + (size_t)n0 * kStride)[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      reinterpret_cast<f32x4*>(dv + (size_t)n0 * kStride)[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    return;
  }
  const int kj = n0 + lq;
  const bool live = kj < L;
  const int q_first = p.causal ? kblk : 0;            // first query block that sees the keys
  const int n_q = (L + kRows - 1) / kRows - q_first;  // query blocks per head
  const size_t q_head0 = (size_t)(b * p.Hq + kvh * group) * N;
  Ring<kStride> ring(smem + wave * (kStages * kChunk), lane);
  const uint32_t rl = row_lane_of(lq, lh), cl = col_lane_of(lq, lh);
  // item x = head * n_q + query block - q_first; its chunks: Q, dO, dO and Q again
  auto src = [&](int x, int s, int st) {
    const int g = x / n_q, qb = q_first + (x - g * n_q);
    const unsigned char* base = reinterpret_cast<const unsigned char*>(s < NC || s >= 3 * NC ? p.q : p.dout) + (q_head0 + (size_t)g * N) * kStride;
    if (s == 0) {  // tau and 1 / sum p (half a wave each) and delta of its queries, in front of the block's first chunk
      int row = qb * kRows + (lane & 31);
      row = row < L ? row : L - 1;
      const size_t at = q_head0 + (size_t)g * N + row;
      dma4((lane < 32 ? p.taus : p.zinv) + at, &scal[wave][0]);
      dma4(p.delta + at, &scal[wave][64]);
    }
    if (s == 0) ring.rows(qb * kRows, L);
    ring.issue_rows(base, s % NC, st);
  };
  if (wave < n_q * group) start<4 * NC>(wave, n_q * group, kWaves, src);
  const size_t own = (kv_row0 + (live ? kj : L - 1)) * kStride;
  const OwnRowLds<NC> kf(reinterpret_cast<const unsigned char*>(p.k) + own, own_lds[0], wave, lane), vf(reinterpret_cast<const unsigned char*>(p.v) + own, own_lds[1], wave, lane);
  __syncthreads();
  f32x16 ov[NC], ok[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int i = 0; i < 16; ++i) ov[c][i] = ok[c][i] = 0.f;
  walk<4 * NC, true>(ring, wave, n_q * group, kWaves, src, [&](int x, auto&& next) {
    const int g = x / n_q, q0 = (q_first + (x - g * n_q)) * kRows;
    f32x16 s, dp, small;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = dp[i] = small[i] = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c) dot_chunk<float>(s, small, next(c), rl, kf, c);
    // tau, 1 / sum p and delta of the lane's sixteen queries: they came in front of the block's first chunk
    auto scalars = [&](int which, float (&y)[16]) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const f32x4 v4 = *reinterpret_cast<const f32x4*>(&scal[wave][which * kRows + 8 * i + 4 * lh]);
#pragma unroll
        for (int e = 0; e < 4; ++e) y[4 * i + e] = v4[e];
      }
    };
    float tau[16], zi[16], de[16];
    scalars(0, tau);
    scalars(1, zi);
    scalars(2, de);
    float r[16], w[16], dx[16];
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      r[i] = fmaf(s[i] + small[i], p.qscale, -tau[i]);
      small[i] = 0.f;
    }
    if (q0 + kRows > L || n0 + kRows > L || (p.causal && n0 + kRows - 1 > q0)) {  // not every query of the block sees every key
      const int first = live ? (p.causal ? kj : 0) : L;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int qrow = q0 + 8 * (i >> 2) + 4 * lh + (i & 3);
        r[i] = (int)(qrow >= first) & (int)(qrow < L) ? r[i] : -INFINITY;
      }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) mx = fmaxf(mx, r[i]);
    if (__builtin_amdgcn_ballot_w64(mx > 0.f) == 0ull) {
#pragma unroll
      for (int c = NC; c < 4 * NC; ++c) next(c);
      return;
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) dot_chunk<float>(dp, small, next(NC + c), rl, vf, c);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float pr, u;
      bwd_prob<AM>(r[i], p.c0, pr, u);
      w[i] = times(pr, zi[i]);
      dx[i] = times(u, dp[i] + small[i] - de[i]);
    }
    Split ws[1][2];
    split16(w, ws[0]);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      f32x16* const to[1] = {&ov[c]};
      acc_chunk(to, next(2 * NC + c), cl, ws);
    }
    split16(dx, ws[0]);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      f32x16* const to[1] = {&ok[c]};
      acc_chunk(to, next(3 * NC + c), cl, ws);
    }
  });
  __syncthreads();  // every wave is done with its ring
  combine_store<D>(ov, smem, reinterpret_cast<float*>(dv), n0, N, wave, lane, [](int) { return 1.f; });
  __syncthreads();
  const float sm = p.sm_scale;
  combine_store<D>(ok, smem, reinterpret_cast<float*>(dk), n0, N, wave, lane, [&](int) { return sm; });
}

}  // namespace f32path
}  // namespace adsp
