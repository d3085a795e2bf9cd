// Tiles in LDS and products on them, for the kernels of the 16-bit types that visit all pairs of a row (attn_fwd16_kernel.h,
// attn_bwd16_kernel.h): head dims 64 and 128.
#pragma once
#include "attn_f32_kernel.h"

namespace adsp {
namespace tile16 {

// What the kernels on the supports left over: all blocks, those with a flag, or (the usual case) none.  Both counters are asked for at
// once and in front of everything else: a launch with nothing to do costs its workgroups one trip to memory.
struct LeftOver {
  const int32_t* flags;
  uint32_t all, some;
  __device__ __forceinline__ LeftOver(const int32_t* f, const uint32_t* queue) : flags(f), all(1u), some(0u) {
    if (f) {
      all = queue[kCtrlAllDense];
      some = queue[kCtrlFlagged];
    }
  }
  __device__ __forceinline__ bool none() const { return (all | some) == 0u; }
  __device__ __forceinline__ bool takes(size_t block) const { return all != 0u || (some != 0u && flags[block] != 0); }
};

// adds u^c0 and u^(c0 - 1)
template <int AM> __device__ __forceinline__ void add_powers(float u, float c0, float& s0, float& s1) {
  if constexpr (AM == ATT_15) {
    s0 = fmaf(u, u, s0);
    s1 += u;
  } else if constexpr (AM == ATT_2) {
    s0 += u;
    s1 += __builtin_amdgcn_fmed3f(u * 3e38f, 0.f, 1.f);
  } else {
    const float e1 = fast_exp2(fast_log2(u) * (c0 - 1.f));  // (0 at 0)
    s0 = fmaf(e1, u, s0);
    s1 += e1;
  }
}

// Tiles of kTR rows of a row-major [N][D] tensor, 16-byte pieces swizzled so that one copy serves both ways of reading: whole
// rows (16 consecutive rows at one piece fall into 16 different places) and the transposing reads (four consecutive rows at four
// neighbouring pieces likewise).  The swizzle has a period of 16 rows.
template <typename T, int D, int TR = 128> struct Tile {
  static constexpr int kRow = D * 2, kC = kRow / 16;
  static constexpr int kTR = TR;
  static constexpr int kBytes = kTR * kRow;
  static constexpr int kLoads = kBytes / 4096;  // 1 KB loads per wave
  static constexpr int kDB = D / 32, kKS = D / 16;
  static constexpr int kG = D / 64;  // groups of four operands in a product over the columns of 32 rows, and over 32 rows for all columns
  static __device__ __forceinline__ int sw(int row) {
    if constexpr (kC == 8) return ((row >> 1) & 1) << 2 | ((row >> 2) & 1) << 1 | ((row >> 3) & 1);
    else return (row & 3) << 2 | ((row >> 2) & 3);
  }
  uint32_t off;  // the lane's place in a tile: for the loads,
  uint32_t rd[kKS], tr[2][kDB];  // for the row reads, the transposing reads
  // lds: LDS address of the tile that is read first (the tiles of a stage lie kBytes apart, read offsets are immediate)
  __device__ __forceinline__ Tile(uint32_t lds, int wave, int lane) {
    const int pos = wave * 64 + lane, row = pos / kC;
    off = (uint32_t)(row * kRow + (((pos % kC) ^ sw(row)) << 4));
    const int lq = lane & 31, lh = lane >> 5;
#pragma unroll
    for (int k = 0; k < kKS; ++k) rd[k] = lds + (uint32_t)(lq * kRow + (((2 * k + lh) ^ sw(lq)) << 4));
    const int a4 = lane & 15, grp = lane >> 4, r = a4 >> 2, c = a4 & 3, dl = grp & 1;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int x = 4 * (grp >> 1) + r + 8 * h;
#pragma unroll
      for (int db = 0; db < kDB; ++db) tr[h][db] = lds + (uint32_t)(x * kRow + (((4 * db + 2 * dl + (c >> 1)) ^ sw(x)) << 4) + (c & 1) * 8);
    }
  }
  // rows [row0, row0 + kTR) into LDS at `lds`; rows from `limit` on are replaced by the last one in front of it
  __device__ __forceinline__ void issue(const unsigned char* g, int row0, int limit, unsigned char* lds, int wave, int lane) const {
    if (row0 + kTR <= limit) {
      const unsigned char* base = uniform_ptr(g + (size_t)row0 * kRow);
#pragma unroll
      for (int j = 0; j < kLoads; ++j) dma16s(base + j * 4096, off, lds + (j * 4 + wave) * 1024);
    } else {
      const unsigned char* base = uniform_ptr(g);
#pragma unroll
      for (int j = 0; j < kLoads; ++j) {
        const int pos = (j * 4 + wave) * 64 + lane, row = pos / kC;
        int r = row0 + row;
        r = r < limit ? r : limit - 1;
        dma16s(base, (uint32_t)r * (uint32_t)kRow + (uint32_t)(((pos % kC) ^ sw(row)) << 4), lds + (j * 4 + wave) * 1024);
      }
    }
  }
  // the same for kTR / 32 blocks of 32 rows that lie anywhere: row_of(r): the tensor's row that becomes row r
  template <typename Row> __device__ __forceinline__ void issue_blocks(const unsigned char* g, Row&& row_of, unsigned char* lds, int wave, int lane) const {
    const unsigned char* base = uniform_ptr(g);
#pragma unroll
    for (int j = 0; j < kLoads; ++j) {
      const int pos = (j * 4 + wave) * 64 + lane, row = pos / kC;
      dma16s(base, (uint32_t)row_of(row) * (uint32_t)kRow + (uint32_t)(((pos % kC) ^ sw(row)) << 4), lds + (j * 4 + wave) * 1024);
    }
  }
  // the reads go on `by` bytes further
  __device__ __forceinline__ void move(uint32_t by) {
#pragma unroll
    for (int k = 0; k < kKS; ++k) {
      rd[k] += by;
      asm volatile("" : "+v"(rd[k]));  // (one addition a tile, not one a read)
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int db = 0; db < kDB; ++db) {
        tr[h][db] += by;
        asm volatile("" : "+v"(tr[h][db]));
      }
  }
  // four operands: row 32 blk + lane of tile `t` of the stage at columns 64 g .. (a product over the columns)
  __device__ __forceinline__ void rows(int t, int blk, int g, u32x4 (&a)[4]) const {
#pragma unroll
    for (int k = 0; k < 4; ++k) a[k] = lds_read16(rd[4 * g + k], t * kBytes + blk * 32 * kRow);
  }
  // four operands that run along the rows of block blk: number 4 g + k is rows 16 s .., columns 32 db .. with s = n / kDB, db = n % kDB
  __device__ __forceinline__ void columns(int t, int blk, int g, u32x4 (&a)[4]) const {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int n = 4 * g + k, s = n / kDB, db = n % kDB, at = t * kBytes + (blk * 32 + 16 * s) * kRow;
      const u32x2_t x0 = lds_read8_tr(tr[0][db], at), x1 = lds_read8_tr(tr[1][db], at);
      a[k] = u32x4{x0[0], x0[1], x1[0], x1[1]};
    }
  }
};
template <int D> __device__ __forceinline__ u32x4 piece(const uint32_t (&f)[D / 4], int k) { return u32x4{f[4 * k], f[4 * k + 1], f[4 * k + 2], f[4 * k + 3]}; }

// Behind the last of a row of products: the wait states that the hardware asks for in front of a vector instruction that reads
// an accumulator (11 behind a product of 8 passes).  The compiler counts them along the first path that it finds back to a
// product; where a short branch and a longer one meet again in front of the reader, that is now and then the longer one.
__device__ __forceinline__ void products_end() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_nop 15");
  __builtin_amdgcn_sched_barrier(0);
}

// Products and vector work side by side: a product keeps the matrix pipe busy for 32 cycles, in which its wave can issue vector
// instructions for another block.  NG groups of four products; load(g, a) reads a group's operands from LDS, kAhead groups
// ahead of their use; mul(g, k, a[k]) is one product, with the vector work that goes beside it.  The order is fixed by hand: the
// compiler would put the products in a row, in which the wave waits for each, and the reads right in front of them.
template <int NG, int kAhead, typename Load, typename Mul> __device__ __forceinline__ void stream(Load&& load, Mul&& mul) {
  u32x4 a[kAhead + 1][4];
#pragma unroll
  for (int g = 0; g < kAhead; ++g)
    if (g < NG) load(g, a[g]);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    if (g + kAhead < NG) load(g + kAhead, a[(g + kAhead) % (kAhead + 1)]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      mul(g, k, a[g % (kAhead + 1)][k]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  products_end();
}

// rows [row0, row0 + 32) below n of a row-major tensor = scale * o, the parts' sums added up in LDS; smem holds 4 x 32 x D floats.
// Waves rg, rg + 4 / P, ... hold the parts of the rows of wave rg.
template <typename T, int D, int P>
__device__ __forceinline__ void store_parts(const f32x16 (&o)[D / 32], float scale, unsigned char* smem, unsigned char* out, int wg_row0, int n, int wave, int lane) {
  using KS = Swz<D * 4>;
  constexpr int kRG = 4 / P, kWave = 32 * D * 4;
  const int lq = lane & 31, lh = lane >> 5, tid = wave * 64 + lane;
  unsigned char* mine = smem + wave * kWave;
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<f32x4*>(mine + KS::off(lq, db * 8 + 2 * g + lh)) =
          f32x4{o[db][4 * g] * scale, o[db][4 * g + 1] * scale, o[db][4 * g + 2] * scale, o[db][4 * g + 3] * scale};
  __syncthreads();
  constexpr int kPieces = kRG * 32 * (D / 8);  // 16 bytes of a row each
#pragma unroll
  for (int j = 0; j < kPieces / 256; ++j) {
    const int id = j * 256 + tid, row = id / (D / 8), c = id % (D / 8);
    const unsigned char* from = smem + (row / 32) * kWave;
    float x[8];
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      f32x4 s = *reinterpret_cast<const f32x4*>(from + KS::off(row & 31, 2 * c + hf));
#pragma unroll
      for (int w = 1; w < P; ++w) {
        const f32x4 y = *reinterpret_cast<const f32x4*>(from + w * kRG * kWave + KS::off(row & 31, 2 * c + hf));
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] += y[e];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) x[4 * hf + e] = s[e];
    }
    if (wg_row0 + row < n)
      *reinterpret_cast<u32x4*>(out + (size_t)(wg_row0 + row) * (D * 2) + c * 16) = u32x4{pack2<T>(x[0], x[1]), pack2<T>(x[2], x[3]), pack2<T>(x[4], x[5]), pack2<T>(x[6], x[7])};
  }
}

template <int D> __device__ __forceinline__ void load_frags(const unsigned char* row, bool ok, int lh, uint32_t (&f)[D / 4]) {
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks) {
    const u32x4 raw = *reinterpret_cast<const u32x4*>(row + ks * 32 + 16 * lh);
#pragma unroll
    for (int e = 0; e < 4; ++e) f[ks * 4 + e] = ok ? raw[e] : 0u;
  }
}
__device__ __forceinline__ void zero_rows(unsigned char* at, int bytes, int tid) {
  for (int i = tid; i < bytes / 16; i += 256) reinterpret_cast<u32x4*>(at)[i] = u32x4{0u, 0u, 0u, 0u};
}
__device__ __forceinline__ f32x16 splat(float x) {
  f32x16 v;
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = x;
  asm volatile("" : "+v"(v));  // sixteen registers that stay: the accumulators' start, instead of sixteen moves a block
  return v;
}

}  // namespace tile16
}  // namespace adsp
