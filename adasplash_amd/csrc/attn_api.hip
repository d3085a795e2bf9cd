// C ABI of the attention forward and backward: argument checks, re-layout launches, kernel dispatch.
#include "common.h"
#include "attn_params.h"
#include "attn_bwd_params.h"
#include <math.h>
#include <stdlib.h>
#include <string.h>
#include "../../include/adasplash_hip.h"

namespace adsp {
// The kernels live in one translation unit per (element type, head dim, instance): attn_fwd_unit.hip and
// attn_bwd_unit.hip, compiled once per combination.
#define ADSP_DECL_D(tag, d)                                                      \
  int launch_attn_fwd_##tag##_d##d##_m0(const AttnParams&, int, hipStream_t);   \
  int launch_attn_fwd_##tag##_d##d##_m1(const AttnParams&, int, hipStream_t);   \
  int launch_attn_bwd_##tag##_d##d(const AttnBwdParams&, int, int, hipStream_t);  // (16-bit: head dims 16, 32 and 256)
#define ADSP_DECL_TAG(tag) ADSP_DECL_D(tag, 16) ADSP_DECL_D(tag, 32) ADSP_DECL_D(tag, 64) ADSP_DECL_D(tag, 128) ADSP_DECL_D(tag, 256)
ADSP_DECL_TAG(f32)
ADSP_DECL_TAG(bf16)
ADSP_DECL_TAG(f16)
// attn_fwd_sparse_kernel (attn_sparse_unit.hip): 16-bit types, head dims 64 and 128
int launch_attn_sparse_bf16_d64(const AttnParams&, int, int, hipStream_t);
int launch_attn_sparse_bf16_d128(const AttnParams&, int, int, hipStream_t);
int launch_attn_sparse_f16_d64(const AttnParams&, int, int, hipStream_t);
int launch_attn_sparse_f16_d128(const AttnParams&, int, int, hipStream_t);
// attn_bwd_dq_sparse_kernel (attn_bwd_sparse_unit.hip): likewise
int launch_attn_bwd_sparse_bf16_d64(const AttnBwdParams&, int, int, int, hipStream_t);
int launch_attn_bwd_sparse_bf16_d128(const AttnBwdParams&, int, int, int, hipStream_t);
int launch_attn_bwd_sparse_f16_d64(const AttnBwdParams&, int, int, int, hipStream_t);
int launch_attn_bwd_sparse_f16_d128(const AttnBwdParams&, int, int, int, hipStream_t);

// the single-precision kernels on 32 rows a workgroup (attn_f32_unit.hip): head dims 64 and 128
int launch_attn_f32_fwd_d64(const AttnParams&, int, hipStream_t);
int launch_attn_f32_fwd_d128(const AttnParams&, int, hipStream_t);
int launch_attn_f32_bwd_d64(const AttnBwdParams&, int, hipStream_t);
int launch_attn_f32_bwd_d128(const AttnBwdParams&, int, hipStream_t);

// 16-bit types, head dims 64 and 128: the forward on 32 rows a workgroup with lists (attn_rows32_unit.hip), the one with a row's
// scores in registers (attn_resident_unit.hip), the one that walks all pairs (attn_fwd16_unit.hip), and dQ and dK/dV on all
// pairs (attn_bwd16_unit.hip)
#define ADSP_DECL_16(tag, d)                                                        \
  int launch_attn_rows32_fwd_##tag##_d##d(const AttnParams&, int, hipStream_t);     \
  int launch_attn_resident_fwd_##tag##_d##d(const AttnParams&, int, hipStream_t);   \
  int launch_attn_fwd16_##tag##_d##d(const AttnParams&, int, hipStream_t);          \
  int launch_attn_bwd16_##tag##_d##d(const AttnBwdParams&, int, int, bool, hipStream_t);
ADSP_DECL_16(bf16, 64)
ADSP_DECL_16(bf16, 128)
ADSP_DECL_16(f16, 64)
ADSP_DECL_16(f16, 128)
#define ADSP_CALL_16(name, D, dtype, ...)                                                                \
  ((dtype) == ADSP_BF16 ? ((D) == 64 ? name##_bf16_d64(__VA_ARGS__) : name##_bf16_d128(__VA_ARGS__))    \
                        : ((D) == 64 ? name##_f16_d64(__VA_ARGS__) : name##_f16_d128(__VA_ARGS__)))

typedef int (*attn_fwd_fn)(const AttnParams&, int, hipStream_t);
typedef int (*attn_bwd_fn)(const AttnBwdParams&, int, int, hipStream_t);
#define ADSP_FWD_ROW(tag, d) {launch_attn_fwd_##tag##_d##d##_m0, launch_attn_fwd_##tag##_d##d##_m1}
#define ADSP_FWD_TAG(tag) {ADSP_FWD_ROW(tag, 16), ADSP_FWD_ROW(tag, 32), ADSP_FWD_ROW(tag, 64), ADSP_FWD_ROW(tag, 128), ADSP_FWD_ROW(tag, 256)}
// (the 16-bit backward at head dims 64 and 128 has kernels of its own, attn_bwd16_unit.hip)
#define ADSP_BWD_TAG16(tag) {launch_attn_bwd_##tag##_d16, launch_attn_bwd_##tag##_d32, nullptr, nullptr, launch_attn_bwd_##tag##_d256}
// indexed by adsp_dtype (ADSP_F32 = 0, ADSP_BF16 = 1, ADSP_F16 = 2), head dim slot, instance
static const attn_fwd_fn kFwdTable[3][5][2] = {ADSP_FWD_TAG(f32), ADSP_FWD_TAG(bf16), ADSP_FWD_TAG(f16)};
static const attn_bwd_fn kBwdTable[3][5] = {
    {launch_attn_bwd_f32_d16, launch_attn_bwd_f32_d32, launch_attn_bwd_f32_d64, launch_attn_bwd_f32_d128, launch_attn_bwd_f32_d256},
    ADSP_BWD_TAG16(bf16), ADSP_BWD_TAG16(f16)};
// An alpha whose 1 / (alpha - 1) is 1 in fp32 is 2 to the kernels: the generic ones raise u = 0 to the power 1 / (alpha - 1) - 1.
static int alpha_mode(double alpha) {
  return alpha == 1.5 ? ATT_15 : (alpha == 2.0 || (float)(1.0 / (alpha - 1.0)) == 1.f ? ATT_2 : ATT_GEN);
}
static int head_dim_slot(int D) { return D == 16 ? 0 : (D == 32 ? 1 : (D == 64 ? 2 : (D == 128 ? 3 : (D == 256 ? 4 : -1)))); }
// dQ and / or dK and dV of whatever is not left to the kernels on the supports
static int launch_bwd_dense(const AttnBwdParams& p, int D, int dtype, int am, int which, hipStream_t s) {
  if (dtype != ADSP_F32 && (D == 64 || D == 128)) return ADSP_CALL_16(launch_attn_bwd16, D, dtype, p, am, which, false, s);
  return kBwdTable[dtype][head_dim_slot(D)](p, am, which, s);
}

// e4m3 copy of K for the first walk of the sparse-support forward: [B * Hkv][Npad][D] bytes in the order of K, values
// beyond the format's range saturated, rows from N on zero.  The values are multiplied by the head's power of two first
// (`ak`, from the probe) and lie on the first walk's grid of 1/16 (see attn_sparse_kernel.h).
// A thread converts 16 values at a time: element `id` of the head's rows.
template <typename T, int D>
struct K8Copy {
  const u32x4* src;  // the head's rows, 8 values a piece
  u32x4* dst;
  long long rows, n;  // of K; of the copy: whole tiles of the sequence's length
  u32x4 lo, hi;
  __device__ K8Copy(const uint16_t* k, unsigned char* k8, size_t head, int N, int Npad, int L)
      : src(reinterpret_cast<const u32x4*>(k + head * (size_t)N * D)), dst(reinterpret_cast<u32x4*>(k8 + head * (size_t)Npad * D)),
        rows((long long)N * (D / 16)), n((long long)((L + kBN - 1) / kBN * kBN) * (D / 16)) {}
  __device__ void load(long long id) {
    lo = hi = u32x4{0u, 0u, 0u, 0u};
    if (id < n && id < rows) {
      lo = src[2 * id];
      hi = src[2 * id + 1];
    }
  }
  __device__ void store(long long id, float ak) const {
    if (id >= n) return;
    auto on_grid = [ak](float x) { return (x * ak + 786432.f) - 786432.f; };
    u32x4 out;
#pragma unroll
    for (int e = 0; e < 4; e += 2) {
      out[e >> 1] = cvt_e4m3_pair(on_grid(unpack_lo<T>(lo[e + 1])), on_grid(unpack_hi<T>(lo[e + 1])), cvt_e4m3_pair(on_grid(unpack_lo<T>(lo[e])), on_grid(unpack_hi<T>(lo[e])), 0u, false), true);
      out[2 + (e >> 1)] = cvt_e4m3_pair(on_grid(unpack_lo<T>(hi[e + 1])), on_grid(unpack_hi<T>(hi[e + 1])), cvt_e4m3_pair(on_grid(unpack_lo<T>(hi[e])), on_grid(unpack_hi<T>(hi[e])), 0u, false), true);
    }
    dst[id] = out;
  }
};

// The copy by itself, behind the probe: a thread to 16 values.  Heads the probe has marked as dense are skipped.
template <typename T, int D>
__global__ __launch_bounds__(256) void k8_layout_kernel(AttnParams p) {
  const int u = blockIdx.y;
  long long L = p.N;
  if (p.varlen) L = p.varlen_bits == 64 ? ((const long long*)p.varlen)[u / p.Hkv] : (long long)((const int*)p.varlen)[u / p.Hkv];
  L = L < 0 ? 0 : (L > p.N ? p.N : L);
  if (p.hints[2 * u] >= (1u << 20)) return;
  K8Copy<T, D> copy(reinterpret_cast<const uint16_t*>(p.k), const_cast<unsigned char*>(p.k8), (size_t)u, p.N, p.Npad, (int)L);
  const long long id = (long long)blockIdx.x * 256 + threadIdx.x;
  copy.load(id);
  copy.store(id, p.w1_scales[4 * u + 1]);
}

static int npad_of(int N) { return (N + kBN - 1) / kBN * kBN; }
static int mblocks_of(int N) { return (N + kMaskRows - 1) / kMaskRows; }
static int mask_words_of(int N) { return ((N + kBN - 1) / kBN + 31) / 32; }

// Control words of the sparse-support forward (the `queue` pointer of AttnParams): eight work counters, the number
// of row blocks it left to the dense kernel, a word saying that the probe below leaves every K/V head to the dense
// kernel; from word 64 on two words per K/V head and two more (the first of a head's pair is 1 << 20 when the probe
// leaves the whole head to the dense kernel; the backward's kernels keep row-block counters in the others), then four
// floats per K/V head (AttnParams::w1_scales).
//
// attn_probe_kernel clears them and looks at a sample of each K/V head's scores (one workgroup per head: four long
// query rows of the group's first head against 256 evenly spaced keys): from the sample's variance the support a
// Gaussian score distribution would have for a row that sees n keys follows in closed form (n s^2 g(a) = 1 with
// g(a) = (1 + a^2) Q(a) - a phi(a) for alpha = 1.5, n s h(a) = 1 with h(a) = phi(a) - a Q(a) for alpha = 2; support
// n Q(a)).  It grows with n: the probe stores the largest n whose predicted support the candidate lists hold, and the
// sparse-support kernels leave the row blocks that see more keys to the dense kernels without spending a walk on
// them.  The prediction only decides which kernel does the work (a row block it gets wrong is caught by the kernel's
// own checks), and it depends on the inputs alone: the same call takes the same way every time.
//
// What bounds it is latency, one workgroup per K/V head in front of the real work: the sampled keys' rows and the query rows are
// all under way at once, and the length whose predicted support just fits comes from the support point instead
// of the other way round -- a lane takes an a, n(a) = 1 / (mass above a per key) and support n(a) Q(a) are closed forms that
// grow with a, and a second look between the two neighbouring lanes refines it (bisecting a for 64 lengths
// took 14 rounds, each an integral of 32 terms at a generic alpha).  192 heads, D = 64: 10.7 -> 6.7 us a launch.
//
// (all 256 threads; `first`: writes what it finds; `share` as in the kernel below, written by thread 0)
template <typename T, int D>
__device__ __forceinline__ void probe_head(const AttnParams& p, int am, int u, int L, bool first, float* share) {
  __shared__ float red[4][2][4];
  __shared__ float ksum[4];
  const int tid = threadIdx.x;
  const int b = u / p.Hkv, kvh = u % p.Hkv, group = p.Hq / p.Hkv;
  if (L < 256) return;  // short sequences: finding out in the kernel costs little
  // Lanes side by side read a row's pieces of 16 bytes, so a load is whole lines; the sums over a row's lanes leave each lane with one
  // key's scores.  (A row to a lane made each load 64 lines, which several workgroups on a CU pay for one after another: 64 heads, D = 128, 11.7 -> 9.4 us a launch; with the copy of 32 workgroups a head 6 us less.)
  constexpr int P = D / 8;  // pieces of a row, and loads of 64 / P rows a wave
  const int lane = tid & 63, piece = lane % P;
  const int last_row = L - 1 - 3 * (L / 16);
  const int span = (p.causal ? last_row + 1 : L);
  const u32x4* kg = reinterpret_cast<const u32x4*>(p.k) + (size_t)(b * p.Hkv + kvh) * p.N * P + piece;
  u32x4 kw[P], qw[4];
#pragma unroll
  for (int i = 0; i < P; ++i) kw[i] = kg[(size_t)(((long long)((tid & ~63) + i * (64 / P) + lane / P) * span) / 256) * P];
  const u32x4* qg = reinterpret_cast<const u32x4*>(p.q) + (size_t)(b * p.Hq + kvh * group) * p.N * P + piece;
#pragma unroll
  for (int j = 0; j < 4; ++j) qw[j] = qg[(size_t)(L - 1 - j * (L / 16)) * P];
  float dot[P][4];
  float ksq = 0.f;
#pragma unroll
  for (int i = 0; i < P; ++i) {
#pragma unroll
    for (int j = 0; j < 4; ++j) dot[i][j] = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float lo = unpack_lo<T>(kw[i][e]), hi = unpack_hi<T>(kw[i][e]);
      ksq = fmaf(lo, lo, fmaf(hi, hi, ksq));
#pragma unroll
      for (int j = 0; j < 4; ++j) dot[i][j] = fmaf(lo, unpack_lo<T>(qw[j][e]), fmaf(hi, unpack_hi<T>(qw[j][e]), dot[i][j]));
    }
  }
#pragma unroll
  for (int h = P / 2; h > 0; h >>= 1) {
    const bool upper = (lane & h) != 0;
#pragma unroll
    for (int i = 0; i < h; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float keep = upper ? dot[i + h][j] : dot[i][j], give = upper ? dot[i][j] : dot[i + h][j];
        dot[i][j] = keep + __shfl_xor(give, h, 64);
      }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float z = dot[0][j] * p.qscale;
    const float s1 = wave_sum(z), s2 = wave_sum(z * z);
    if (lane == 0) {
      red[tid >> 6][0][j] = s1;
      red[tid >> 6][1][j] = s2;
    }
  }
  {
    const float ks = wave_sum(ksq);
    if (lane == 0) ksum[tid >> 6] = ks;
  }
  __syncthreads();
  if (tid == 0 && p.w1_scales) {
    // Scales of the first walk's operands: the sampled raw scores' root mean square goes to about 8 (the walk's
    // tags hold scores up to 512), shared between q and k so that k's own root mean square comes near 8 / sqrt(D).
    float raw2 = 0.f;
    for (int j = 0; j < 4; ++j) raw2 += red[0][1][j] + red[1][1][j] + red[2][1][j] + red[3][1][j];
    const float s_rms = sqrtf(raw2 / 1024.f) / p.qscale;
    const float k_rms = sqrtf((ksum[0] + ksum[1] + ksum[2] + ksum[3]) / (256.f * (float)D));
    if (s_rms > 0.f && k_rms > 0.f && s_rms < INFINITY && k_rms < INFINITY) {
      const float a = exp2f(rintf(log2f(8.f / s_rms)));
      float ak = exp2f(rintf(log2f(8.f / (sqrtf((float)D) * k_rms))));
      ak = fminf(fmaxf(ak, 0x1p-40f), 0x1p40f);
      float aq = fminf(fmaxf(a / ak, 0x1p-40f), 0x1p40f);
      if (first) {
        p.w1_scales[4 * u] = aq;
        p.w1_scales[4 * u + 1] = ak;
      }
      share[0] = ak;
    }
  }
  if (tid >= 64) return;
  // The first wave: the score spread pooled over the four sampled rows, and the largest n whose support, were the scores
  // Gaussian with that spread, still fits: what the sparse-support kernels compare a row block's keys with.
  float var = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float s1 = red[0][0][j] + red[1][0][j] + red[2][0][j] + red[3][0][j];
    const float s2 = red[0][1][j] + red[1][1][j] + red[2][1][j] + red[3][1][j];
    const float mean = s1 / 256.f;
    var += 0.25f * fmaxf(s2 / 256.f - mean * mean, 0.f);
  }
  const float sd = sqrtf(var);
  // keys whose rows have their threshold `a` spreads above the mean, and the support of such a row
  auto keys_at = [&](float a, float& support) -> float {
    const float Q = 0.5f * erfcf(a * 0.70710678f), phi = 0.39894228f * __expf(-0.5f * a * a);
    float f;  // mass of one key
    if (am == ATT_2) f = sd * (phi - a * Q);
    else if (am == ATT_15) f = var * ((1.f + a * a) * Q - a * phi);
    else {  // any alpha: E[(sd (Z - a))_+^c0] by the midpoint rule over [a, a + 8]
      float acc = 0.f;
#pragma unroll 4
      for (int i = 0; i < 32; ++i) {
        const float x = 0.25f * ((float)i + 0.5f);
        acc += __expf(p.c0 * __logf(sd * x)) * 0.39894228f * __expf(-0.5f * (a + x) * (a + x));
      }
      f = acc * 0.25f;
    }
    const float n = f > 0.f ? 1.f / f : INFINITY;
    support = n * Q;
    return n;
  };
  float lo = -2.f, width = 9.f, n_true = 0.f;
  for (int round = 0; round < 2; ++round) {
    const float step = width * (1.f / 63.f);
    float support;
    const float n = keys_at(lo + (float)tid * step, support);
    const unsigned long long fits = __builtin_amdgcn_ballot_w64(support <= p.probe_max_support);
    // (support grows with a: the lanes that fit are the first ones.  None: the threshold lies below every key of any length
    // considered, the support is the whole row; a spread of zero or a NaN ends here too)
    const int last = fits == ~0ull ? 63 : __builtin_ctzll(~fits) - 1;
    if (last < 0) {
      if (round == 0) n_true = p.probe_max_support * (1.f / 0.97725f);
      break;
    }
    // (all of them: even the shortest lengths have their threshold above the range, and so few keys there that any fits)
    n_true = round == 0 && last == 63 ? INFINITY : __shfl(n, last, 64);
    lo += (float)last * step;
    width = step;
    if (last == 63) break;
  }
  // on a geometric grid of lengths from 64 to a million keys, rounded down
  const float top = floorf(log2f(n_true * (1.f / 64.f)) * (63.f / 14.f) + 1e-4f);
  const float n_fit = n_true < 64.f ? 0.f : (top >= 63.f ? INFINITY : 64.f * exp2f(top * (14.f / 63.f)));
  if (tid != 0) return;
  // A head goes one way as a whole: by its longest rows, which see all L keys and hold most of the work.  (Serving only
  // its shorter row blocks from their supports was measured and loses: for a row block of few tiles the fixed cost of the
  // lists outweighs the walks saved, and a launch split between the two kernels took 15 % longer than the dense kernel
  // alone.)  A marked head: the copy of K skips it and the sparse-support kernels leave its row blocks to the dense ones.
  const bool fits_all = n_fit >= (float)L;
  if (p.w1_scales && first) p.w1_scales[4 * u + 2] = fits_all ? INFINITY : 0.f;
  if (!fits_all) {
    if (first) p.queue[64 + 2 * u] = 1u << 20;
    share[1] = 1.f;
  }
}

// In front of a backward it clears the control words and flags of the dK/dV kernels as well (`ctrl2`, `kv_flags`).
//
// COPY, in front of a forward: gridDim.y workgroups look at a head, each to the same result, the first of them writes it, and
// all of them go on with the e4m3 copy of the head's K (none where the head is marked; tiles that lie wholly behind a
// sequence's length, which no walk reads, are left out).  A launch and the
// wait for the probe's end are saved by that; where and how it is worth it: launch_probe_as.
template <typename T, int D, bool COPY>
__global__ __launch_bounds__(256) void attn_probe_kernel(AttnParams p, int am, uint32_t* ctrl2, int32_t* kv_flags) {
  __shared__ float share[2];  // COPY: k's scale; nonzero where the head is marked
  const int u = blockIdx.x, tid = threadIdx.x;
  const int units = p.B * p.Hkv;
  uint32_t* const ctrl = p.queue;
  const int b = u / p.Hkv, kvh = u % p.Hkv, group = p.Hq / p.Hkv;
  const bool first = !COPY || blockIdx.y == 0;
  int L = p.N;
  if (p.varlen) {
    long long l = p.varlen_bits == 64 ? ((const long long*)p.varlen)[b] : (long long)((const int*)p.varlen)[b];
    L = (int)(l < 0 ? 0 : (l > p.N ? p.N : l));
  }
  if (first) {
    if (u == 0 && tid < 11) ctrl[tid] = 0u;
    if (u == 0 && tid < 2) ctrl[64 + 2 * units + tid] = 0u;
    if (tid < 2) ctrl[64 + 2 * u + tid] = 0u;
    if (ctrl2 && u == 0 && tid < 11) ctrl2[tid] = 0u;
    if (kv_flags) {
      const int n_mblk = (p.N + kMaskRows - 1) / kMaskRows;
      for (int i = tid; i < n_mblk; i += 256) kv_flags[(size_t)u * n_mblk + i] = 0;
    }
    if (p.save_flags)  // supports kept for the backward: no row block of this K/V head has a valid stream yet
      for (int i = tid; i < group * p.n_mblk; i += 256) p.save_flags[(size_t)(b * p.Hq + kvh * group) * p.n_mblk + i] = 0;
    if (p.w1_scales && tid < 4) p.w1_scales[4 * u + tid] = tid < 2 ? 1.f : (tid == 2 ? INFINITY : 0.f);
  }
  if constexpr (COPY) {
    K8Copy<T, D> copy(reinterpret_cast<const uint16_t*>(p.k), const_cast<unsigned char*>(p.k8), (size_t)u, p.N, p.Npad, L);
    long long id = (long long)blockIdx.y * 256 + tid;
    copy.load(id);  // (under way while the probe works)
    if (tid == 0) {
      share[0] = 1.f;
      share[1] = 0.f;
    }
    probe_head<T, D>(p, am, u, L, first, share);
    __syncthreads();
    const float ak = share[0];
    if (share[1] != 0.f) return;
    const long long step = (long long)gridDim.y * 256;
    for (; id - tid < copy.n; id += step) {
      K8Copy<T, D> now = copy;
      copy.load(id + step);
      now.store(id, ak);
    }
  } else {
    probe_head<T, D>(p, am, u, L, true, share);
  }
}

// Workspace of the forward for the 16-bit types, for the head dims the sparse-support kernel serves: its work
// counters, its per-row-block flags, its candidate streams and the e4m3 copy of K that its first walk reads.  (The
// dense kernel needs none: it reads V row-major and transposes in the LDS read.)
constexpr int kSparseMaxSlots = 1024;                       // workgroups of the persistent kernel
constexpr size_t kSparseSlotBytes = (size_t)4 * 1616 * 8;   // four waves x 1616 candidates x (score, key)
struct FwdWorkspace {
  size_t vt_bytes, queue_off, scales_off, flags_off, events_off, k8_off, total;
  int slots;  // 0: no sparse-support kernel for these dimensions
};
static size_t align256(size_t x) { return (x + 255) / 256 * 256; }
static FwdWorkspace fwd_workspace(int B, int Hq, int Hkv, int N, int D, int dtype) {
  FwdWorkspace w = {};
  if (dtype == ADSP_F32) return w;
  w.vt_bytes = 0;
  w.total = 0;
  if ((D == 64 || D == 128) && N <= 65536) {  // (the candidate lists hold 16-bit key indices)
    const long long items = (long long)B * Hq * mblocks_of(N);
    long long slots = (items + 7) / 8 * 8;
    if (slots > kSparseMaxSlots) slots = kSparseMaxSlots;
    w.slots = (int)slots;
    w.queue_off = align256(w.vt_bytes);
    // eight counters, then two hint words per K/V head and two more, then four floats per K/V head
    w.scales_off = w.queue_off + 256 + ((size_t)B * Hkv + 1) * 8;
    w.flags_off = align256(w.scales_off + (size_t)B * Hkv * 16);
    w.events_off = align256(w.flags_off + (size_t)items * 4);
    w.k8_off = align256(w.events_off + (size_t)slots * kSparseSlotBytes);
    w.total = w.k8_off + (size_t)B * Hkv * npad_of(N) * D;  // the e4m3 copy of K
  }
  return w;
}

// Supports the forward keeps for the backward (adsp_attn_supports_bytes): a flag per row block, the length of every
// (row block, wave) stream, every row's threshold minus lower bound, and the streams.
struct SupportsLayout {
  size_t flags_off, lens_off, tshift_off, streams_off, total;  // total = 0: nothing to keep for these dimensions
};
static SupportsLayout supports_layout(int B, int Hq, int Hkv, int N, int D, int dtype) {
  SupportsLayout l = {};
  if (dtype == ADSP_F32 || fwd_workspace(B, Hq, Hkv, N, D, dtype).slots == 0) return l;
  const size_t items = (size_t)B * Hq * mblocks_of(N);
  l.flags_off = 0;
  l.lens_off = align256(items * 4);
  l.tshift_off = align256(l.lens_off + items * 4 * 2);
  l.streams_off = align256(l.tshift_off + (size_t)B * Hq * N * 4);
  l.total = l.streams_off + items * kSparseSlotBytes;
  return l;
}
__global__ __launch_bounds__(256) void fill_zero_kernel(int32_t* x, long long n) {
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256) x[i] = 0;
}

// The probe, and in front of a forward (COPY) the e4m3 copy of K, for the head dims the sparse-support kernels serve.
constexpr long long kCopyPieces = 4096;  // pieces of 256 threads x 16 values that the probe's own workgroups copy
template <typename T, int D, bool COPY>
static void launch_probe_as(const AttnParams& p, int am, uint32_t* ctrl2, int32_t* kv_flags, hipStream_t s) {
  const long long units = (long long)p.B * p.Hkv;
  if constexpr (COPY) {
    const long long pieces = ((long long)p.Npad * (D / 16) + 255) / 256;
    // Up to 32 MiB of K the probe's workgroups copy it.  About one to a CU: looking at a head again costs each of them the sample's loads (2 x 32/8
    // heads, N = 2048, D = 128: forward 150 us with the copy behind the probe, 146.5 with 256 workgroups, 147.2 with 512, 152 with 1024), and more, to
    // what a CU holds, once eight pieces and more are left to each.  The forward, copy behind the probe against this: 32/8 heads, N = 2048, D = 128
    // 98.4 -> 93.6; 8 heads, N = 4096, D = 64 116.4 -> 113.0; 4 x 16 heads 329 -> 326 (16 MiB).  For larger K the copy
    // wants more bytes in flight than these workgroups have: 4 x 16 heads, N = 4096, D = 128 (64 MiB) 304 -> 309; 8 x 8 heads, N <= 8192 2223 -> 2250.
    if (units * pieces <= kCopyPieces) {
      long long parts = (255 + units) / units;
      const long long more = pieces / 8 < 768 / units ? pieces / 8 : 768 / units;
      parts = parts > more ? parts : more;
      parts = parts < pieces ? parts : pieces;
      hipLaunchKernelGGL((attn_probe_kernel<T, D, true>), dim3((unsigned)units, (unsigned)parts), dim3(256), 0, s, p, am, ctrl2, kv_flags);
      return;
    }
    hipLaunchKernelGGL((attn_probe_kernel<T, D, false>), dim3((unsigned)units), dim3(256), 0, s, p, am, ctrl2, kv_flags);
    hipLaunchKernelGGL((k8_layout_kernel<T, D>), dim3((unsigned)pieces, (unsigned)units), dim3(256), 0, s, p);
  } else {
    hipLaunchKernelGGL((attn_probe_kernel<T, D, false>), dim3((unsigned)units), dim3(256), 0, s, p, am, ctrl2, kv_flags);
  }
}
template <bool COPY>
static void launch_probe(const AttnParams& p, int D, int dtype, int am, uint32_t* ctrl2, int32_t* kv_flags, hipStream_t s) {
  if (dtype == ADSP_BF16) {
    if (D == 64) launch_probe_as<bf16_t, 64, COPY>(p, am, ctrl2, kv_flags, s);
    else launch_probe_as<bf16_t, 128, COPY>(p, am, ctrl2, kv_flags, s);
  } else {
    if (D == 64) launch_probe_as<f16_t, 64, COPY>(p, am, ctrl2, kv_flags, s);
    else launch_probe_as<f16_t, 128, COPY>(p, am, ctrl2, kv_flags, s);
  }
}

// ADSP_SPARSE=0 in the environment keeps every row block of a 16-bit call on the dense kernels (for comparisons and tests).
static bool sparse_enabled() {
  const char* e = getenv("ADSP_SPARSE");
  return !(e && strcmp(e, "0") == 0);
}
// The probe leaves a K/V head to the dense kernel when the support its Gaussian model predicts exceeds this many keys.
// ADSP_PROBE_MAX_SUPPORT in the environment overrides it (0: every head is left to the dense kernel, which then runs
// behind the sparse-support kernel as it does for the row blocks that kernel gives up; for comparisons).
static float probe_max_support() {
  const char* e = getenv("ADSP_PROBE_MAX_SUPPORT");
  return e ? (float)atof(e) : 28.f;
}

// ADSP_BWD_STREAMS=0 in the environment makes the sparse-support dK/dV kernel walk for itself instead of taking the
// dQ kernel's streams (for comparisons and tests).
static bool bwd_streams_enabled() {
  const char* e = getenv("ADSP_BWD_STREAMS");
  return !(e && strcmp(e, "0") == 0);
}

// With a causal mask the kernel on the dQ kernel's streams serves the key blocks from this share (in 256ths) of a
// sequence on with one item for all query heads of a K/V head (attn_bwd_dkdv_stream_kernel).  ADSP_DKDV_MERGE256 in the
// environment overrides it (0: every key block per query head, with partial rows; for comparisons and tests).
// Where the line lies: in units of the first key block's item, whose queries are a head's all, the longest merged item is
// group * (1 - share), and a workgroup's part of the launch (two of them a CU) half of the row blocks / 512.  Merging saves partial rows, so it
// starts as early as it can without an item that takes longer than the rest of the launch, or than the first key block's, which is there anyway; not before
// 80 / 256, where long launches do best.  Training steps with 80 / 256 against
// this, D = 128: 32/8 heads, N = 2048 346 -> 320 us, 16/4, N = 4096 456 -> 413, 32/8, N = 8192 1266 -> 1255; D = 64: 2 x 16/2, N = 2048 396 -> 246, 2 x 16/1, N = 4096
// 906 -> 434, 4 x 16/4, N <= 1500 286 -> 252.  (224 throughout: 4 x 32/8, N <= 3000, D = 128 945 -> 983, which this leaves at 80.)
static int dkdv_merge256(int B, int Hq, int Hkv, int N) {
  const char* e = getenv("ADSP_DKDV_MERGE256");
  int v = 80;
  if (e) {
    v = atoi(e);
  } else {
    const double part = (double)B * Hq * mblocks_of(N) / 1024.0, longest = part > 1.0 ? part : 1.0;
    const double share = 256.0 * (1.0 - longest * Hkv / Hq);
    if (share > v) v = (int)share;
  }
  return v < 0 ? 0 : (v > 256 ? 256 : v);
}

// Whether a single-precision call takes the kernels of attn_f32_kernel.h: the head dims they are made for, key indices that
// fit their 16-bit list entries, and an alpha whose powers u^(1 / (alpha - 1)) stay inside fp32 (the limit of the other
// list-keeping kernels).
static bool f32_split(int N, int D, int dtype, double alpha) {
  return dtype == ADSP_F32 && (D == 64 || D == 128) && N <= 65536 && alpha >= 1.125 && alpha <= 2.0;
}

// Whether a 16-bit forward of which nobody wants the tile mask or the supports, and which the kernel with resident scores does not
// take, runs in the single kernel on 32 rows a workgroup (attn_f32_kernel.h): more than 1024 keys and few heads, for which the
// probe, the copy of K, the sparse-support kernel's items of 128 rows and the dense kernel behind it take longer than the work.
// Two workgroups fit a CU: up to 512 run at once, and the rule allows two rounds of them.  The second condition is the time the work
// itself takes, about 20 ns a workgroup and 1.35 ns a block of 32 x 32 scores with the chip full.
// Measured at the line, four launches -> this kernel, us for q of spread 1, 3 and 1/8: 16/4 heads, D = 128, N = 2048: 132 -> 93, 89 -> 54,
// 135 -> 124; beyond it 32/8 heads: 147 -> 132, 96 -> 100, 139 -> 236.
// Long sequences of few heads pass that line too, and the longest workgroup's walk is then all of the time; hence the limit on N.
// One head, D = 64 and 128 (GPU times): causal N = 4096: 147 -> 56, 103 -> 44, 171 -> 97 and 171 -> 63, 127 -> 50, 246 -> 142; N = 8192:
// 226 -> 226, 164 -> 69, 323 -> 187 and 275 -> 268, 211 -> 81, 475 -> 290; beyond it 9472: 260 -> 253, 187 -> 79, 371 -> 243 and
// 305 -> 333, 236 -> 94, 545 -> 322; full N = 4096: 155 -> 127, 102 -> 45, 597 -> 102 and 177 -> 167, 128 -> 51, 766 -> 144; beyond it 6144
// with D = 128: 238 -> 252, 170 -> 68, 1137 -> 236.  (For alpha < 1.5, where supports are longer, a list now and then overflows with
// spread 3 as well: 2 heads, N = 3015, D = 128, alpha = 1.333: 1512 -> 164, 135 -> 167, 1205 -> 113.)
static double rows32_cost_ns(int B, int Hq, int N, bool causal) {
  const double heads = (double)B * Hq, r = (N + 31) / 32;
  return heads * (20.0 * r + 1.35 * (causal ? 0.5 * r * (r + 1.0) : r * r));
}
static bool rows32_16bit(int B, int Hq, int N, int D, int dtype, double alpha, bool causal) {
  if (dtype == ADSP_F32 || (D != 64 && D != 128) || !(alpha >= 1.125 && alpha <= 2.0) || !sparse_enabled()) return false;
  if (N > (causal ? 8192 : 4096)) return false;
  const long long groups = (long long)B * Hq * ((N + 31) / 32);
  return groups <= 1024 && rows32_cost_ns(B, Hq, N, causal) <= 66e3;
}
// blocks of 32 x 32 scores of a call, padding included
static long long score_blocks(int B, int Hq, int N, bool causal) {
  const long long r = (N + 31) / 32;
  return (long long)B * Hq * (causal ? r * (r + 1) / 2 : r * r);
}
static bool resident_takes(int N, int D, int dtype, double alpha) {
  return dtype != ADSP_F32 && (D == 64 || D == 128) && N <= kResidentMaxKeys && alpha >= 1.125 && alpha <= 2.0 && sparse_enabled();
}
// Whether a 16-bit forward of which nobody wants the tile mask or the supports takes the single kernel that holds its rows' scores in
// registers (attn_resident_kernel.h).  It does the same work whatever the scores are, so the lines lie where the kernels on
// the supports, which do less where scores are peaked and rows are long, catch up with unit spread.  Up to 512 keys never; up to 1024
// where the chip has more than a few rounds of it; beyond, where a workgroup of sixteen waves fills a CU, after one or two.  us, the others
// -> this kernel, q of spread 1, 3 and 1/8:
//   16 x 12 heads, N <= 500, D = 64: 86 -> 35, 64 -> 33, 147 -> 34; 32 x 16 heads, N <= 512, D = 128: 256 -> 122, 172 -> 125, 394 -> 127;
//   N = 1024: 8 x 8/4 heads, D = 64: 93 -> 46, 63 -> 42, 59 -> 43; 3 x 16/8, D = 128: 151 -> 56, 82 -> 52, 84 -> 52; at the line 5 x 16, D = 128,
//     causal: 173 -> 92, 100 -> 83, 90 -> 86; 13 x 8/2, D = 128: 187 -> 114, 106 -> 98, 96 -> 102; beyond it 3 x 64/16, D = 128: 258 -> 186, 148 -> 172, 151 -> 180;
//   N > 1024: 1750, 8/2 heads, D = 64: 38 -> 28, 30 -> 26, 51 -> 27; 7 x 2 of 1994: 43 -> 40, 34 -> 37, 60 -> 39; 4/1 of 1684, D = 128: 40 -> 26, 30 -> 25, 64 -> 28; beyond it
//     2 x 32/8 of 1339, D = 64: 94 -> 84, 62 -> 76, 72 -> 77; 2 x 8 of 1138, D = 128: 37 -> 39, 28 -> 37, 54 -> 38.
static bool resident_16bit(int B, int Hq, int N, int D, int dtype, double alpha, bool causal) {
  if (!resident_takes(N, D, dtype, alpha)) return false;
  const long long blocks = score_blocks(B, Hq, N, causal);
  if (N <= 512) return true;
  if (N <= 1024) return blocks <= (D == 64 ? 100000 : 55000);
  return blocks <= (D == 64 ? 28000 : 8000);
}
// The training steps whose backward computes all pairs (attn_bwd16_kernel.h, dQ's weights in two parts) and whose forward keeps nothing
// for it.  Short ones as above, at less load, and none where a dK/dV workgroup, which walks the queries of all heads of its group,
// had more than 128 blocks of them to visit.  us, kernels on the supports -> these, q of spread 1, 3 and 1/8:
//   N <= 512: 16 x 12 heads, N <= 500, D = 64: 210 -> 112 (spread 1); 4 x 16/8, D = 128: 252 -> 89, 149 -> 89, 138 -> 90; 8 x 32/16, D = 128: 411 -> 227, 253 -> 224,
//     261 -> 225;
//   N <= 1024: 8 x 8/4 heads, D = 64: 235 -> 133, 145 -> 128, 161 -> 129; 3 x 16/8, D = 128: 347 -> 177, 188 -> 169, 216 -> 166; 4 x 4, D = 128, full: 251 -> 105, 133 -> 102, 160 -> 102;
//     beyond the line 2 x 32/16, D = 128: 361 -> 220, 195 -> 214, 250 -> 208; 11 x 4, D = 128, full, alpha = 2: 174 -> 280, 156 -> 265, 438 -> 271;
//   N > 1024: 7 x 2 of 1994, D = 64: 228 -> 110, 135 -> 106, 179 -> 109; 2 x 8 of 1138, D = 128: 125 -> 109, 116 -> 107, 142 -> 108; beyond it 32/8 of 1173, D = 64:
//     242 -> 161, 134 -> 156, 188 -> 157.
// And long sequences of few heads, where the forward is that on 32 rows a workgroup: one head, N = 3000, D = 64: 144 -> 133, 130 -> 123,
// 164 -> 154 (gradients on 32 rows a workgroup -> these kernels), N = 4096: 239 -> 225, 165 -> 155, 214 -> 201 (on the supports 283, 162, 492).
static bool all_pairs_training(int B, int Hq, int Hkv, int N, int D, int dtype, double alpha, bool causal) {
  if (resident_takes(N, D, dtype, alpha) && (long long)(Hq / Hkv) * ((N + 31) / 32) <= 128) {
    const long long blocks = score_blocks(B, Hq, N, causal);
    if (N <= 512) return true;
    if (blocks <= (D == 64 ? (N <= 1024 ? 50000 : (causal ? 26000 : 20000)) : (!causal ? 10000 : (N <= 1024 ? 25000 : 14000)))) return true;
  }
  if (!rows32_16bit(B, Hq, N, D, dtype, alpha, causal)) return false;
  const double cost = rows32_cost_ns(B, Hq, N, causal);
  const long long blocks = (N + 31) / 32, walk = (long long)(Hq / Hkv) * blocks;
  if (!(walk <= 64 ? cost <= 50e3 : (walk <= 128 && cost <= 25e3))) return false;
  const long long pairs = (long long)B * Hq * blocks * blocks / (causal ? 2 : 1);
  if (D == 64) return causal || (walk <= 96 && pairs <= 16384);
  if (causal) return N <= 3072 && pairs <= 18432;
  const long long rounds = ((long long)B * Hkv * blocks + 255) / 256;
  return rounds * walk <= (rounds == 1 ? 64 : 48);
}

static int attn_common(const void* q, const void* k, const void* v, void* out, float* taus, int32_t* bmask,
                       const void* varlen, int varlen_bits, int B, int Hq, int Hkv, int N, int D, int dtype,
                       double alpha, int is_causal, int niter, int use_hist, void* workspace, size_t workspace_bytes,
                       unsigned long long* tile_counts, hipStream_t s, void* supports = nullptr, size_t supports_bytes = 0) {
  if (!q || !k || !v || !out) return ADSP_ERR_NULL;
  if (dtype != ADSP_F32 && dtype != ADSP_BF16 && dtype != ADSP_F16) return ADSP_ERR_DTYPE;
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || N <= 0 || Hq % Hkv != 0) return ADSP_ERR_SHAPE;
  if (D != 16 && D != 32 && D != 64 && D != 128 && D != 256) return ADSP_ERR_SHAPE;
  if (mask_words_of(N) > kMaskWords) return ADSP_ERR_SHAPE;
  if (!(alpha > 1.0) || niter < 0) return ADSP_ERR_UNSUPPORTED;
  if (varlen && varlen_bits != 32 && varlen_bits != 64) return ADSP_ERR_UNSUPPORTED;
  if ((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out) & 15) != 0) return ADSP_ERR_ALIGN;

  AttnParams p;
  p.q = q;
  p.k = k;
  p.v = v;
  p.out = out;
  p.taus = taus;
  p.bmask = bmask;
  p.varlen = varlen;
  p.varlen_bits = varlen_bits;
  p.tile_counts = tile_counts;
  p.B = B;
  p.Hq = Hq;
  p.Hkv = Hkv;
  p.N = N;
  p.Npad = npad_of(N);
  p.n_mblk = mblocks_of(N);
  p.mask_words = mask_words_of(N);
  // The dense kernel takes the reference's extra update when it serves the call alone: the reference's solver makes
  // `niter` refinements and one more behind the mask pass (adasplash/adasplash_v2.py:567-611 and :617-681), which is
  // what brings the default niter = 1 to 1e-4 in fp32 and keeps the thresholds the backward reads within 1e-5 for the
  // 16-bit types.  The second and later steps run on the candidate lists of the list-carrying instance when they fit,
  // without another K walk.  Behind the sparse-support kernel (which converges fully) the dense kernel serves the
  // row blocks whose supports did not fit that kernel's lists, longer than its own: there it walks `niter` steps.
  const int am = alpha_mode(alpha);
  const FwdWorkspace w = dtype == ADSP_F32 ? FwdWorkspace{} : fwd_workspace(B, Hq, Hkv, N, D, dtype);
  // Sparse-support kernel first (16-bit types, alpha 1.5 / 2 or any other in [1.125, 2): below that its solver on the
  // lists would need too many rounds; either entry point, no tile statistics asked for): it serves the row blocks
  // whose supports are short and flags the others for the dense kernel.
  const bool sparse = w.slots > 0 && (am == ATT_15 || am == ATT_2 || (alpha >= 1.125 && alpha < 2.0)) &&
                      !tile_counts && (long long)B * Hq * mblocks_of(N) < (1ll << 31) && sparse_enabled();
  if (!sparse) niter += 1;
  p.niter = niter;
  p.causal = is_causal ? 1 : 0;
  p.use_hist = use_hist;
  p.alpha = (float)alpha;
  p.c0 = (float)(1.0 / (alpha - 1.0));
  p.qscale = (float)((alpha - 1.0) / sqrt((double)D));

  p.block_flags = nullptr;
  p.queue = nullptr;
  p.hints = nullptr;
  p.events = nullptr;
  p.k8 = nullptr;
  p.w1_scales = nullptr;
  p.probe_max_support = 0.f;
  p.save_flags = nullptr;
  p.save_lens = nullptr;
  p.save_tshift = nullptr;
  p.save_streams = nullptr;

  (void)hipGetLastError();
  if (!tile_counts && f32_split(N, D, dtype, alpha)) {
    if (bmask) {  // several workgroups share a row block's words
      const long long words = (long long)B * Hq * p.n_mblk * p.mask_words;
      hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)((words + 255) / 256 > 1024 ? 1024 : (words + 255) / 256)), dim3(256), 0, s, bmask, words);
    }
    if ((D == 64 ? launch_attn_f32_fwd_d64(p, am, s) : launch_attn_f32_fwd_d128(p, am, s)) != 0) return ADSP_ERR_LAUNCH;
    return hipGetLastError() == hipSuccess ? ADSP_OK : ADSP_ERR_LAUNCH;
  }
  const bool resident = resident_16bit(B, Hq, N, D, dtype, alpha, is_causal != 0);
  if (!tile_counts && !bmask && !supports && (resident || rows32_16bit(B, Hq, N, D, dtype, alpha, is_causal != 0))) {
    // (not touched, but asked for as below: the size query does not know the call)
    if (w.total && (!workspace || workspace_bytes < w.total || ((uintptr_t)workspace & 15) != 0)) return ADSP_ERR_WORKSPACE;
    const int rc = resident ? ADSP_CALL_16(launch_attn_resident_fwd, D, dtype, p, am, s) : ADSP_CALL_16(launch_attn_rows32_fwd, D, dtype, p, am, s);
    return rc == 0 && hipGetLastError() == hipSuccess ? ADSP_OK : ADSP_ERR_LAUNCH;
  }
  if (dtype != ADSP_F32) {
    const SupportsLayout sl = supports ? supports_layout(B, Hq, Hkv, N, D, dtype) : SupportsLayout{};
    if (sl.total && (supports_bytes < sl.total || ((uintptr_t)supports & 15) != 0)) return ADSP_ERR_WORKSPACE;
    if (w.total && (!workspace || workspace_bytes < w.total || ((uintptr_t)workspace & 15) != 0)) return ADSP_ERR_WORKSPACE;
    unsigned char* ws = (unsigned char*)workspace;
    if (sparse) {
      p.queue = (uint32_t*)(ws + w.queue_off);
      p.hints = p.queue + 64;
      p.block_flags = (int32_t*)(ws + w.flags_off);
      p.events = ws + w.events_off;
      p.k8 = ws + w.k8_off;
      p.w1_scales = (float*)(ws + w.scales_off);
      p.probe_max_support = probe_max_support();
      if (sl.total) {
        unsigned char* sp = (unsigned char*)supports;
        p.save_flags = (int32_t*)(sp + sl.flags_off);
        p.save_lens = (uint16_t*)(sp + sl.lens_off);
        p.save_tshift = (float*)(sp + sl.tshift_off);
        p.save_streams = sp + sl.streams_off;
      }
      launch_probe<true>(p, D, dtype, am, nullptr, nullptr, s);
      int rc = dtype == ADSP_BF16 ? (D == 64 ? launch_attn_sparse_bf16_d64(p, am, w.slots, s) : launch_attn_sparse_bf16_d128(p, am, w.slots, s))
                                  : (D == 64 ? launch_attn_sparse_f16_d64(p, am, w.slots, s) : launch_attn_sparse_f16_d128(p, am, w.slots, s));
      if (rc != 0) return ADSP_ERR_LAUNCH;
    } else if (sl.total) {  // nothing is kept by this call: the backward must not take what the buffer happens to hold
      const long long items = (long long)B * Hq * mblocks_of(N);
      hipLaunchKernelGGL(fill_zero_kernel, dim3((unsigned)((items + 255) / 256 > 1024 ? 1024 : (items + 255) / 256)), dim3(256), 0, s,
                         (int32_t*)((unsigned char*)supports + sl.flags_off), items);
    }
  }
  // All pairs, 16-bit types: where more than one solver step is asked for, or a step without the histogram, the kernel that starts
  // from a sample of the keys converges in one or two walks.  4 x 16 heads, N = 4096, D = 64, flat scores, not causal (ten steps allowed):
  // 2240 -> 644 us; D = 128: 3530 -> 1067; 8 heads, N = 8192, alpha = 1.333: 2860 -> 1020.  A single step behind the histogram, the causal
  // entry point's default, stays with the kernel below: it is less exact (relative error 6.1e-3 against 2.3e-3, more for longer rows), but its results are those of
  // one step, and of the times either kernel has the better ones: causal, 391 against 391 us, D = 128 599 against 597, 2 x 8 heads, N = 16384, D = 128 2174 against 1980, but
  // with q of spread 1/2 338 against 486.
  if (dtype != ADSP_F32 && (D == 64 || D == 128) && !tile_counts && alpha >= 1.125 && alpha <= 2.0 && (niter >= 2 || (niter == 1 && !use_hist))) {
    const int rc = ADSP_CALL_16(launch_attn_fwd16, D, dtype, p, am, s);
    return rc == 0 && hipGetLastError() == hipSuccess ? ADSP_OK : ADSP_ERR_LAUNCH;
  }
  // The list-carrying instance serves two and more solver steps, and a single step without the histogram (the
  // block-mask variant's, made for sparse supports); the other one no step, or one behind the histogram -- and
  // whatever the sparse-support kernel leaves over: those row blocks did not fit its lists, which are longer than
  // this kernel's, so they are walked step by step, and the walk-only instance does that with fewer registers.
  const bool multi = (niter >= 2 || (niter == 1 && !use_hist)) && p.queue == nullptr;
  int rc = kFwdTable[dtype][head_dim_slot(D)][multi ? 1 : 0](p, am, s);
  if (rc != 0) return ADSP_ERR_LAUNCH;
  return hipGetLastError() == hipSuccess ? ADSP_OK : ADSP_ERR_LAUNCH;
}
}  // namespace adsp

extern "C" size_t adsp_attn_workspace_bytes(int B, int Hq, int Hkv, int N, int D, int dtype) {
  if (dtype == ADSP_F32 || B <= 0 || Hq <= 0 || Hkv <= 0 || N <= 0 || D <= 0) return 0;
  return adsp::fwd_workspace(B, Hq, Hkv, N, D, dtype).total;
}

extern "C" size_t adsp_attn_supports_bytes(int B, int Hq, int Hkv, int N, int D, int dtype) {
  if (dtype == ADSP_F32 || B <= 0 || Hq <= 0 || Hkv <= 0 || N <= 0 || D <= 0) return 0;
  return adsp::supports_layout(B, Hq, Hkv, N, D, dtype).total;
}

extern "C" int adsp_attn_bwd_reads_bmask(int B, int Hq, int Hkv, int N, int D, int dtype, double alpha, int is_causal) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || N <= 0) return 1;
  return adsp::f32_split(N, D, dtype, alpha) || adsp::all_pairs_training(B, Hq, Hkv, N, D, dtype, alpha, is_causal != 0) ? 0 : 1;
}

extern "C" size_t adsp_attn_bmask_words(int N) {
  if (N <= 0) return 0;
  return (size_t)adsp::mblocks_of(N) * adsp::mask_words_of(N);
}

extern "C" int adsp_attn_v2_fwd(const void* q, const void* k, const void* v, void* out, float* taus, int32_t* bmask,
                                const void* varlen, int varlen_bits, int B, int Hq, int Hkv, int N, int D, int dtype,
                                int niter, void* workspace, size_t workspace_bytes, void* stream) {
  return adsp::attn_common(q, k, v, out, taus, bmask, varlen, varlen_bits, B, Hq, Hkv, N, D, dtype, 1.5, 1, niter, 1,
                           workspace, workspace_bytes, nullptr, (hipStream_t)stream);
}

// ---- the entry point that allocates nothing -------------------------------------------------------------------
namespace adsp {
// Same work as adsp_attn_v2_fwd with the workspace taken from a file-scope device array instead of the caller.
// `noalloc_scratch` is a host-side stand-in for the symbol here: the address the kernels can use is looked up once
// per device with hipGetSymbolAddress (every GPU holds its own copy of the array) and only that pointer is passed on.
constexpr size_t kNoAllocScratchBytes = (size_t)64 << 20;
static __device__ __align__(256) unsigned char noalloc_scratch[kNoAllocScratchBytes];
constexpr int kMaxDevices = 64;
static void* g_noalloc_ptr[kMaxDevices] = {};

static int noalloc_scratch_ptr(void** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return ADSP_ERR_LAUNCH;
  void* ptr = __atomic_load_n(&g_noalloc_ptr[dev], __ATOMIC_ACQUIRE);
  if (!ptr) {
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(noalloc_scratch)) != hipSuccess || !ptr) return ADSP_ERR_LAUNCH;
    __atomic_store_n(&g_noalloc_ptr[dev], ptr, __ATOMIC_RELEASE);  // (two threads racing here store the same address)
  }
  *out = ptr;
  return ADSP_OK;
}
}  // namespace adsp

extern "C" size_t adsp_attn_v2_fwd_noalloc_max_bytes(void) { return adsp::kNoAllocScratchBytes; }

extern "C" int adsp_attn_v2_fwd_noalloc(const void* q, const void* k, const void* v, void* out, float* taus,
                                        int32_t* bmask, const void* varlen, int varlen_bits, int B, int Hq, int Hkv,
                                        int N, int D, int dtype, int niter, void* stream) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || N <= 0) return ADSP_ERR_SHAPE;
  if (D != 16 && D != 32 && D != 64 && D != 128 && D != 256) return ADSP_ERR_SHAPE;
  if (dtype != ADSP_F32 && dtype != ADSP_BF16 && dtype != ADSP_F16) return ADSP_ERR_DTYPE;
  const size_t need = adsp_attn_workspace_bytes(B, Hq, Hkv, N, D, dtype);
  if (need > adsp::kNoAllocScratchBytes) return ADSP_ERR_TOO_LARGE;
  void* ws = nullptr;
  if (need > 0) {
    const int rc = adsp::noalloc_scratch_ptr(&ws);
    if (rc != ADSP_OK) return rc;
  }
  return adsp::attn_common(q, k, v, out, taus, bmask, varlen, varlen_bits, B, Hq, Hkv, N, D, dtype, 1.5, 1, niter, 1, ws,
                           need, nullptr, (hipStream_t)stream);
}

extern "C" int adsp_attn_v1_fwd(const void* q, const void* k, const void* v, void* out, float* taus, int32_t* bmask,
                                const void* varlen, int varlen_bits, int B, int H, int N, int D, int dtype, double alpha,
                                int is_causal, int niter, void* workspace, size_t workspace_bytes,
                                unsigned long long* tile_counts, void* stream) {
  if (alpha > 2.0) return ADSP_ERR_UNSUPPORTED;
  return adsp::attn_common(q, k, v, out, taus, bmask, varlen, varlen_bits, B, H, H, N, D, dtype, alpha, is_causal, niter,
                           0, workspace, workspace_bytes, tile_counts, (hipStream_t)stream);
}

extern "C" int adsp_attn_v2_fwd_keep(const void* q, const void* k, const void* v, void* out, float* taus, int32_t* bmask,
                                     const void* varlen, int varlen_bits, int B, int Hq, int Hkv, int N, int D, int dtype,
                                     int niter, void* workspace, size_t workspace_bytes, void* supports,
                                     size_t supports_bytes, void* stream) {
  return adsp::attn_common(q, k, v, out, taus, bmask, varlen, varlen_bits, B, Hq, Hkv, N, D, dtype, 1.5, 1, niter, 1,
                           workspace, workspace_bytes, nullptr, (hipStream_t)stream, supports, supports_bytes);
}

extern "C" int adsp_attn_v1_fwd_keep(const void* q, const void* k, const void* v, void* out, float* taus, int32_t* bmask,
                                     const void* varlen, int varlen_bits, int B, int H, int N, int D, int dtype,
                                     double alpha, int is_causal, int niter, void* workspace, size_t workspace_bytes,
                                     void* supports, size_t supports_bytes, void* stream) {
  if (alpha > 2.0) return ADSP_ERR_UNSUPPORTED;
  return adsp::attn_common(q, k, v, out, taus, bmask, varlen, varlen_bits, B, H, H, N, D, dtype, alpha, is_causal, niter,
                           0, workspace, workspace_bytes, nullptr, (hipStream_t)stream, supports, supports_bytes);
}

namespace adsp {
// Workspace of the backward for the 16-bit types, for the head dims the sparse-support kernels serve: their work
// counters, per-row-block flags and candidate streams (the forward's layout without the copy of K).  (The dense
// kernels need none: they read k, q and dout row-major and transpose in the LDS read.)
struct BwdWorkspace {
  size_t copies_bytes, queue_off, flags_off, events_off, queue2_off, kvflags_off, scratch_off, part_off, part_bytes, streams_off, dir_off, total;
  int slots;       // 0: no sparse-support kernels for these dimensions
  int dir_stride;  // offsets per stream of the hand-over table
  int part_rows;   // rows per query head of the partial rows
  int merge256;    // what the dK/dV kernel on the streams is launched with
};
static BwdWorkspace bwd_workspace(int B, int Hq, int Hkv, int N, int D, int dtype, int causal) {
  BwdWorkspace w = {};
  if (dtype == ADSP_F32) return w;
  w.copies_bytes = 0;
  w.total = 0;
  if ((D == 64 || D == 128) && N <= 65536) {
    const long long items = (long long)B * Hq * mblocks_of(N);
    long long slots = (items + 7) / 8 * 8;
    if (slots > kSparseMaxSlots) slots = kSparseMaxSlots;
    w.slots = (int)slots;
    w.queue_off = align256(w.copies_bytes);
    w.flags_off = align256(w.queue_off + 256 + ((size_t)B * Hkv + 1) * 8);
    w.events_off = align256(w.flags_off + (size_t)items * 4);
    // the dK/dV kernel: control words, a flag per (K/V head, key
    // block), fp32 sums per workgroup and fp32 partial rows of dK and dV per query head
    w.queue2_off = align256(w.events_off + (size_t)slots * kSparseSlotBytes);
    w.kvflags_off = align256(w.queue2_off + 256);
    // (fp32 sums of an item worked off in parts: 32 rows of dK | dV per wave of every workgroup)
    w.scratch_off = align256(w.kvflags_off + (size_t)B * Hkv * mblocks_of(N) * 4);
    w.part_off = align256(w.scratch_off + (size_t)slots * 4 * 32 * 2 * D * 4);
    // (with one query head per K/V head the kernel on the streams writes dK and dV itself: no partial rows; with a
    // causal mask it does so for the key blocks it merges, and the others start in front of N * merge256 / 256)
    w.merge256 = (bwd_streams_enabled() && causal && Hq != Hkv) ? dkdv_merge256(B, Hq, Hkv, N) : 0;
    w.part_rows = N;
    if (w.merge256 > 0) {
      const long long bound = ((long long)N * w.merge256 + 255) / 256;
      const long long rows = (bound + kMaskRows - 1) / kMaskRows * kMaskRows;
      if (rows < N) w.part_rows = (int)rows;
    }
    w.part_bytes = (Hq == Hkv && bwd_streams_enabled()) ? 0 : (size_t)B * Hq * w.part_rows * D * 4;
    // the dQ kernel's streams, kept per (row block, wave) for the dK/dV kernel, and where their 32-key blocks start
    w.streams_off = align256(w.part_off + 2 * w.part_bytes);
    w.dir_stride = (mblocks_of(N) * 4 + 2) / 2 * 2;
    w.dir_off = align256(w.streams_off + (size_t)items * kSparseSlotBytes);  // (a slot = the streams of four waves)
    w.total = w.dir_off + align256((size_t)items * 4 * w.dir_stride * 2);
  }
  return w;
}

// dK, dV = sum over the query heads of a K/V head of the sparse-support kernel's fp32 partial rows; key blocks left to
// attn_bwd16_dkdv_kernel are skipped (that kernel writes them), and so are those the kernel on the streams served for all
// heads at once.  A thread adds up 8 columns of
// one key row.  Rows past the valid length are zeros and their partial rows are not read (the key blocks that lie
// wholly in the padding have none).
typedef float reduce_f32x4 __attribute__((ext_vector_type(4)));
template <typename T>
__global__ __launch_bounds__(256) void dkdv_reduce_kernel(const float* __restrict__ dk_part, const float* __restrict__ dv_part,
                                                         void* dk, void* dv, const int32_t* kv_flags, const uint32_t* ctrl2,
                                                         const void* varlen, int varlen_bits, int B, int Hq, int Hkv, int N, int D,
                                                         int causal, int merge256, int part_rows) {
  if (ctrl2[kCtrlAllDense] != 0u) return;
  const int per_row = D / 8;
  const long long id = (long long)blockIdx.x * 256 + threadIdx.x;
  if (id >= (long long)B * Hkv * N * per_row) return;
  const int c = (int)(id % per_row);
  const long long rg = id / per_row;
  const int row = (int)(rg % N), bkv = (int)(rg / N);
  if (kv_flags[(size_t)bkv * ((N + kMaskRows - 1) / kMaskRows) + row / kMaskRows] != 0) return;
  const int group = Hq / Hkv, b = bkv / Hkv, kvh = bkv % Hkv;
  long long L = N;
  if (varlen) {
    L = varlen_bits == 64 ? ((const long long*)varlen)[b] : (long long)((const int*)varlen)[b];
    L = L < 0 ? 0 : (L > N ? N : L);
  }
  if (dkdv_block_merged(causal, group, row / kMaskRows * kMaskRows, (int)L, merge256)) return;  // (written by the kernel on the streams)
  float sk[8], sv[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) sk[i] = sv[i] = 0.f;
  for (int g = 0; g < (row < L ? group : 0); ++g) {
    const size_t at = (((size_t)(b * Hq + kvh * group + g) * part_rows) + row) * D + c * 8;
    const reduce_f32x4 k0 = __builtin_nontemporal_load(reinterpret_cast<const reduce_f32x4*>(dk_part + at));
    const reduce_f32x4 k1 = __builtin_nontemporal_load(reinterpret_cast<const reduce_f32x4*>(dk_part + at + 4));
    const reduce_f32x4 v0 = __builtin_nontemporal_load(reinterpret_cast<const reduce_f32x4*>(dv_part + at));
    const reduce_f32x4 v1 = __builtin_nontemporal_load(reinterpret_cast<const reduce_f32x4*>(dv_part + at + 4));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      sk[i] += k0[i];
      sk[4 + i] += k1[i];
      sv[i] += v0[i];
      sv[4 + i] += v1[i];
    }
  }
  const size_t out = (((size_t)bkv * N) + row) * D + c * 8;
  const u32x4 wk = {pack2<T>(sk[0], sk[1]), pack2<T>(sk[2], sk[3]), pack2<T>(sk[4], sk[5]), pack2<T>(sk[6], sk[7])};
  const u32x4 wv = {pack2<T>(sv[0], sv[1]), pack2<T>(sv[2], sv[3]), pack2<T>(sv[4], sv[5]), pack2<T>(sv[6], sv[7])};
  *reinterpret_cast<u32x4*>(reinterpret_cast<uint16_t*>(dk) + out) = wk;
  *reinterpret_cast<u32x4*>(reinterpret_cast<uint16_t*>(dv) + out) = wv;
}
}  // namespace adsp

extern "C" size_t adsp_attn_bwd_workspace_bytes(int B, int Hq, int Hkv, int N, int D, int dtype) {
  if (dtype == ADSP_F32 || B <= 0 || Hq <= 0 || Hkv <= 0 || N <= 0 || D <= 0) return 0;
  return adsp::bwd_workspace(B, Hq, Hkv, N, D, dtype, 0).total;
}

extern "C" size_t adsp_attn_bwd_workspace_bytes_causal(int B, int Hq, int Hkv, int N, int D, int dtype, int is_causal) {
  if (dtype == ADSP_F32 || B <= 0 || Hq <= 0 || Hkv <= 0 || N <= 0 || D <= 0) return 0;
  return adsp::bwd_workspace(B, Hq, Hkv, N, D, dtype, is_causal ? 1 : 0).total;
}

static int attn_bwd_impl(const void* q, const void* k, const void* v, const void* dout, const float* taus,
                         const int32_t* bmask, const void* varlen, int varlen_bits, void* dq, void* dk, void* dv,
                         float* delta, float* zinv, int B, int Hq, int Hkv, int N, int D, int dtype, double alpha,
                         int is_causal, void* workspace, size_t workspace_bytes, const void* supports, size_t supports_bytes,
                         void* stream) {
  using namespace adsp;
  hipStream_t s = (hipStream_t)stream;
  if (!q || !k || !v || !dout || !taus || !dq || !dk || !dv || !delta || !zinv) return ADSP_ERR_NULL;
  if (dtype != ADSP_F32 && dtype != ADSP_BF16 && dtype != ADSP_F16) return ADSP_ERR_DTYPE;
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || N <= 0 || Hq % Hkv != 0) return ADSP_ERR_SHAPE;
  if (D != 16 && D != 32 && D != 64 && D != 128 && D != 256) return ADSP_ERR_SHAPE;
  if (mask_words_of(N) > kMaskWords) return ADSP_ERR_SHAPE;
  if (!(alpha > 1.0) || alpha > 2.0) return ADSP_ERR_UNSUPPORTED;
  if (varlen && varlen_bits != 32 && varlen_bits != 64) return ADSP_ERR_UNSUPPORTED;
  if ((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)dout | (uintptr_t)dq | (uintptr_t)dk | (uintptr_t)dv) & 15) != 0)
    return ADSP_ERR_ALIGN;

  AttnBwdParams p;
  p.q = q;
  p.k = k;
  p.v = v;
  p.dout = dout;
  p.dq = dq;
  p.dk = dk;
  p.dv = dv;
  p.taus = taus;
  p.delta = delta;
  p.zinv = zinv;
  p.bmask = bmask;
  p.varlen = varlen;
  p.varlen_bits = varlen_bits;
  p.B = B;
  p.Hq = Hq;
  p.Hkv = Hkv;
  p.N = N;
  p.Npad = npad_of(N);
  p.n_mblk = mblocks_of(N);
  p.mask_words = mask_words_of(N);
  p.causal = is_causal ? 1 : 0;
  p.qscale = (float)((alpha - 1.0) / sqrt((double)D));
  p.sm_scale = (float)(1.0 / sqrt((double)D));
  p.c0 = (float)(1.0 / (alpha - 1.0));
  p.block_flags = nullptr;
  p.queue = nullptr;
  p.hints = nullptr;
  p.events = nullptr;
  p.queue2 = nullptr;
  p.kv_flags = nullptr;
  p.dk_part = nullptr;
  p.dv_part = nullptr;
  p.part_scratch = nullptr;
  p.merge256 = 0;
  p.part_rows = N;
  p.streams = nullptr;
  p.stream_dir = nullptr;
  p.dir_stride = 0;
  p.fwd_flags = nullptr;
  p.fwd_lens = nullptr;
  p.fwd_tshift = nullptr;
  p.fwd_streams = nullptr;
  const int am = alpha_mode(alpha);
  bool sparse = false;
  BwdWorkspace w = {};

  (void)hipGetLastError();
  const bool short16 = !bmask && !supports && all_pairs_training(B, Hq, Hkv, N, D, dtype, alpha, is_causal != 0);
  if (dtype != ADSP_F32) {
    w = bwd_workspace(B, Hq, Hkv, N, D, dtype, is_causal ? 1 : 0);
    const size_t need = w.total;
    if (need && (!workspace || workspace_bytes < need || ((uintptr_t)workspace & 15) != 0)) return ADSP_ERR_WORKSPACE;
    // Sparse-support dQ kernel first (alpha 1.5 / 2): it serves the row blocks whose supports are short and flags the
    // others for attn_bwd16_dq_kernel below; the dK/dV kernel reads delta and 1 / sum p from whichever of the two wrote them.
    sparse = !short16 && w.slots > 0 && (am == ATT_15 || am == ATT_2 || (alpha >= 1.125 && alpha < 2.0)) &&
             (long long)B * Hq * mblocks_of(N) < (1ll << 31) && sparse_enabled();
    if (sparse) {
      unsigned char* ws = (unsigned char*)workspace;
      p.queue = (uint32_t*)(ws + w.queue_off);
      p.hints = p.queue + 64;
      p.block_flags = (int32_t*)(ws + w.flags_off);
      p.events = ws + w.events_off;
      if (bwd_streams_enabled()) {
        p.streams = ws + w.streams_off;
        p.stream_dir = (uint16_t*)(ws + w.dir_off);
        p.dir_stride = w.dir_stride;
      }
      if (supports) {  // what the forward kept: its candidate streams stand in for the dQ kernel's walk
        const SupportsLayout sl = supports_layout(B, Hq, Hkv, N, D, dtype);
        if (sl.total && (supports_bytes < sl.total || ((uintptr_t)supports & 15) != 0)) return ADSP_ERR_WORKSPACE;
        if (sl.total) {
          const unsigned char* sp = (const unsigned char*)supports;
          p.fwd_flags = (const int32_t*)(sp + sl.flags_off);
          p.fwd_lens = (const uint16_t*)(sp + sl.lens_off);
          p.fwd_tshift = (const float*)(sp + sl.tshift_off);
          p.fwd_streams = sp + sl.streams_off;
        }
      }
      AttnParams pp = {};  // what the probe reads: q, k, lengths, dimensions, scale and the control words it clears
      pp.q = q;
      pp.k = k;
      pp.varlen = varlen;
      pp.varlen_bits = varlen_bits;
      pp.B = B;
      pp.Hq = Hq;
      pp.Hkv = Hkv;
      pp.N = N;
      pp.causal = p.causal;
      pp.qscale = p.qscale;
      pp.c0 = p.c0;
      pp.queue = p.queue;
      pp.hints = p.hints;
      pp.probe_max_support = probe_max_support();
      launch_probe<false>(pp, D, dtype, am, (uint32_t*)(ws + w.queue2_off), (int32_t*)(ws + w.kvflags_off), s);
      int rc;
      if (dtype == ADSP_BF16) {
        rc = D == 64 ? launch_attn_bwd_sparse_bf16_d64(p, am, 0, w.slots, s) : launch_attn_bwd_sparse_bf16_d128(p, am, 0, w.slots, s);
      } else {
        rc = D == 64 ? launch_attn_bwd_sparse_f16_d64(p, am, 0, w.slots, s) : launch_attn_bwd_sparse_f16_d128(p, am, 0, w.slots, s);
      }
      if (rc != 0) return ADSP_ERR_LAUNCH;
    }
  }
  if (short16) {
    const int rc = ADSP_CALL_16(launch_attn_bwd16, D, dtype, p, am, 3, true, s);
    return rc == 0 && hipGetLastError() == hipSuccess ? ADSP_OK : ADSP_ERR_LAUNCH;
  }
  if (f32_split(N, D, dtype, alpha)) {
    if ((D == 64 ? launch_attn_f32_bwd_d64(p, am, s) : launch_attn_f32_bwd_d128(p, am, s)) != 0) return ADSP_ERR_LAUNCH;
    return hipGetLastError() == hipSuccess ? ADSP_OK : ADSP_ERR_LAUNCH;
  }
  if (!sparse) {
    if (launch_bwd_dense(p, D, dtype, am, 3, s) != 0) return ADSP_ERR_LAUNCH;
    return hipGetLastError() == hipSuccess ? ADSP_OK : ADSP_ERR_LAUNCH;
  }
  // dense dQ kernel on the row blocks the sparse one flagged (delta and 1 / sum p are complete behind it), then dK and
  // dV: the sparse-support kernel per (key block, query head), the dense kernel on the key blocks it flagged, and the
  // sum of the partial rows over the query heads of each K/V head
  if (launch_bwd_dense(p, D, dtype, am, 1, s) != 0) return ADSP_ERR_LAUNCH;
  {
    unsigned char* ws = (unsigned char*)workspace;
    p.queue2 = (uint32_t*)(ws + w.queue2_off);
    p.kv_flags = (int32_t*)(ws + w.kvflags_off);
    p.part_scratch = (float*)(ws + w.scratch_off);
    if (p.streams) p.merge256 = w.merge256;
    p.part_rows = w.part_rows;
    if (w.part_bytes) {
      p.dk_part = (float*)(ws + w.part_off);
      p.dv_part = (float*)(ws + w.part_off + w.part_bytes);
    }
    int rc;
    const int kind = p.streams ? 2 : 1;  // from the dQ kernel's streams, or with a walk of its own
    if (dtype == ADSP_BF16) rc = D == 64 ? launch_attn_bwd_sparse_bf16_d64(p, am, kind, w.slots, s) : launch_attn_bwd_sparse_bf16_d128(p, am, kind, w.slots, s);
    else rc = D == 64 ? launch_attn_bwd_sparse_f16_d64(p, am, kind, w.slots, s) : launch_attn_bwd_sparse_f16_d128(p, am, kind, w.slots, s);
    if (rc != 0) return ADSP_ERR_LAUNCH;
    if (launch_bwd_dense(p, D, dtype, am, 2, s) != 0) return ADSP_ERR_LAUNCH;
    if (w.part_bytes && !(p.streams && Hq == Hkv)) {  // (with one query head per K/V head the kernel on the streams writes dK and dV itself)
      const long long threads = (long long)B * Hkv * N * (D / 8);
      const dim3 grid((unsigned)((threads + 255) / 256));
      if (dtype == ADSP_BF16)
        hipLaunchKernelGGL(dkdv_reduce_kernel<bf16_t>, grid, dim3(256), 0, s, (const float*)p.dk_part, (const float*)p.dv_part, dk, dv,
                           (const int32_t*)p.kv_flags, (const uint32_t*)p.queue2, varlen, varlen_bits, B, Hq, Hkv, N, D, p.causal, p.merge256, p.part_rows);
      else
        hipLaunchKernelGGL(dkdv_reduce_kernel<f16_t>, grid, dim3(256), 0, s, (const float*)p.dk_part, (const float*)p.dv_part, dk, dv,
                           (const int32_t*)p.kv_flags, (const uint32_t*)p.queue2, varlen, varlen_bits, B, Hq, Hkv, N, D, p.causal, p.merge256, p.part_rows);
    }
  }
  return hipGetLastError() == hipSuccess ? ADSP_OK : ADSP_ERR_LAUNCH;
}

extern "C" int adsp_attn_bwd(const void* q, const void* k, const void* v, const void* dout, const float* taus,
                             const int32_t* bmask, const void* varlen, int varlen_bits, void* dq, void* dk, void* dv,
                             float* delta, float* zinv, int B, int Hq, int Hkv, int N, int D, int dtype, double alpha,
                             int is_causal, void* workspace, size_t workspace_bytes, void* stream) {
  return attn_bwd_impl(q, k, v, dout, taus, bmask, varlen, varlen_bits, dq, dk, dv, delta, zinv, B, Hq, Hkv, N, D, dtype, alpha,
                       is_causal, workspace, workspace_bytes, nullptr, 0, stream);
}

extern "C" int adsp_attn_bwd_kept(const void* q, const void* k, const void* v, const void* dout, const float* taus,
                                  const int32_t* bmask, const void* varlen, int varlen_bits, void* dq, void* dk, void* dv,
                                  float* delta, float* zinv, int B, int Hq, int Hkv, int N, int D, int dtype, double alpha,
                                  int is_causal, void* workspace, size_t workspace_bytes, const void* supports,
                                  size_t supports_bytes, void* stream) {
  return attn_bwd_impl(q, k, v, dout, taus, bmask, varlen, varlen_bits, dq, dk, dv, delta, zinv, B, Hq, Hkv, N, D, dtype, alpha,
                       is_causal, workspace, workspace_bytes, supports, supports_bytes, stream);
}

extern "C" int adsp_version(void) { return 3; }

#ifndef ADSP_BUILD_ID
#define ADSP_BUILD_ID "unknown"
#endif
extern "C" const char* adsp_build_id(void) { return ADSP_BUILD_ID; }
#ifndef ADSP_BUILD_FLAGS
#define ADSP_BUILD_FLAGS ""
#endif
extern "C" const char* adsp_build_flags(void) { return ADSP_BUILD_FLAGS; }

extern "C" const char* adsp_status_string(int status) {
  switch (status) {
    case ADSP_OK: return "ok";
    case ADSP_ERR_NULL: return "a required pointer is NULL";
    case ADSP_ERR_SHAPE: return "a dimension is out of the supported range";
    case ADSP_ERR_DTYPE: return "unknown element type";
    case ADSP_ERR_ALIGN: return "a tensor base pointer is not 16-byte aligned";
    case ADSP_ERR_UNSUPPORTED: return "unsupported parameter combination";
    case ADSP_ERR_WORKSPACE: return "workspace missing, misaligned or too small";
    case ADSP_ERR_LAUNCH: return "HIP launch failed";
    case ADSP_ERR_TOO_LARGE: return "problem needs more scratch than the allocation-free entry point holds";
  }
  return "unknown status";
}
