// One translation unit per (16-bit type, head dim) of attn_bwd16_kernel.h, compiled with -DADSP_T=<bf16_t|f16_t>
// -DADSP_TAG=<bf16|f16> -DADSP_D=<head dim>.
#include "attn_bwd16_kernel.h"

#define ADSP_CAT_(n, a, d) n##a##_d##d
#define ADSP_CAT(n, a, d) ADSP_CAT_(n, a, d)

namespace adsp {
using namespace bwd16;

template <int AM, int P, bool kSplit> static void launch_dq(const AttnBwdParams& p, hipStream_t s) {
  const long long blocks = (p.N + 128 / P - 1) / (128 / P);
  hipLaunchKernelGGL((attn_bwd16_dq_kernel<ADSP_T, ADSP_D, AM, P, kSplit>), dim3(xcd_grid((long long)p.B * p.Hkv, blocks * (p.Hq / p.Hkv))), dim3(256), 0, s, p);
}
template <int AM, int P> static void launch_dkdv(const AttnBwdParams& p, hipStream_t s) {
  const long long blocks = (p.N + 128 / P - 1) / (128 / P);
  hipLaunchKernelGGL((attn_bwd16_dkdv_kernel<ADSP_T, ADSP_D, AM, P>), dim3(xcd_grid((long long)p.B * p.Hkv, blocks)), dim3(256), 0, s, p);
}
// Parts a row's walk is split in: as few as give every CU a workgroup of 128 / parts rows.  Training, us for 1, 2 and 4 parts: 16 x 12
// heads, N <= 500, D = 64: 112, 114, 140; 4 x 16, N = 512, D = 128: 86, 93, 131; 8 x 8, N <= 300, D = 128: 81, 71, 79; dQ's rows 32000 and dK/dV's
// 8000 (2 x 16/4, N <= 1000, D = 64): 138, 111, 110.
// Where the kernels stand in for those on the supports, which add up an item of a batch in the same order whatever the batch is, so do
// these: the rows are those of an item then, and the lines lie where a batch of sixteen does not lose what a single item gains.
// Training, flat scores, causal, us, one part from 16384 rows of an item and two from 4096 against 8192 and 2048 (the kernels before):
// 8 heads, N <= 1383, D = 128, 1, 4 and 16 items: 107 (137), 283 (335), 510 (474) against 105, 246, 421; 16/4 heads, N <= 2600, D = 64,
// 1 and 4: 365 (675), 427 (711) against 426, 482; 4 heads, N <= 900, D = 128, 1 and 16: 74 (94), 323 (255) against 73, 228.
static int parts_of(long long heads, int B, int N, bool split) {
  const long long rows = heads * N;
  if (split) return rows * B >= 256ll * 128 ? 1 : (rows * B >= 256ll * 64 ? 2 : 4);
  return rows >= 64ll * 128 ? 1 : (rows >= 32ll * 64 ? 2 : 4);
}
template <int AM> static void launch(const AttnBwdParams& p, int which, bool split, hipStream_t s) {
  if (which & 1) {
    const int parts = parts_of(p.Hq, p.B, p.N, split);
    if (split) {
      if (parts == 1) launch_dq<AM, 1, true>(p, s);
      else if (parts == 2) launch_dq<AM, 2, true>(p, s);
      else launch_dq<AM, 4, true>(p, s);
    } else {
      if (parts == 1) launch_dq<AM, 1, false>(p, s);
      else if (parts == 2) launch_dq<AM, 2, false>(p, s);
      else launch_dq<AM, 4, false>(p, s);
    }
  }
  if (which & 2) {
    const int parts = parts_of(p.Hkv, p.B, p.N, split);
    if (parts == 1) launch_dkdv<AM, 1>(p, s);
    else if (parts == 2) launch_dkdv<AM, 2>(p, s);
    else launch_dkdv<AM, 4>(p, s);
  }
}
int ADSP_CAT(launch_attn_bwd16_, ADSP_TAG, ADSP_D)(const AttnBwdParams& p, int am, int which, bool split, hipStream_t s) {
  if (am == ATT_15) launch<ATT_15>(p, which, split, s);
  else if (am == ATT_2) launch<ATT_2>(p, which, split, s);
  else launch<ATT_GEN>(p, which, split, s);
  return 0;
}
}  // namespace adsp
