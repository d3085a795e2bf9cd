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
// 8000 (2 x 16/4, N <= 1000, D = 64): 138, 111, 110.  Where the kernels stand in for those on the supports, which add up an item of a
// batch in the same order whatever the batch is, so do these: the rows are those of an item then (flat scores, 32/8 heads,
// N = 4096, D = 128: 1308, 1247 and with dQ in one part and dK/dV in two 1143; 4 x 16/4, N <= 1000, D = 128: 309, 270, 311).
static int parts_of(long long heads, int B, int N, bool split) {
  const long long rows = heads * N;
  if (split) return rows * B >= 256ll * 128 ? 1 : (rows * B >= 256ll * 64 ? 2 : 4);
  return rows >= 128ll * 128 ? 1 : (rows >= 64ll * 64 ? 2 : 4);
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
