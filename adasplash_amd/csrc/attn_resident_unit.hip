// One translation unit per (16-bit type, head dim) of the forward with resident scores (attn_resident_kernel.h), compiled with
// -DADSP_T=<bf16_t|f16_t> -DADSP_TAG=<bf16|f16> -DADSP_D=<head dim>.
#include "attn_resident_kernel.h"

#define ADSP_CAT_(n, a, d) n##a##_d##d
#define ADSP_CAT(n, a, d) ADSP_CAT_(n, a, d)

namespace adsp {
using namespace resident;

template <int AM, int W> static void launch_one(const AttnParams& p, hipStream_t s) {
  const dim3 grid(xcd_grid((long long)p.B * p.Hkv, (long long)((p.N + kRows - 1) / kRows) * (p.Hq / p.Hkv)));
  hipLaunchKernelGGL((attn_resident_fwd_kernel<ADSP_T, ADSP_D, AM, W>), grid, dim3(64 * W), 0, s, p);
}
// the fewest waves whose registers hold the longest rows (kMaxWaves of them: kResidentMaxKeys)
template <int AM> static void launch_fwd(const AttnParams& p, hipStream_t s) {
  if (p.N <= kRows * kBlocks * 4) launch_one<AM, 4>(p, s);
  else if (p.N <= kRows * kBlocks * 8) launch_one<AM, 8>(p, s);
  else launch_one<AM, kMaxWaves>(p, s);
}
int ADSP_CAT(launch_attn_resident_fwd_, ADSP_TAG, ADSP_D)(const AttnParams& p, int am, hipStream_t s) {
  if (p.N > kResidentMaxKeys) return -1;
  if (am == ATT_15) launch_fwd<ATT_15>(p, s);
  else if (am == ATT_2) launch_fwd<ATT_2>(p, s);
  else launch_fwd<ATT_GEN>(p, s);
  return 0;
}
}  // namespace adsp
