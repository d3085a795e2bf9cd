// One translation unit per (16-bit type, head dim) of attn_fwd16_kernel.h, compiled with -DADSP_T=<bf16_t|f16_t>
// -DADSP_TAG=<bf16|f16> -DADSP_D=<head dim>.
#include "attn_fwd16_kernel.h"

#define ADSP_CAT_(n, a, d) n##a##_d##d
#define ADSP_CAT(n, a, d) ADSP_CAT_(n, a, d)

namespace adsp {
using namespace fwd16;

template <int AM> static void launch(const AttnParams& p, hipStream_t s) {
  const dim3 grid(xcd_grid((long long)p.B * p.Hkv, (long long)((p.N + kMaskRows - 1) / kMaskRows) * (p.Hq / p.Hkv)));
  const size_t mask = p.bmask ? p.mask_words * sizeof(uint32_t) : 0;
  if (p.taus) hipLaunchKernelGGL((attn_fwd16_kernel<ADSP_T, ADSP_D, AM, true>), grid, dim3(256), mask, s, p);
  else hipLaunchKernelGGL((attn_fwd16_kernel<ADSP_T, ADSP_D, AM, false>), grid, dim3(256), mask, s, p);
}
int ADSP_CAT(launch_attn_fwd16_, ADSP_TAG, ADSP_D)(const AttnParams& p, int am, hipStream_t s) {
  if (am == ATT_15) launch<ATT_15>(p, s);
  else if (am == ATT_2) launch<ATT_2>(p, s);
  else launch<ATT_GEN>(p, s);
  return 0;
}
}  // namespace adsp
