// One translation unit per (16-bit type, head dim) of the forward kernel on 32 rows a workgroup (attn_f32_kernel.h), compiled
// with -DADSP_T=<bf16_t|f16_t> -DADSP_TAG=<bf16|f16> -DADSP_D=<head dim>.
#include "attn_f32_kernel.h"

#define ADSP_CAT_(a, d) launch_attn_rows32_##a##_d##d
#define ADSP_CAT(a, d) ADSP_CAT_(a, d)

namespace adsp {
using namespace f32path;
template <int AM> static void launch(const AttnParams& p, hipStream_t s) {
  hipLaunchKernelGGL((attn_rows32_fwd_kernel<ADSP_T, ADSP_D, AM>), dim3(xcd_grid((long long)p.B * p.Hkv, (long long)((p.N + kRows - 1) / kRows) * (p.Hq / p.Hkv))),
                     dim3(256), 0, s, p);
}
int ADSP_CAT(ADSP_TAG, ADSP_D)(const AttnParams& p, int am, hipStream_t s) {
  if (am == ATT_15) launch<ATT_15>(p, s);
  else if (am == ATT_2) launch<ATT_2>(p, s);
  else launch<ATT_GEN>(p, s);
  return 0;
}
}  // namespace adsp
