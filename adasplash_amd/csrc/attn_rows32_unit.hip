// One translation unit per (16-bit type, head dim) of the forward on 32 rows a workgroup (attn_f32_kernel.h), compiled with
// -DADSP_T=<bf16_t|f16_t> -DADSP_TAG=<bf16|f16> -DADSP_D=<head dim>.
#include "attn_f32_kernel.h"

#define ADSP_CAT_(n, a, d) n##a##_d##d
#define ADSP_CAT(n, a, d) ADSP_CAT_(n, a, d)

namespace adsp {
using namespace f32path;
static dim3 grid_of(int B, int Hkv, int group, int N) { return dim3(xcd_grid((long long)B * Hkv, (long long)((N + kRows - 1) / kRows) * group)); }

template <int AM> static void launch_fwd(const AttnParams& p, hipStream_t s) {
  hipLaunchKernelGGL((attn_rows32_fwd_kernel<ADSP_T, ADSP_D, AM>), grid_of(p.B, p.Hkv, p.Hq / p.Hkv, p.N), dim3(256), 0, s, p);
}
int ADSP_CAT(launch_attn_rows32_fwd_, ADSP_TAG, ADSP_D)(const AttnParams& p, int am, hipStream_t s) {
  if (am == ATT_15) launch_fwd<ATT_15>(p, s);
  else if (am == ATT_2) launch_fwd<ATT_2>(p, s);
  else launch_fwd<ATT_GEN>(p, s);
  return 0;
}
}  // namespace adsp
