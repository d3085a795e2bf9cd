// One translation unit per head dim of the single-precision kernels (attn_f32_kernel.h), compiled with -DADSP_D=<head dim>.
#include "attn_f32_kernel.h"

namespace adsp {
using namespace f32path;
#define ADSP_CAT_(a, d) a##d
#define ADSP_CAT(a, d) ADSP_CAT_(a, d)

// one workgroup per 32 rows of each of `group` heads of every (batch, K/V head)
static dim3 grid_of(int B, int Hkv, int group, int N) { return dim3(xcd_grid((long long)B * Hkv, (long long)((N + kRows - 1) / kRows) * group)); }

template <int AM> static void launch_bwd(const AttnBwdParams& p, hipStream_t s) {
  hipLaunchKernelGGL((attn_rows32_dq_kernel<ADSP_D, AM>), grid_of(p.B, p.Hkv, p.Hq / p.Hkv, p.N), dim3(256), 0, s, p);
  hipLaunchKernelGGL((attn_rows32_dkdv_kernel<ADSP_D, AM>), grid_of(p.B, p.Hkv, 1, p.N), dim3(256), 0, s, p);
}
template <int AM> static void launch_fwd(const AttnParams& p, hipStream_t s) {
  hipLaunchKernelGGL((attn_rows32_fwd_kernel<float, ADSP_D, AM>), grid_of(p.B, p.Hkv, p.Hq / p.Hkv, p.N), dim3(256), 0, s, p);
}
int ADSP_CAT(launch_attn_f32_fwd_d, ADSP_D)(const AttnParams& p, int am, hipStream_t s) {
  if (am == ATT_15) launch_fwd<ATT_15>(p, s);
  else if (am == ATT_2) launch_fwd<ATT_2>(p, s);
  else launch_fwd<ATT_GEN>(p, s);
  return 0;
}
int ADSP_CAT(launch_attn_f32_bwd_d, ADSP_D)(const AttnBwdParams& p, int am, hipStream_t s) {
  if (am == ATT_15) launch_bwd<ATT_15>(p, s);
  else if (am == ATT_2) launch_bwd<ATT_2>(p, s);
  else launch_bwd<ATT_GEN>(p, s);
  return 0;
}
}  // namespace adsp
