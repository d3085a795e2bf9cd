// The launchers of the entmax rows kernels, one pair per element type (entmax_rows_unit.hip, compiled once per type).
#pragma once
#include <hip/hip_runtime.h>

namespace adsp {
#define ADSP_ROWS_DECL(tag)                                                                                           \
  void launch_rows_fwd_##tag(const void* x, void* y, long long rows, long long cols, double alpha, hipStream_t s);    \
  void launch_rows_bwd_##tag(const void* y, const void* dy, void* dx, long long rows, long long cols, double alpha, hipStream_t s);
ADSP_ROWS_DECL(f32)
ADSP_ROWS_DECL(bf16)
ADSP_ROWS_DECL(f16)
}  // namespace adsp
