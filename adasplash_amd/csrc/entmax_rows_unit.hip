// The entmax rows kernels of one element type (ADSP_T, tag ADSP_TAG).
#include "entmax_rows_kernel.h"
#include "entmax_rows.h"

#define ADSP_CAT2(a, b) a##b
#define ADSP_CAT(a, b) ADSP_CAT2(a, b)

namespace adsp {
void ADSP_CAT(launch_rows_fwd_, ADSP_TAG)(const void* x, void* y, long long rows, long long cols, double alpha, hipStream_t s) {
  RowsParams p;
  p.x = x;
  p.y = y;
  p.rows = rows;
  p.cols = cols;
  p.scale = (float)(alpha - 1.0);
  p.c0 = (float)(1.0 / (alpha - 1.0));
  p.inv_c0 = (float)(alpha - 1.0);
  if (alpha == 1.5) launch_fwd<ADSP_T, AM_15>(p, s);
  else if (alpha == 2.0) launch_fwd<ADSP_T, AM_2>(p, s);
  else launch_fwd<ADSP_T, AM_GEN>(p, s);
}
void ADSP_CAT(launch_rows_bwd_, ADSP_TAG)(const void* y, const void* dy, void* dx, long long rows, long long cols, double alpha,
                                          hipStream_t s) {
  const float cf = (float)(2.0 - alpha);
  if (alpha == 1.5) launch_bwd<ADSP_T, AM_15>(y, dy, dx, rows, cols, cf, s);
  else if (alpha == 2.0) launch_bwd<ADSP_T, AM_2>(y, dy, dx, rows, cols, cf, s);
  else launch_bwd<ADSP_T, AM_GEN>(y, dy, dx, rows, cols, cf, s);
}
}  // namespace adsp
