// C ABI of the entmax rows kernels: argument checks and the launch for the element type.
#include "entmax_rows.h"
#include "../../include/adasplash_hip.h"

extern "C" int adsp_entmax_rows_fwd(const void* x, void* y, int64_t rows, int64_t cols, int dtype, double alpha,
                                    int n_iter, int use_histogram, int fast_math, void* stream) {
  using namespace adsp;
  // (the solver runs to convergence from a bound of its own: how many steps and from where the reference starts do not matter)
  (void)use_histogram;
  (void)fast_math;
  if (rows < 0 || cols < 0) return ADSP_ERR_SHAPE;
  if (rows == 0 || cols == 0) return ADSP_OK;
  if (!x || !y) return ADSP_ERR_NULL;
  if (!(alpha > 1.0) || n_iter < 0) return ADSP_ERR_UNSUPPORTED;
  if (dtype != ADSP_F32 && dtype != ADSP_BF16 && dtype != ADSP_F16) return ADSP_ERR_DTYPE;
  hipStream_t s = (hipStream_t)stream;
  (void)hipGetLastError();
  if (dtype == ADSP_F32) launch_rows_fwd_f32(x, y, rows, cols, alpha, s);
  else if (dtype == ADSP_BF16) launch_rows_fwd_bf16(x, y, rows, cols, alpha, s);
  else launch_rows_fwd_f16(x, y, rows, cols, alpha, s);
  return hipGetLastError() == hipSuccess ? ADSP_OK : ADSP_ERR_LAUNCH;
}

extern "C" int adsp_entmax_rows_bwd(const void* y, const void* dy, void* dx, int64_t rows, int64_t cols, int dtype,
                                    double alpha, void* stream) {
  using namespace adsp;
  if (rows < 0 || cols < 0) return ADSP_ERR_SHAPE;
  if (rows == 0 || cols == 0) return ADSP_OK;
  if (!y || !dy || !dx) return ADSP_ERR_NULL;
  if (!(alpha > 1.0)) return ADSP_ERR_UNSUPPORTED;
  if (dtype != ADSP_F32 && dtype != ADSP_BF16 && dtype != ADSP_F16) return ADSP_ERR_DTYPE;
  hipStream_t s = (hipStream_t)stream;
  (void)hipGetLastError();
  if (dtype == ADSP_F32) launch_rows_bwd_f32(y, dy, dx, rows, cols, alpha, s);
  else if (dtype == ADSP_BF16) launch_rows_bwd_bf16(y, dy, dx, rows, cols, alpha, s);
  else launch_rows_bwd_f16(y, dy, dx, rows, cols, alpha, s);
  return hipGetLastError() == hipSuccess ? ADSP_OK : ADSP_ERR_LAUNCH;
}
