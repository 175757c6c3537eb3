// What the FP8 weight kernels share: the parameter block and the weight-scale lookup.
#pragma once

#include "common.h"

namespace cm {

struct VecmatParams {
  const void* x;
  const float* scale_x;
  const unsigned char* w;
  const float* scale_w;
  void* out;
  float* partial;          // [splits][M][N] fp32 (kernels that split K)
  int m, n, k;
  int x_dtype, out_dtype;
  int srow_shift;          // scale row index = n >> srow_shift
  int srow_stride;         // floats between scale rows
  int scol_stride;         // floats between 128-wide K blocks (0 or 1)
  int rows_per_wg;
  int k_splits;
};

__device__ __forceinline__ float wscale(const VecmatParams& p, int n, int kb) {
  return p.scale_w[(size_t)(n >> p.srow_shift) * p.srow_stride + (size_t)kb * p.scol_stride];
}

// The tiled GEMM for more activation rows than the streaming kernels are made for (fp8_gemm.hip).
bool fp8_gemm_shape(const cppmega_mi355_vecmat_args_t& a);
size_t fp8_gemm_workspace_bytes(const cppmega_mi355_vecmat_args_t& a);
int fp8_gemm_launch(VecmatParams p, size_t workspace_bytes, hipStream_t stream);      // with fewer K splits where they do not fit
int device_cus();

}  // namespace cm
