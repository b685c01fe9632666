// Launchers of dense_solve_kernels.hip: whole dense matrices factored and solved on one wavefront per
// world.  IM_ERR_UNSUPPORTED, with nothing launched, for sizes they do not take.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace im {

int blocked_solve_wave(const float *M, int64_t ldM, int nM, const int32_t *block_idx, int block_size, int nv, int pad, const float *y,
                       int64_t ldy, float *U, float *x, int64_t ldx, const int32_t *active, int nworld, hipStream_t stream);
int jtdj_solve_wave(const float *Mdense, const float *J, int njmax, const float *D, const int32_t *state, const int32_t *nefc, int quad,
                    float *H, int nv, int nv_pad, const float *y, int64_t ldy, float *U, int pad, float *x, int64_t ldx, int nworld,
                    hipStream_t stream);

}  // namespace im
