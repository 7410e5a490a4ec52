/* Entry points that this package's own Python side calls beside those of
 * llattn.h: fused steps of its language model and block.  Same conventions
 * (status codes, llattn_last_error, explicit stream, caller-supplied memory). */
#ifndef LLATTN_STEPS_H
#define LLATTN_STEPS_H

#include "llattn.h"

#ifdef __cplusplus
extern "C" {
#endif

/* llattn_rmsnorm_bwd with dx also written in bf16 (dx16, may be null; needs
 * dres): the gradient of a bf16 residual addend, which autograd holds apart
 * from dx. */
int32_t llattn_rmsnorm_bwd_residual(const void* dy, int32_t dy_dtype, int64_t lddy, const void* x, int32_t x_dtype,
                                    int64_t ldx, const float* rstd, const float* weight, int32_t M, int32_t D,
                                    void* dx, int64_t lddx, float* dweight, const void* dres, int64_t lddres,
                                    void* dx16, int64_t lddx16, void* workspace, size_t workspace_bytes,
                                    void* stream);

#ifdef __cplusplus
}
#endif

#endif
