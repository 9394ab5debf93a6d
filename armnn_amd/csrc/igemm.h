// Launches of the register-staged implicit GEMM (IgemmKernel, conv_kernels.h).
#pragma once

#include "plan.h"

namespace mi355x
{

// `tile`: 64, 96 (128 x 64) or anything else (128 x 128, 128 x 64 for at most 64 output channels).  `p` is a MI355X_ALGO_MFMA plan.
int LaunchIgemm(const mi355x_conv2d_s* p, int tile, uint32_t batch, const void* x, void* y, hipStream_t stream);

} // namespace mi355x
