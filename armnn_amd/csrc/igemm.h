// Launches of the register-staged implicit GEMM (IgemmKernel, conv_kernels.h).
#pragma once

#include "plan.h"

namespace mi355x
{

// `tile`: 64, 96 (128 x 64) or anything else (128 x 128, 128 x 64 for at most 64 output channels).  `p` is a MI355X_ALGO_MFMA plan.
int LaunchIgemm(const mi355x_conv2d_s* p, int tile, uint32_t batch, const void* x, void* y, hipStream_t stream);

// The weights of an MFMA plan in operand order (PackFragKernel) as a new device array; waits for it (an UploadScope must be open).
int PackFragments(const mi355x_conv2d_s* p, bool interleave, int8_t** out);

// Whether a launch of some batch reads an MFMA plan's w_frag.
bool FragmentsWanted(const mi355x_conv2d_s* p);

// SmallConvKernel (small_conv_kernel.h) for a plan with w_frag.  res / add: an Addition behind the layer (output channels
// % 16 == 0, aligned tensors), or null.
int LaunchSmallConv(const mi355x_conv2d_s* p, uint32_t batch, const void* x, void* y, const uint8_t* res, const AddFuse* add, hipStream_t stream);

// RowPanelKernel (row_panel_kernel.h) for a 1x1 plan with w_frag; res / add as above, any output channels % 16 == 0.
int LaunchRowPanel(const mi355x_conv2d_s* p, uint32_t batch, const void* x, void* y, const uint8_t* res, const AddFuse* add, hipStream_t stream);

} // namespace mi355x
