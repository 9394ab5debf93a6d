// Launches of the kernel that holds its weights in registers (held_conv_kernel.h).
#pragma once

#include "plan.h"

namespace mi355x
{

// Whether the kernel can run launches of a MI355X_ALGO_MFMA plan with w_frag.
bool HeldConvTakes(const mi355x_conv2d_s* p);

// The groups of 16 outputs that a block of a launch of a MI355X_ALGO_MFMA plan works on (1 to 1024; tensors aligned to 16 bytes); 0 where the kernel does not
// take the launch or another one is faster.
int HeldConvGroups(const mi355x_conv2d_s* p, uint32_t batch);

// `groups`: of HeldConvGroups.
int LaunchHeldConv(const mi355x_conv2d_s* p, int groups, uint32_t batch, const void* x, void* y, hipStream_t stream);

} // namespace mi355x
