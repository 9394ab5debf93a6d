// Depthwise 3x3 + 1x1 convolution in one launch with the layer between them in LDS (dwpw_panel_kernel.h).
#pragma once

#include "plan.h"

namespace mi355x
{

// Whether the kernel takes the pair; that the layers chain -- shapes, quantization -- is the caller's to check.
bool DwPwPanelTakes(const mi355x_conv2d_s* dw, const mi355x_conv2d_s* pw);

// Builds what the kernel reads of the two plans in an order of its own, where it is not there yet (any thread, also under a graph
// capture: nothing of it goes into the graph).
int PrepareDwPwPanel(const mi355x_conv2d_s* dw, const mi355x_conv2d_s* pw);

// For a pair that has been prepared.
int LaunchDwPwPanel(const mi355x_conv2d_s* dw, const mi355x_conv2d_s* pw, uint32_t batch, const void* x, void* y, hipStream_t stream);

} // namespace mi355x
