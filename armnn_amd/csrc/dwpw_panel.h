// Depthwise 3x3 + 1x1 convolution in one launch with the layer between them in LDS (dwpw_panel_kernel.h).
#pragma once

#include "plan.h"

namespace mi355x
{

// Whether the kernel takes the pair; that the layers chain -- shapes, quantization -- is the caller's to check.
bool DwPwPanelTakes(const mi355x_conv2d_s* dw, const mi355x_conv2d_s* pw);

int LaunchDwPwPanel(const mi355x_conv2d_s* dw, const mi355x_conv2d_s* pw, uint32_t batch, const void* x, void* y, hipStream_t stream);

} // namespace mi355x
