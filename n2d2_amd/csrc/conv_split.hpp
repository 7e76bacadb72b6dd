// Interface between the convolution host code (conv_igemm.hip) and the kernel for layers of few output tiles (conv_split.hip).
#pragma once

#include "conv_pipe.hpp"

namespace n2d2hip {

// Does the kernel take this layer's shape?  (A multiple of 128 channels, at most 31 taps, no dilation; a rescale on 32-bit
// integers, or none for an unpadded 1x1 layer.  `valid` as conv_pipe_kernel's.)
bool conv_split_takes(const n2d2hip_conv_desc& d, int epi_kind, int valid);
// Is it the faster one for M output pixels and O outputs of `ktot` weights, packed (w4) or not, with a folded sum or without?
bool conv_split_pays(long long M, int O, int ktot, bool w4, bool sum);
// `a` as for conv_pipe_kernel with 64 bytes per K step, its tables not scaled up (neither the rescale's nor the folded
// ScalingCell's); `w4`: a.c.w is the packed image conv_pipe_w4_image() makes; `valid` as there.
int conv_split_launch(ConvPipeArgs a, int valid, bool w4, hipStream_t stream);

} // namespace n2d2hip
