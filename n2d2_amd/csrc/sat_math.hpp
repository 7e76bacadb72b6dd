// The SAT activation quantizer of one value, for its own kernel and for the normalisation that applies it on the way out.
#pragma once

#include <hip/hip_runtime.h>

#include "epilogue.hpp"

namespace n2d2hip {

// a: |alpha|.  ref: src/Quantizer/QAT/Kernel/SATQuantizer_Frame_Kernels.cpp:268-322 (std::round: half away from zero)
__device__ __forceinline__ float sat_quantize(float v, float range, float a)
{
    const float xc = (v < 0.0f) ? 0.0f : (v < a) ? v : a;
    float q = xc / a;
    q = round_half_away(__fmul_rn(range, q)) / range;
    return __fmul_rn(q, a);
}

} // namespace n2d2hip
