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
// The quantizer behind a kernel that writes a tensor: fp receives what goes into it (or null), the output what comes out;
// alpha null: no quantizer
struct SatStore {
    float* fp;
    float range;
    const float* alpha;
};
// Its derivatives by alpha and by its input, ref: SATQuantizer_Frame_Kernels.cpp:410-448
__device__ __forceinline__ float sat_alpha_slope(float v, float range, float a)
{
    const float xc = (v < 0.0f) ? 0.0f : (v < a) ? v : a;
    const float q = xc / a;
    const float qd = round_half_away(__fmul_rn(range, q)) / range;
    return (v >= a) ? 1.0f : __fsub_rn(qd, q);
}
__device__ __forceinline__ float sat_input_slope(float v, float a) { return (v <= 0.0f) ? 0.0f : (v > a) ? 0.0f : 1.0f; }

} // namespace n2d2hip
