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

// What the SAT weights' backward pass refuses
int sat_weight_grad_check(const n2d2hip_sat_weight_grad_item& t);
// The gradient of a weight from that of its level, ref: SATQuantizer_Frame_Kernels.cpp:349-404.  inv_factor: 1 over the largest |tanh| times the
// scaling; mode_factor: the slope of the quantizer's line, 0: none
__device__ __forceinline__ float sat_weight_gradient(float w, float dq, float inv_factor, float mode_factor)
{
    const float inv_cosh = 1.0f / coshf(w);
    float grad = __fmul_rn(__fmul_rn(inv_cosh, inv_cosh), inv_factor);
    if (mode_factor != 0.0f)
        grad = __fmul_rn(grad, mode_factor);
    return __fmul_rn(dq, grad);
}
__device__ __forceinline__ float sat_weight_inv_factor(const n2d2hip_sat_weight_grad_item& t)
{
    return 1.0f / (t.apply_scaling ? __fmul_rn(t.stats[0], t.stats[1]) : t.stats[0]);
}
// ref: SATQuantizerCell_Frame.cpp:249-283: Asymmetric and FullRange have their own slope factor
inline float sat_weight_mode_factor(const n2d2hip_sat_weight_grad_item& t)
{
    if (t.mode == N2D2HIP_SAT_FULLRANGE) return 1.0f + 0.9998f / t.range;
    if (t.mode != N2D2HIP_SAT_ASYMRANGE && t.mode != N2D2HIP_SAT_NONE_ASYM) return 0.0f;
    const float r2 = floorf(t.range / 2.0f);
    return 1.0f + 1.0f / (2.0f * r2);
}

} // namespace n2d2hip
