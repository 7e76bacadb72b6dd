// Interface between the two kernels that run a 3x3 depthwise convolution and the 1x1 convolution that reads it in one launch,
// dw_pw.hip for many pixels and dw_pw_small.hip for few: what they take, from the cells alone, and where the first is faster
// than the cells' own launches.
#pragma once

#include "conv_handle.hpp"

namespace n2d2hip {

bool dw_pw_takes(const n2d2hip_conv_s* dw, const n2d2hip_conv_s* pw);
bool dw_pw_small_takes(const n2d2hip_conv_s* dw, const n2d2hip_conv_s* pw);
bool dw_pw_wins(int C, int O, int batch, int OH, int OW);

inline int byte_type_of(const n2d2hip_act_s* a) { return a->min_out >= 0 ? N2D2HIP_U8B : N2D2HIP_I8; }
inline bool plain_1x1(const n2d2hip_conv_desc& d)
{
    return d.kW == 1 && d.kH == 1 && d.strideX == 1 && d.strideY == 1 && d.padL == 0 && d.padT == 0 && d.padR == 0 && d.padB == 0
        && d.dilX == 1 && d.dilY == 1 && d.groups == 1 && d.weight_bits == 8;
}
// (undilated, of stride 1 or 2, over channels that make whole chunks)
inline bool plain_3x3_depthwise(const n2d2hip_conv_s* dw)
{
    const n2d2hip_conv_desc& d = dw->desc;
    return dw->depthwise && dw->d_wdw && d.kW == 3 && d.kH == 3 && d.dilX == 1 && d.dilY == 1 && d.strideX == d.strideY && (d.strideX == 1 || d.strideX == 2)
        && dw->act->cpad >= d.C && dw->in_cs == d.C && (d.C == 32 || d.C % 64 == 0) && (int)dw->act->htab.size() >= 5 * dw->act->cpad;
}

} // namespace n2d2hip
