// What a run of fully-connected cells holds (shared by the translation units that launch it alone and behind other cells).
#pragma once

#include "common.h"

namespace n2d2hip {

enum { FC_CHAIN_MAX = 3, FC_CHAIN_K4 = 256 /* dwords of K per cell at most */, FC_CHAIN_O = 128 };

} // namespace n2d2hip

struct n2d2hip_fc_chain_s {
    int n;
    n2d2hip_fc_t fc[n2d2hip::FC_CHAIN_MAX];
    unsigned* d_wt[n2d2hip::FC_CHAIN_MAX];      // [K / 4][128] dwords: the four weights of output o for bytes 4k .. 4k + 3
    std::vector<unsigned> hwt[n2d2hip::FC_CHAIN_MAX];       // the same on the host
    int k4[n2d2hip::FC_CHAIN_MAX];
};
