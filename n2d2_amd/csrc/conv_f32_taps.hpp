// Float32 convolution, forward and backward-data, on the bf16 matrix cores with every operand in three parts (conv_f32_patch.hpp), where no
// run of source positions serves a tile: 1x1 kernels, strided backward-data, strided kernels on long rows, and few rows of q.
//
// K goes in steps of 32 products.  A wave loads 8 of a step's rows of k for all pixels of the tile, a pixel to a lane, takes them apart and
// leaves them in LDS, 16 bytes to 8 products of a pixel; the weights, taken apart and laid out before, come from the L2 as fragments.
// Two steps are in LDS and one more on its way in registers, so that a step costs one barrier.  Where padding the channels to 32 costs
// less than a fifth a step is 32 channels at one tap (CHUNK: a load's test whether its tap lies inside the source is one for all); else its
// products are consecutive ones of (channel, tap).  All residue classes of a strided backward-data are one launch, as in the chunk kernel.
//
// us, fp32 matrix cores (chunk, pixel and 3x3 kernel) / now, with the launches that lay the weights out and add ranges, error against 64 bits:
//   forward 164 -> 377, 5x5 stride 2, 9 x 85, batch 16    214 /  98    3.6e-7 / 2.5e-7
//   forward 17 -> 253, 5x5, 105 x 98, batch 3              85 /  59    3.7e-7 / 1.3e-7
//   forward 37 -> 90, 3x3, 112 x 75, batch 64             409 / 310
//   forward 256 -> 64, 1x1, 56 x 56, batch 64              73 /  60    2.9e-7 / 1.0e-7
//   data 164 <- 53, 5x5, 105 x 98, batch 3                210 / 130
//   data 13 <- 20, 5x5, 61 x 82, batch 107                235 / 188
//   data 128 <- 256, 3x3 stride 2, 27 x 27, batch 33       55 /  47    2.4e-7 / 1.7e-7
//   data 64 <- 256, 1x1, 56 x 56, batch 64                 76 /  63    2.9e-7 / 1.0e-7
// A step of a 64 x 64 tile is 384 cycles of matrix instructions and some 400 of others, a third of which take the floats apart: what a SIMD's waves
// overlap of the two is what bounds it, and with a block or two to a CU (the last: 102, 188 and 88 tiles of 32, 16 and 8 steps x 2) the latency of
// a step, 0.5 to 1 us.  (Two steps of weights ahead, three in registers; eight waves that share K; 64 x 128 tiles: the same or slower.)
#pragma once

#include "conv_f32_patch.hpp"

namespace n2d2hip {

// Product k = 32 step + j of a class: its channel and tap (ch >= Ch: none)
template <bool CHUNK>
__device__ __forceinline__ void taps_product(const PixelGemm& g, const PixelClass& c, int step, int j, int* ch, int* t)
{
    if (CHUNK) {
        const int chunk = div_f32(step, c.nt);
        *t = step - chunk * c.nT;
        *ch = chunk * PK + j;
    } else {
        const int k = step * PK + j;
        *ch = div_f32(k, c.nt);
        *t = k - *ch * c.nT;
    }
}
__device__ __forceinline__ int taps_weight(const PixelGemm& g, const PixelClass& c, int q, int ch, int t)
{
    const int i = div_f32(t, c.nxd), j = t - i * c.nx;
    return q * g.qs + ch * g.chs + (c.ty0 + i * g.osy) * g.kW + c.tx0 + j * g.osx;
}

// Weights as the matrix instructions take them: [class][step][16 rows of q][part][lane][8 products]; what does not exist is zero.
template <bool CHUNK>
__global__ __launch_bounds__(256) void conv_f32_lay_taps_kernel(PixelGemm g, const float* __restrict__ w, v4u* __restrict__ wt, int total)
{
    const int nq = g.qpad / 16;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256) {
        const int lane = i & 63, frag = __builtin_amdgcn_readfirstlane(i >> 6), row = frag / nq, qb = frag - row * nq;
        int ci = 0;                              // (scalar: by lane, the class's fields would be loads that wait for each other)
#pragma unroll
        for (int k = 1; k < PIXEL_CLASSES; ++k)
            if (k < g.nclass && row >= g.c[k].w0) ci = k;
        const PixelClass& c = g.c[ci];
        const int q = qb * 16 + (lane & 15);
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            int ch, t;
            taps_product<CHUNK>(g, c, row - c.w0, 8 * (lane >> 4) + j, &ch, &t);
            v[j] = q < g.Q && ch < g.Ch ? w[taps_weight(g, c, q, ch, t)] : 0.0f;
        }
        v4u parts[3];
        bf16_parts(v, parts);
#pragma unroll
        for (int p = 0; p < 3; ++p) wt[(size_t)frag * (PATCH_FRAG / 16) + p * 64 + lane] = parts[p];
    }
}

// A tile is 16 MQ WQ rows of q x 16 NP WP pixels of a class.
template <int WQ, int WP, int MQ, int NP, bool CHUNK, bool FOLD>
__global__ __launch_bounds__(256, 2) void conv_f32_taps_kernel(PixelGemm g, const float* __restrict__ srcX, const float* __restrict__ srcW,
                                                               const v4u* __restrict__ wt, const float* __restrict__ bias, float beta,
                                                               float* __restrict__ out, size_t partial)
{
    static_assert(WQ * WP == 4, "four waves, one to 8 products of a step");
    constexpr int QT = 16 * MQ * WQ, PT = 16 * NP * WP, PH = PT / 64;
    constexpr int OCT = PT * 16, PART = 4 * OCT, STAGE = 3 * PART;
    __shared__ __attribute__((aligned(16))) char smem[2 * STAGE];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, lo = lane >> 4, wq = wave / WP, wp = wave % WP;
    int tile, qtile, ci;
    if (!pixel_tile(g, &tile, &qtile, &ci))
        return;
    const PixelClass& c = g.c[ci];
    const int p0 = (tile - c.tile0) * PT, q0 = qtile * QT, nT = c.nT, plane4 = g.planeS * 4, K = g.Ch * nT;
    const int steps = CHUNK ? (g.Ch + PK - 1) / PK * nT : (K + PK - 1) / PK;
    const int beg = blockIdx.z * c.kchunk, end = min(beg + c.kchunk, steps);
    const __amdgpu_buffer_rsrc_t rsrcX = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(srcX) - c.bias, 0, g.bytesX + 4u * c.bias, 0x00020000);
    const int nq = g.qpad / 16;
    const __amdgpu_buffer_rsrc_t rsrcW = __builtin_amdgcn_make_buffer_rsrc(const_cast<v4u*>(wt) + (size_t)c.w0 * nq * (PATCH_FRAG / 16), 0,
                                                                           steps * nq * PATCH_FRAG, 0x00020000);
    unsigned voff[PH];
    TapMask<false> mask[PH];
#pragma unroll
    for (int h = 0; h < PH; ++h)
        pixel_source(g, c, p0 + h * 64 + lane, &voff[h], &mask[h]);
    // tap t lives in lane t, as in the other kernels
    const int tl = min(lane, max(nT - 1, 0)), ti = div_f32(tl, c.nxd), tj = tl - ti * c.nx;
    const int tap_off = 4 * (c.soff0 + ti * c.stepy + tj * c.stepx), tap_bit = (1 << tj) | (1 << (c.nx + ti));

    // ---- the step to load next: its tap (CHUNK), or the tap and channel of each of the wave's rows
    int row_t[CHUNK ? 1 : 8], row_ch[CHUNK ? 1 : 8];         // row_ch: the channel's byte offset
    int left;                                                // channels (CHUNK) or products behind the wave's first row
    const int adv = nT > 0 ? div_f32(PK, c.nt) : 0, adv_t = PK - adv * nT;
    {
        int ch = 0, t = 0;
        if (nT > 0) taps_product<CHUNK>(g, c, beg, 8 * wave, &ch, &t);
        left = CHUNK ? g.Ch - ch : K - beg * PK - 8 * wave;
#pragma unroll
        for (int r = 0; r < (CHUNK ? 1 : 8); ++r) {
            row_t[r] = t; row_ch[r] = ch * plane4;
            if (++t >= nT) { t = 0; ++ch; }
        }
    }
    float v[2][PH][8];
    int ahead = end - beg;                                   // steps not yet requested; past the last one zeros are
    auto load = [&](auto set_) {
        constexpr int set = decltype(set_)::value;
        const int there = ahead > 0 ? left : 0;
        --ahead;
        if constexpr (CHUNK) {
            const unsigned bit = (unsigned)__builtin_amdgcn_readlane(tap_bit, row_t[0]);
            const int soff = row_ch[0] + __builtin_amdgcn_readlane(tap_off, row_t[0]);
            unsigned at[PH];
#pragma unroll
            for (int h = 0; h < PH; ++h) at[h] = mask[h].inside(row_t[0], bit) ? voff[h] : F32_OOB;
#pragma unroll
            for (int r = 0; r < 8; ++r)
#pragma unroll
                for (int h = 0; h < PH; ++h)
                    v[set][h][r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrcX, at[h], r < there ? soff + r * plane4 : 0x7ffffffc, 0));
            if (++row_t[0] >= nT) {
                row_t[0] = 0;
                row_ch[0] += PK * plane4;
                left -= PK;
            }
        } else {
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                const int t = row_t[r];
                const unsigned bit = tap_test<false>(t, tap_bit, there - 1 - r);
                const int soff = row_ch[r] + __builtin_amdgcn_readlane(tap_off, t);
#pragma unroll
                for (int h = 0; h < PH; ++h)
                    v[set][h][r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrcX, mask[h].inside(t, bit) ? voff[h] : F32_OOB, soff, 0));
                const int tn = t + adv_t;
                const bool carry = tn >= nT;
                row_t[r] = carry ? tn - nT : tn;
                row_ch[r] += adv * plane4 + (carry ? plane4 : 0);
            }
            left -= PK;
        }
    };
    auto put = [&](auto set_, int h) {
        constexpr int set = decltype(set_)::value;
        v4u parts[3];
        bf16_parts(v[set][h], parts);
#pragma unroll
        for (int p = 0; p < 3; ++p) *(v4u*)(smem + set * STAGE + p * PART + wave * OCT + (h * 64 + lane) * 16) = parts[p];
    };
    const bool live = q0 + wq * MQ * 16 < g.Q;
    v4u a[2][MQ][3];
    auto weights = [&](auto set_, int step) {
        const int at = (step * nq + qtile * (QT / 16) + wq * MQ) * PATCH_FRAG;
#pragma unroll
        for (int m = 0; m < MQ; ++m)
#pragma unroll
            for (int p = 0; p < 3; ++p)
                a[decltype(set_)::value][m][p] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(rsrcW, lane * 16, at + m * PATCH_FRAG + p * 1024, 0));
    };
    v4f acc[MQ][NP];
    double folded[FOLD ? MQ : 1][NP][4];
    auto each = [&](auto&& f) {
#pragma unroll
        for (int m = 0; m < MQ; ++m)
#pragma unroll
            for (int n = 0; n < NP; ++n)
#pragma unroll
                for (int r = 0; r < 4; ++r) f(m, n, r);
    };
    each([&](int m, int n, int r) {
        acc[m][n][r] = 0.0f;
        if (FOLD) folded[m][n][r] = 0.0;
    });
    auto fold = [&]() {
        each([&](int m, int n, int r) { folded[m][n][r] += (double)acc[m][n][r]; acc[m][n][r] = 0.0f; });
    };
    const char* const pixels = smem + lo * OCT + (wp * NP * 16 + l16) * 16;
    int until = FOLD ? c.fold : 0;
    // One step, from the LDS half and the weights of `set`: meanwhile the next one's values are taken apart into the other half and those of
    // the one behind it requested.  (Without a condition, also past the end: where paths of more and of fewer loads meet, the compiler waits
    // as if the fewer had been issued, for all of them.)
    auto step = [&](auto set_, int s) {
        constexpr int set = decltype(set_)::value;
        using Other = std::integral_constant<int, 1 - set>;
        __syncthreads();
        weights(Other{}, s + 1);
        load(set_);
        // (rows past the last, too: their weights are zero, and with a branch here the compiler does first in both of its ways what they have in
        // common, which waits for the loads)
#pragma unroll
        for (int n = 0; n < NP; ++n) {
            v4u x[3];
#pragma unroll
            for (int p = 0; p < 3; ++p) x[p] = *(const v4u*)(pixels + set * STAGE + p * PART + n * 256);
            v4f small[MQ];
#pragma unroll
            for (int m = 0; m < MQ; ++m) small[m] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                constexpr int pa[5] = {1, 0, 2, 0, 1}, pb[5] = {1, 2, 0, 1, 0};
#pragma unroll
                for (int m = 0; m < MQ; ++m)
                    small[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a[set][m][pa[k]]), __builtin_bit_cast(v8bf, x[pb[k]]), small[m], 0, 0, 0);
            }
#pragma unroll
            for (int m = 0; m < MQ; ++m)
                acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a[set][m][0]), __builtin_bit_cast(v8bf, x[0]), acc[m][n], 0, 0, 0);
            if (n >= NP - PH) {
                __builtin_amdgcn_sched_barrier(0);
                put(Other{}, n - (NP - PH));
            }
#pragma unroll
            for (int m = 0; m < MQ; ++m)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[m][n][r] += small[m][r];
        }
        if (FOLD && --until == 0) {
            fold();
            until = c.fold;
        }
    };
    static_assert(PH <= NP, "a wave's part of the next step between its products");
    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    if (beg < end) {
        load(S0{});
        weights(S0{}, beg);
        load(S1{});
#pragma unroll
        for (int h = 0; h < PH; ++h) put(S0{}, h);
        for (int s = beg; s < end; s += 2) {
            step(S0{}, s);
            step(S1{}, s + 1);
        }
    }
    if (!live) return;
    if (FOLD) fold();
    float finite = 0.0f;
    each([&](int m, int n, int r) {
        if constexpr (FOLD) acc[m][n][r] = (float)(folded[m][n][r] * (double)PARTS_UNSCALE);
        else acc[m][n][r] *= PARTS_UNSCALE;
        finite = __builtin_fmaf(acc[m][n][r], 0.0f, finite);
    });
    if (__any(finite != finite)) {
        // Infinities, and what rounds to one in bf16, leave NaN where float products might not: a wave that holds such sums adds them again, on the
        // fp32 matrix cores straight from memory, in double from one step to the next.
        // us, data 128 <- 256, stride 2, finite 47; NaN throughout 333; one weight NaN 306; 164 -> 377, 5x5 stride 2, 104; 1517; 869.
        int here = lane;                         // (opaque: nothing of this is worked out ahead, and held, by waves that never come here)
        asm volatile("" : "+v"(here));
        const int l16 = here & 15, lo = here >> 4;
        const __amdgpu_buffer_rsrc_t rsrcV = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(srcW), 0, g.bytesW, 0x00020000);
#pragma unroll
        for (int n = 0; n < NP; ++n) {
            unsigned from;
            TapMask<false> there;
            pixel_source(g, c, p0 + (wp * NP + n) * 16 + l16, &from, &there);
            double sum[MQ][4] = {};
#pragma unroll 1
            for (int s = beg; s < end; ++s) {
                v4f part[MQ];
#pragma unroll
                for (int m = 0; m < MQ; ++m) part[m] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
                for (int j = 0; j < PK; j += 4) {
                    int ch, t;
                    taps_product<CHUNK>(g, c, s, j + lo, &ch, &t);
                    const bool is = ch < g.Ch;
                    const int i = div_f32(t, c.nxd), jx = t - i * c.nx;
                    const unsigned bit = (1u << jx) | (1u << (c.nx + i));
                    const float x = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                        rsrcX, is && (there.m & bit) == bit ? from + 4u * (unsigned)(c.soff0 + i * c.stepy + jx * c.stepx) + (unsigned)(ch * plane4) : F32_OOB, 0, 0));
#pragma unroll
                    for (int m = 0; m < MQ; ++m) {
                        const int q = q0 + (wq * MQ + m) * 16 + l16;
                        const float w = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                            rsrcV, is && q < g.Q ? 4u * (unsigned)taps_weight(g, c, q, ch, t) : F32_OOB, 0, 0));
                        part[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(w, x, part[m], 0, 0, 0);
                    }
                }
#pragma unroll
                for (int m = 0; m < MQ; ++m)
#pragma unroll
                    for (int r = 0; r < 4; ++r) sum[m][r] += (double)part[m][r];
            }
#pragma unroll
            for (int m = 0; m < MQ; ++m)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (!(__builtin_fabsf(acc[m][n][r]) < __builtin_inff())) acc[m][n][r] = (float)sum[m][r];
        }
    }
    // A lane holds pixel .. + lane % 16 and rows .. + 4 (lane / 16) + r.
    float* const dst = out + (size_t)blockIdx.z * partial;
#pragma unroll
    for (int n = 0; n < NP; ++n) {
        const int p = p0 + (wp * NP + n) * 16 + l16;
        if (p >= c.P) continue;
        const int img = div_f32(p, c.ghw), rem = p - img * c.gHW, py = div_f32(rem, c.gw), px = rem - py * c.gW;
        const size_t base = (size_t)img * g.Q * g.planeO + (py * g.osy + c.ry) * g.Wo + px * g.osx + c.rx;
#pragma unroll
        for (int m = 0; m < MQ; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int q = q0 + (wq * MQ + m) * 16 + 4 * lo + r;
                if (q >= g.Q) continue;
                const size_t idx = base + (size_t)q * g.planeO;
                float s = acc[m][n][r];
                if (partial == 0) {
                    if (beta != 0.0f) s += beta * dst[idx];
                    if (bias) s = bias[q] + s;
                }
                dst[idx] = s;
            }
    }
}

} // namespace n2d2hip
