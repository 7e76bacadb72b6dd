// Float32 convolution, forward, backward-data at stride 1 and of 3x3 kernels at stride 2, on the bf16 matrix cores with every operand in three parts.
//
// A float is the sum of three bf16 numbers without a rest (8 + 8 + 8 bits of mantissa, each part the rounded rest of the ones
// before; scaled, so that the parts of small floats keep their bits): a = a0 + a1 + a2.  Of the nine products of a b, a1 b2 and a2 b1 are
// below 2^-25 of it and a2 b2 below 2^-34: left out, all three are just below 2^-24 of a b at most (a sum of one product that is not zero is off by
// up to 1.9 half units of the last place, a float product by 1.0; the sums of more terms are below).  The other six are matrix
// instructions.  Random data, two waves to a SIMD, register operands only: 16x16x32 bf16 2040 TFLOP/s, 340 of six products; 32x32x16
// bf16 1350 (two waves in turn slow it down; one alone has 1800); 32x32x2 fp32 98.
// An instruction adds its 32 products to the sum in four roundings: the five smaller products have a sum of their own, which one
// addition brings to that of the largest, so that a sum is rounded 5 times in 32 terms where the fp32 instructions round it 32
// times.  Error against 64 bits, random data (forward; before, now): 64 channels, 3x3 4.3e-7, 1.5e-7; 256 channels, 3x3, 14 x 14
// 3.2e-7, 2.2e-7; 48 channels, 5x5 3.0e-7, 1.7e-7.  All six in one sum: 3.6e-7, 3.5e-7, 3.8e-7.
//
// us, forward / data, fp32 matrix cores (conv_f32_3x3_kernel, conv_f32_pixel_kernel), now:
//   64 -> 64, 3x3, 56 x 56, batch 64            139 / 138     93 /  85
//   64 -> 64, 3x3, 32 x 32, batch 64             48 /  49     36 /  35
//   256 -> 256, 3x3, 14 x 14, batch 32          100 /  91     63 /  62
//   512 -> 512, 3x3, 14 x 14, batch 8           115 / 103     80 /  73
//   48 -> 96, 5x5, 30 x 30, batch 16             71 /  64     41 /  43
//   128 -> 256, 3x3 stride 2, 27 x 27, batch 33  53 /         42
//   256 -> 512, 3x3 stride 2, 28 x 28, batch 8      /  75        /  54      (data: four pixels a place, below)
//   128 -> 128, 3x3 stride 2, 56 x 56, batch 64     / 152        / 109
// 64 -> 64 on 56 x 56 is 42 us of matrix instructions at the 2.0 GHz that they leave; what is beside them, in a block's cycles (of
// 160000, two blocks to a CU): 8 steps of 13700 that are matrix instructions of both blocks, 8 x 1700 that take a step's floats
// apart, 4 x 9000 for a tile's results and the next one's addresses, 15000 until the first step is there; and 6.1 tiles to a CU take
// as long as 7.  (Three blocks to a CU with less in flight, 64 x 64 tiles of a wave, a second stage in LDS, and the second block half a
// step behind the first: all the same or slower.)
#pragma once

#include "conv_f32_gemm.hpp"

namespace n2d2hip {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

// What operands are multiplied by before they are taken apart, and sums afterwards: a bf16 has no bits below 2^-133, which is 2^-149, a
// float's last, 2^16 larger.  Error of sums of 32 products, one operand of size 2^-112 / 2^-116 / 2^-120 / 2^-124, without: 1.4e-7 / 2.2e-6 /
// 3.5e-5 / 5.7e-4, with: as of size 1.
constexpr float PARTS_SCALE = 0x1p16f, PARTS_UNSCALE = 0x1p-32f;

// (a, b) -> their first parts, packed; a and b become the rests
__device__ __forceinline__ unsigned bf16_part(float& a, float& b)
{
    const unsigned u = __builtin_bit_cast(unsigned, __builtin_convertvector(v2f{a, b}, v2bf));
    a -= __builtin_bit_cast(float, u << 16);
    b -= __builtin_bit_cast(float, u & 0xffff0000u);
    return u;
}
__device__ __forceinline__ void bf16_parts(float (&v)[8], v4u (&parts)[3])
{
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        float a = v[2 * j] * PARTS_SCALE, b = v[2 * j + 1] * PARTS_SCALE;
        parts[0][j] = bf16_part(a, b);
        parts[1][j] = bf16_part(a, b);
        parts[2][j] = __builtin_bit_cast(unsigned, __builtin_convertvector(v2f{a, b}, v2bf));
    }
}

constexpr int PK = 32;                           // channels of a step: K of one matrix instruction
constexpr int PATCH_FRAG = 3 * 1024;             // bytes of a weight fragment: 16 rows x 32 channels in three parts

// Weights as the matrix instructions take them: [chunk of 32 channels][tap][16 rows of q][part][lane][8 channels]; rows and
// channels that do not exist are zero.  Loads scattered over lines bound it, a line to a lane, so each wave is a block and few weights are spread over as
// many compute units as they can be; what a fragment is is worked out once a wave.  us, the layer's forward pass, four waves a block and by lane / now:
// 512 -> 512, 5x5, 14 x 14, batch 16 307.6 / 300.7; 64 -> 64, 3x3, 56 x 56, batch 64 136.9 / 136.1; 32 -> 32 74.1 / 73.4.  (conv_f32_lay_taps_kernel: no change.)
constexpr int LAY_THREADS = 64;
__global__ __launch_bounds__(LAY_THREADS) void conv_f32_lay_parts_kernel(const float* __restrict__ w, v4u* __restrict__ wt, int total, int Q, int nq, int Ch, int T,
                                                                 int qs, int chs)
{
    for (int i = blockIdx.x * LAY_THREADS + threadIdx.x; i < total; i += gridDim.x * LAY_THREADS) {
        const int lane = i & 63, frag = __builtin_amdgcn_readfirstlane(i >> 6), qb = frag % nq, rest = frag / nq, tap = rest % T, chunk = rest / T;
        const int q = qb * 16 + (lane & 15), ch = chunk * PK + 8 * (lane >> 4);
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = (q < Q && ch + j < Ch) ? w[(size_t)q * qs + (size_t)(ch + j) * chs + tap] : 0.0f;
        v4u parts[3];
        bf16_parts(v, parts);
#pragma unroll
        for (int p = 0; p < 3; ++p) wt[(size_t)frag * (PATCH_FRAG / 16) + p * 64 + lane] = parts[p];
    }
}

// What the kernel's blocks run through: a block of an XCD takes every so many-th of the XCD's items, (pixel tile, q tile), q tiles of a
// pixel tile one behind the other.
struct PatchItem {
    int item, tile, qtile;
    __device__ __forceinline__ bool at(const PixelGemm& g)
    {
        const int pt = item / g.qtiles;
        qtile = item - pt * g.qtiles;
        tile = (blockIdx.x & 7) * g.ptiles8 + pt;
        return pt < g.ptiles8 && tile < g.ptiles;
    }
};

// A tile is 16 MQ WQ rows of q x 16 NP WP consecutive pixels.  What its pixels' taps read is one run of source positions (rows
// are consecutive, and so are a channel's images, up to the other channels between them): a step brings 32 channels of that
// run into LDS, in parts, 16 bytes to 8 channels of a position, and runs through the taps from there; a tap outside the
// source reads a position that holds zeros.  A block stays for a run of tiles, whose loads go on across their ends.
// CL 4: backward-data of a 3x3 kernel at stride 2.  A tile's pixels are places of a grid of half the resolution, and each is the four
// pixels (2 py, 2 px) ... (2 py + 1, 2 px + 1): every tap belongs to one of them, and all read from 2 x 2 source positions.  Axis by axis, taps 0 and 2
// go to the pixel c.ry (c.rx) and tap 1 to the other.
template <int WQ, int WP, int MQ, int NP, int PB, int NT, bool FOLD, int CL = 1>
__global__ __launch_bounds__(256, 2) void conv_f32_patch_kernel(PixelGemm g, const float* __restrict__ srcX, const float* __restrict__ srcW,
                                                                const v4u* __restrict__ wt, const float* __restrict__ bias, float beta,
                                                                float* __restrict__ out, size_t partial)
{
    static_assert(WQ * WP == 4, "four waves, one to 8 channels of a step");
    static_assert(NP == 2 || NP == 4, "a tap's first 16 pixels are in b[0]; a lane for each of a wave's pixels");
    constexpr int QT = 16 * MQ * WQ, PT = 16 * NP * WP;
    constexpr int POS = 64 * PB + 16;            // positions of 8 channels, zeros behind them (16: what lanes of an LDS read share no banks)
    constexpr int OCT = POS * 16, PART = 4 * OCT;
    constexpr int LOADS = 8 * PB;
    __shared__ __attribute__((aligned(16))) char smem[3 * PART];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, lo = lane >> 4, wq = wave / WP, wp = wave % WP;
    const int nchunks = (g.Ch + PK - 1) / PK, plane4 = g.planeS * 4, tstep = g.qpad / 16 * PATCH_FRAG;
    const unsigned zaddr = lo * OCT + 64 * PB * 16;
    const __amdgpu_buffer_rsrc_t rsrcX = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(srcX), 0, g.bytesX, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrcW = __builtin_amdgcn_make_buffer_rsrc(const_cast<v4u*>(wt), 0, nchunks * g.T * tstep, 0x00020000);
    if (threadIdx.x < 12) *(v4u*)(smem + threadIdx.x * OCT + 64 * PB * 16) = v4u{0, 0, 0, 0};

    const PixelClass& c = g.c[0];                // (forward, or backward-data at stride 1)
    static_assert(CL == 1 || (NT == 9 && !FOLD), "3x3 kernels, float sums");
    const int nT = NT ? NT : c.nT;
    const int nx = CL == 4 ? 2 : NT == 9 ? 3 : c.nx, ny = CL == 4 ? 2 : NT == 9 ? 3 : div_f32(c.nT, c.nxd);      // source positions of the taps
    // of tap (i, j): its source row and column, and which of the four pixels it belongs to
    auto row_of = [&](int i) { return CL == 4 ? (i == 1 ? c.ry : i >> 1) : i; };
    auto column_of = [&](int j) { return CL == 4 ? (j == 1 ? c.rx : j >> 1) : j; };
    auto class_of = [](int i, int j) { return CL == 4 ? 2 * (i == 1) + (j == 1) : 0; };
    const int reach = (ny - 1) * g.Ws + nx - 1, back = g.d > 0 ? 0 : reach, ahead = reach - back;
    const int cbeg = blockIdx.z * c.kchunk, cend = min(cbeg + c.kchunk, nchunks);
    // a tile's run: source positions of its first pixel's first tap to its last pixel's last one, counted over a channel's images
    auto source = [&](int p) {
        const int b = div_f32(p, c.ghw), rem = p - b * c.gHW, py = div_f32(rem, c.gw), px = rem - py * c.gW;
        return b * g.planeS + (py * g.sy + c.y0) * g.Ws + px * g.sx + c.x0;
    };
    // loader: a wave takes 8 of a step's channels, 64 positions at a time
    unsigned voff[PB];
#pragma unroll
    for (int u = 0; u < PB; ++u) voff[u] = F32_OOB;
    auto locate = [&](int p0) {
        const int run0 = source(p0) - back, run1 = source(min(p0 + PT, c.P) - 1) + ahead;
#pragma unroll
        for (int u = 0; u < PB; ++u) {
            const int l = run0 + u * 64 + lane;
            const bool there = l >= 0 && l <= run1 && l < g.npos;
            const int b = there ? div_f32(l, g.dplane) : 0;
            voff[u] = there ? 4u * (unsigned)(l + b * (g.Ch - 1) * g.planeS) : F32_OOB;
        }
    };
    float v[PB][8];
    auto load_part = [&](int chunk, int from, int to) {
        const int ch0 = chunk * PK + 8 * wave;
#pragma unroll
        for (int i = from; i < to; ++i) {
            const int u = i >> 3, j = i & 7;
            v[u][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrcX, voff[u], ch0 + j < g.Ch ? (ch0 + j) * plane4 : 0x7ffffffc, 0));
        }
    };
    auto put = [&]() {
#pragma unroll
        for (int u = 0; u < PB; ++u) {
            v4u parts[3];
            bf16_parts(v[u], parts);
#pragma unroll
            for (int p = 0; p < 3; ++p) *(v4u*)(smem + p * PART + wave * OCT + (u * 64 + lane) * 16) = parts[p];
        }
    };
    v4f acc[CL][MQ][NP];
    double folded[FOLD ? MQ : 1][NP][4];
    auto each = [&](auto&& f) {
#pragma unroll
        for (int k = 0; k < CL; ++k)
#pragma unroll
            for (int m = 0; m < MQ; ++m)
#pragma unroll
                for (int n = 0; n < NP; ++n)
#pragma unroll
                    for (int r = 0; r < 4; ++r) f(k, m, n, r);
    };
    auto fold = [&]() {
        each([&](int k, int m, int n, int r) { folded[m][n][r] += (double)acc[k][m][n][r]; acc[k][m][n][r] = 0.0f; });
    };
    // a wave's weights: consecutive taps of a chunk are a fragment of every 16 rows of q apart
    v4u a[3][MQ][3], b[2][3];
    auto weights = [&](v4u (&w)[MQ][3], int qtile, int chunk, int t) {
        const int at = (qtile * (QT / 16) + wq * MQ) * PATCH_FRAG + (chunk * nT + t) * tstep;
#pragma unroll
        for (int m = 0; m < MQ; ++m)
#pragma unroll
            for (int p = 0; p < 3; ++p) w[m][p] = __builtin_bit_cast(v4u, __builtin_amdgcn_raw_buffer_load_b128(rsrcW, lane * 16, at + m * PATCH_FRAG + p * 1024, 0));
    };
    auto first_weights = [&](int qtile) {
        weights(a[0], qtile, cbeg, 0);
        if (NT == 9) weights(a[1], qtile, cbeg, 1);
    };
    unsigned xaddr[NP], mask[NP];                // of a lane's pixels: where tap (0, 0) is in LDS; the taps that exist

    // Infinities, and what rounds to one in bf16, leave NaN where float products might not.  A wave that holds such sums adds them
    // again, on the fp32 matrix cores straight from memory, in double from four channels to the next.
    // us of 64 -> 64, 56 x 56, batch 64, forward / data: finite 93 / 85; NaN throughout 624 / 507; a channel of the input NaN 617 / 505; one weight
    // NaN 852 / 815 (a sum after the other by the lane that held it: 6520 / 6570, 6500 / 6590, 970 / 1500).
    // (32 pixels of one class at a time: of more the sums would take the registers that hold the next step's operands)
    auto again_in_float = [&](auto k_, auto n_, int p0, int q0) {
        constexpr int k = decltype(k_)::value, n0 = decltype(n_)::value;
        int here = lane;                         // (opaque: nothing of this is worked out ahead, and held, by waves that never come here)
        const float* weights_ = srcW;
        asm volatile("" : "+v"(here), "+s"(weights_));
        const int l16 = here & 15, lo = here >> 4;
        const int rows = CL == 4 ? 3 : ny, columns = CL == 4 ? 3 : nx, chend = min(cend * PK, g.Ch);
        const __amdgpu_buffer_rsrc_t rsrcV = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(weights_), 0, g.bytesW, 0x00020000);
        int img[2], y0[2], x0[2];
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            const int p = p0 + (wp * NP + n0 + n) * 16 + l16;
            img[n] = div_f32(min(p, c.P - 1), c.ghw);
            const int rem = p - img[n] * c.gHW, py = div_f32(rem, c.gw);
            y0[n] = p < c.P ? py * g.sy + c.y0 : -(1 << 24);         // (no row at all)
            x0[n] = (rem - py * c.gW) * g.sx + c.x0;
        }
        auto there = [&](int n, int i, int j) {
            return (unsigned)(y0[n] + g.d * row_of(i)) < (unsigned)g.Hs && (unsigned)(x0[n] + g.d * column_of(j)) < (unsigned)g.Ws;
        };
        auto source_of = [&](int n, int ch, int i, int j) { return (img[n] * g.Ch + ch) * g.planeS + (y0[n] + g.d * row_of(i)) * g.Ws + x0[n] + g.d * column_of(j); };
        double sum[MQ][2][4] = {};
        bool odd = false;                        // a weight is not finite
#pragma unroll 1
        for (int ch0 = cbeg * PK; ch0 < chend; ch0 += 4) {
            const int ch = ch0 + lo;
            v4f part[MQ][2];
#pragma unroll
            for (int m = 0; m < MQ; ++m)
#pragma unroll
                for (int n = 0; n < 2; ++n) part[m][n] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
            for (int i = 0; i < rows; ++i)
#pragma unroll 1
                for (int j = 0; j < columns; ++j) {
                    if (class_of(i, j) != k) continue;
                    float w[MQ], x[2];
#pragma unroll
                    for (int m = 0; m < MQ; ++m) {
                        const int q = q0 + (wq * MQ + m) * 16 + l16;
                        w[m] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                            rsrcV, q < g.Q && ch < chend ? 4u * (unsigned)(q * g.qs + ch * g.chs + i * columns + j) : F32_OOB, 0, 0));
                        odd |= !(__builtin_fabsf(w[m]) < __builtin_inff());
                    }
#pragma unroll
                    for (int n = 0; n < 2; ++n)
                        x[n] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                            rsrcX, ch < chend && there(n, i, j) ? 4u * (unsigned)source_of(n, ch, i, j) : F32_OOB, 0, 0));
#pragma unroll
                    for (int m = 0; m < MQ; ++m)
#pragma unroll
                        for (int n = 0; n < 2; ++n) part[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[m], x[n], part[m][n], 0, 0, 0);
                }
#pragma unroll
            for (int m = 0; m < MQ; ++m)
#pragma unroll
                for (int n = 0; n < 2; ++n)
#pragma unroll
                    for (int r = 0; r < 4; ++r) sum[m][n][r] += (double)part[m][n][r];
        }
        odd = __any(odd);
        unsigned nans = 0;                       // sums that a tap outside the source may have made NaN: above there was a product with 0, of which there is none
#pragma unroll
        for (int m = 0; m < MQ; ++m)
#pragma unroll
            for (int n = 0; n < 2; ++n)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (__builtin_fabsf(acc[k][m][n0 + n][r]) < __builtin_inff()) continue;
                    const float s = (float)sum[m][n][r];
                    acc[k][m][n0 + n][r] = s;
                    if (odd && s != s && q0 + (wq * MQ + m) * 16 + 4 * lo + r < g.Q) nans |= 1u << ((m * 2 + n) * 4 + r);
                }
        // (one after the other, and the code once: sixteen times, in each of the kernel's instances, the compiler takes seven minutes for the file
        // instead of 40 s, and one weight NaN is 1240 / 1260 us)
#pragma unroll 1
        for (int at = 0; at < 8 * MQ; ++at) {
            if (!__any(nans >> at & 1)) continue;
            const int n = at >> 2 & 1, q = q0 + (wq * MQ + (at >> 3)) * 16 + 4 * lo + (at & 3);
            const int y = n ? y0[1] : y0[0], x_ = n ? x0[1] : x0[0], b = n ? img[1] : img[0];
            float s = 0.0f;
            if (nans >> at & 1) {
#pragma unroll 1
                for (int i = 0; i < rows; ++i)
#pragma unroll 1
                    for (int j = 0; j < columns; ++j) {
                        const int ys = y + g.d * row_of(i), xs = x_ + g.d * column_of(j);
                        if (class_of(i, j) != k || (unsigned)ys >= (unsigned)g.Hs || (unsigned)xs >= (unsigned)g.Ws) continue;
#pragma unroll 1
                        for (int ch = cbeg * PK; ch < chend && s == s; ch += 8) {
                            float w[8], x[8];
#pragma unroll
                            for (int u = 0; u < 8; ++u) {
                                const bool is = ch + u < chend;
                                w[u] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                    rsrcV, is ? 4u * (unsigned)(q * g.qs + (ch + u) * g.chs + i * columns + j) : F32_OOB, 0, 0));
                                x[u] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                    rsrcX, is ? 4u * (unsigned)((b * g.Ch + ch + u) * g.planeS + ys * g.Ws + xs) : F32_OOB, 0, 0));
                            }
#pragma unroll
                            for (int u = 0; u < 8; ++u) s += w[u] * x[u];
                        }
                    }
            }
#pragma unroll
            for (int m = 0; m < MQ; ++m)
#pragma unroll
                for (int n = 0; n < 2; ++n)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (at == (m * 2 + n) * 4 + r && (nans >> at & 1)) acc[k][m][n0 + n][r] = s;
        }
    };

    // (before its first tile a block runs through one step that only loads: its code is that of the others)
    PatchItem it, to;
    it.item = (int)(blockIdx.x >> 3) - (int)(gridDim.x >> 3);
    it.tile = it.qtile = 0;
    to.item = blockIdx.x >> 3;
    for (bool again = to.at(g);;) {
        const bool first = it.item < 0;
        if (first && !again) return;
        const int p0 = it.tile * PT, q0 = it.qtile * QT;
        const int qn = q0 + wq * MQ * 16 + 4 * lo;           // this lane's rows of q: qn + 16 m + r
        const bool live = !first && q0 + wq * MQ * 16 < g.Q;
        if (live) {
            // a lane works out one of the wave's pixels, and hands it to those that take it
            const int run0 = source(p0) - back;
            // taps first .. end - 1 of an axis lie inside it
            auto inside = [&](int at, int size, int n) {
                const int first = min(max(g.d > 0 ? -at : at - size + 1, 0), n), end = min(max(g.d > 0 ? size - at : at + 1, 0), n);
                return ((1u << end) - 1u) & ~((1u << first) - 1u);
            };
            const int p = p0 + wp * NP * 16 + lane, pp = min(p, c.P - 1);
            const int img = div_f32(pp, c.ghw), rem = pp - img * c.gHW, py = div_f32(rem, c.gw), px = rem - py * c.gW;
            const int y = py * g.sy + c.y0, x = px * g.sx + c.x0;
            const unsigned m = p < c.P ? inside(x, g.Ws, nx) | (inside(y, g.Hs, ny) << nx) : 0u;
            const unsigned at = 16 * (img * g.planeS + y * g.Ws + x - run0);
#pragma unroll
            for (int n = 0; n < NP; ++n) {
                mask[n] = __shfl((int)m, n * 16 + l16);
                xaddr[n] = lo * OCT + __shfl((int)at, n * 16 + l16);
            }
        }
        each([&](int k, int m, int n, int r) {
            acc[k][m][n][r] = 0.0f;
            if (FOLD) folded[m][n][r] = 0.0;
        });
        auto pixels = [&](v4u (&x)[3], int n, int i, int j) {
            const int row = row_of(i), column = column_of(j);
            const unsigned bit = (1u << column) | (1u << (nx + row));
            const unsigned at = (mask[n] & bit) == bit ? xaddr[n] + 16 * g.d * (row * g.Ws + column) : zaddr;
#pragma unroll
            for (int p = 0; p < 3; ++p) x[p] = *(const v4u*)(smem + at + p * PART);
        };
        // the products but the largest in a sum of their own: a matrix instruction rounds its sum four times
        auto products = [&](const v4u (&w)[MQ][3], const v4u (&x)[3], int n, int k) {
            v4f small[MQ];
#pragma unroll
            for (int m = 0; m < MQ; ++m) small[m] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s = 0; s < 5; ++s) {
                constexpr int pa[5] = {1, 0, 2, 0, 1}, pb[5] = {1, 2, 0, 1, 0};
#pragma unroll
                for (int m = 0; m < MQ; ++m)
                    small[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, w[m][pa[s]]), __builtin_bit_cast(v8bf, x[pb[s]]), small[m], 0, 0, 0);
            }
#pragma unroll
            for (int m = 0; m < MQ; ++m)
                acc[k][m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, w[m][0]), __builtin_bit_cast(v8bf, x[0]), acc[k][m][n], 0, 0, 0);
#pragma unroll
            for (int m = 0; m < MQ; ++m)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[k][m][n][r] += small[m][r];
        };
        // a tap's products, 16 pixels at a time, the next 16 (of tap (i1, j1) after the last) on their way from LDS
        auto tap = [&](const v4u (&w)[MQ][3], int i, int j, int i1, int j1, bool last) {
#pragma unroll
            for (int n = 0; n < NP; ++n) {
                if (n + 1 < NP) pixels(b[(n + 1) & 1], n + 1, i, j);
                else if (!last) pixels(b[(n + 1) & 1], 0, i1, j1);
                __builtin_amdgcn_sched_barrier(0);
                products(w, b[n & 1], n, class_of(i, j));
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        int until = FOLD ? c.fold : 0;
        for (int chunk = first ? cend - 1 : cbeg; chunk < cend; ++chunk) {
            if (!first) __syncthreads();         // (the chunk is in LDS)
            // what is loaded meanwhile: the next chunk, or the next tile's first (or this one again, to no use)
            const bool more = chunk + 1 < cend, next_tile = !more && again;
            const int lchunk = next_tile ? cbeg : more ? chunk + 1 : chunk, lqtile = next_tile ? to.qtile : it.qtile;
            if (next_tile) locate(to.tile * PT);
            if constexpr (NT == 9) {
                if (live) {
                    pixels(b[0], 0, 0, 0);
                    auto row = [&](int i) {
#pragma unroll
                        for (int j = 0; j < 3; ++j) {
                            if (i == 0) load_part(lchunk, j * LOADS / 3, (j + 1) * LOADS / 3);
                            const bool on = i == 2 && j > 0;         // (two taps on: in the next chunk)
                            weights(a[(j + 2) % 3], on ? lqtile : it.qtile, on ? lchunk : chunk, on ? j - 1 : 3 * i + j + 2);
                            tap(a[j], i, j, j == 2 ? i + 1 : i, (j + 1) % 3, i == 2 && j == 2);
                        }
                    };
                    if constexpr (CL == 4) {     // (which sums a row's taps go to is in the code)
                        row(0);
                        row(1);
                        row(2);
                    } else {
                        for (int i = 0; i < 3; ++i) row(i);
                    }
                } else {
                    load_part(lchunk, 0, LOADS);
                    if (next_tile) first_weights(to.qtile);
                }
            } else {
                load_part(lchunk, 0, LOADS);
                if (live) {
                    int i = 0, j = 0;
                    pixels(b[0], 0, 0, 0);
                    for (int t = 0; t < nT; ++t) {
                        int i1 = i, j1 = j + 1;
                        if (j1 == nx) { j1 = 0; ++i1; }
                        const bool last = t + 1 == nT;
                        weights(a[1], last ? lqtile : it.qtile, last ? lchunk : chunk, last ? 0 : t + 1);
                        tap(a[0], i, j, i1, j1, last);
                        i = i1; j = j1;
#pragma unroll
                        for (int p = 0; p < 3; ++p)
#pragma unroll
                            for (int m = 0; m < MQ; ++m) a[0][m][p] = a[1][m][p];
                    }
                } else if (next_tile) {
                    first_weights(to.qtile);
                }
            }
            if (FOLD && --until == 0) {
                fold();
                until = c.fold;
            }
            __syncthreads();
            if (more || next_tile) put();
        }
        if (FOLD) fold();
        each([&](int k, int m, int n, int r) {
            if constexpr (FOLD) acc[k][m][n][r] = (float)(folded[m][n][r] * (double)PARTS_UNSCALE);
            else acc[k][m][n][r] *= PARTS_UNSCALE;
        });
        // A lane holds pixel .. + lane % 16 and rows qn + 16 m + r.
        if (live) {
            const size_t zoff = (size_t)blockIdx.z * partial;
            unsigned obase[NP];                  // of the pixels, in `out`; CL 4: of (2 py, 2 px), and whether row 2 py + 1 and column 2 px + 1 are there
            const int p = p0 + wp * NP * 16 + lane, pp = min(p, c.P - 1), img = div_f32(pp, c.ghw);
            unsigned o;
            if constexpr (CL == 4) {
                const int rem = pp - img * c.gHW, py = div_f32(rem, c.gw), px = rem - py * c.gW;
                o = 4u * (unsigned)(img * g.Q * g.planeO + 2 * py * g.Wo + 2 * px) | (2 * px + 1 < g.Wo ? 2u : 0u)
                    | ((2 * py + 1) * g.Wo < g.planeO ? 1u : 0u);
            } else {
                o = 4u * (unsigned)(img * (g.Q - 1) * g.planeO + pp);
            }
            if (p >= c.P) o = F32_OOB;
#pragma unroll
            for (int n = 0; n < NP; ++n) obase[n] = __shfl((int)o, n * 16 + l16);
            auto place = [&](int k, int n) {     // of one of a place's pixels; F32_OOB: there is none
                if (CL == 1 || obase[n] == F32_OOB) return obase[n];
                const unsigned ry = k & 2 ? 1 - c.ry : c.ry, rx = k & 1 ? 1 - c.rx : c.rx, needs = ry | rx << 1;
                return (obase[n] & needs) == needs ? (obase[n] & ~3u) + 4u * (ry * g.Wo + rx) : F32_OOB;
            };
            const __amdgpu_buffer_rsrc_t rsrcO = __builtin_amdgcn_make_buffer_rsrc(out + zoff, 0, g.bytesO, 0x00020000);
            const int planeO4 = 4 * g.planeO;
            const unsigned qrow = qn * planeO4;
            float finite = 0.0f;
            each([&](int k, int m, int n, int r) { finite = __builtin_fmaf(acc[k][m][n][r], 0.0f, finite); });
            if (__any(finite != finite)) {
                const auto pixels_of = [&](auto k_) {
                    again_in_float(k_, std::integral_constant<int, 0>{}, p0, q0);
                    if constexpr (NP == 4) again_in_float(k_, std::integral_constant<int, 2>{}, p0, q0);
                };
                pixels_of(std::integral_constant<int, 0>{});
                if constexpr (CL == 4) {
                    pixels_of(std::integral_constant<int, 1>{});
                    pixels_of(std::integral_constant<int, 2>{});
                    pixels_of(std::integral_constant<int, 3>{});
                }
            }
            if (partial != 0 || (beta == 0.0f && !bias)) {
                unsigned at = F32_OOB;
                each([&](int k, int m, int n, int r) {
                    if (q0 + wq * MQ * 16 + 16 * m + r >= g.Q) return;
                    if (CL == 1 || r == 0) at = place(k, n);
                    const float s = acc[k][m][n][r];     // (the cast of a vector's element reads its first one)
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, s), rsrcO, qn + 16 * m + r < g.Q && at != F32_OOB ? at + qrow : F32_OOB,
                                                          (16 * m + r) * planeO4, 0);
                });
            } else {
                each([&](int k, int m, int n, int r) {
                    const unsigned base = place(k, n);
                    if (base == F32_OOB || qn + 16 * m + r >= g.Q) return;
                    float* at = out + base / 4u + (size_t)(qn + 16 * m + r) * g.planeO;
                    float s = acc[k][m][n][r];
                    if (beta != 0.0f) s += beta * *at;
                    if (bias) s = bias[qn + 16 * m + r] + s;
                    *at = s;
                });
            }
        }
        if (!again) return;
        it = to;
        to.item += gridDim.x >> 3;
        again = to.at(g);
    }
}

} // namespace n2d2hip
