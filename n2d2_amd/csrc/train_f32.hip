// Float32 cells of a quantization-aware training step: convolution forward, its three backward kernels, softmax,
// the loss at the output and the SGD update.  Tensors are N2D2's own NCHW / OCHW float tensors (X fastest), so a
// training graph exchanges them without conversion.
//
// Convolutions run on the matrix cores (conv_f32_gemm.hpp) wherever they are neither grouped nor dilated, but for small forward
// sums (f32_path).  The kernels here are direct: one thread per produced element, walking channels and taps in the reference's order (so forward and
// backward-data give the reference's float sums term for term), and one block per weight for backward-filter, whose long
// sum over batch and pixels is wavefront-reduced in double.
#include <algorithm>
#include <type_traits>
#include <vector>

#include "common.h"
#include "conv_f32_gemm.hpp"
#include "conv_f32_patch.hpp"
#include "conv_f32_taps.hpp"
#include "conv_f32_filter_rows.hpp"
#include "sat_math.hpp"
#include "depthwise_f32.hpp"

namespace n2d2hip {

constexpr int TBLOCK = 256;

struct ConvF32 {
    int B, C, H, W, O, oH, oW, kW, kH, Cw;      // Cw = C / groups
    int sx, sy, pl, pt, pr, pb, dx, dy;
    int depthwise;                                // groups == C == O
    int choice;                                   // the descriptor's kernel_choice bits
    int ranges = 0;                               // a product that stands for a pass: float sums of K / ranges terms at most
};

__device__ __forceinline__ double wave_sum_d(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        v += __shfl_xor(v, off, 64);
    return v;
}
__device__ __forceinline__ double block_sum_d(double v)
{
    __shared__ double red[TBLOCK / 64];
    v = wave_sum_d(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0.0;
#pragma unroll
    for (int i = 0; i < TBLOCK / 64; ++i) t += red[i];
    return t;
}

// out[b,o,oy,ox] = alpha-less weighted sum (+ bias) + beta * out.  The window is clipped at the borders (no padded
// zeros are read); a full 3x3 window is summed row by row, then the rows, as the reference's unrolled branch does.
__global__ __launch_bounds__(TBLOCK) void conv_f32_forward_kernel(ConvF32 q, const float* __restrict__ x, const float* __restrict__ w,
                                                                  const float* __restrict__ bias, float beta, float* __restrict__ y)
{
    const size_t total = (size_t)q.B * q.O * q.oH * q.oW;
    for (size_t idx = (size_t)blockIdx.x * TBLOCK + threadIdx.x; idx < total; idx += (size_t)gridDim.x * TBLOCK) {
        const int ox = idx % q.oW, oy = (idx / q.oW) % q.oH;
        const int o = (idx / ((size_t)q.oW * q.oH)) % q.O, b = idx / ((size_t)q.oW * q.oH * q.O);
        const int dilKx = q.kW + (q.dx - 1) * (q.kW - 1), dilKy = q.kH + (q.dy - 1) * (q.kH - 1);
        const int sxMin = max(q.pl - ox * q.sx, 0), syMin = max(q.pt - oy * q.sy, 0);
        const int sxMax = min(max(q.W + q.pl - ox * q.sx, 0), dilKx), syMax = min(max(q.H + q.pt - oy * q.sy, 0), dilKy);
        const int ix = ox * q.sx - q.pl, iy = oy * q.sy - q.pt;
        const int c0 = q.depthwise ? o : 0, c1 = q.depthwise ? o + 1 : q.C;
        const bool full3 = sxMin == 0 && syMin == 0 && sxMax == 3 && syMax == 3 && q.kW == 3 && q.kH == 3;
        float sum = 0.0f;
        for (int c = c0; c < c1; ++c) {
            const float* xc = x + ((size_t)b * q.C + c) * q.H * q.W;
            const float* wc = w + ((size_t)o * q.Cw + (q.depthwise ? 0 : c)) * q.kH * q.kW;
            if (full3) {
                const float* r0 = xc + (size_t)iy * q.W + ix;
                const float* r1 = r0 + q.W;
                const float* r2 = r1 + q.W;
                sum = sum + (wc[0] * r0[0] + wc[1] * r0[1] + wc[2] * r0[2])
                          + (wc[3] * r1[0] + wc[4] * r1[1] + wc[5] * r1[2])
                          + (wc[6] * r2[0] + wc[7] * r2[1] + wc[8] * r2[2]);
            } else {
                for (int ty = syMin; ty * q.dy < syMax; ++ty)
                    for (int tx = sxMin; tx * q.dx < sxMax; ++tx)
                        sum += wc[ty * q.kW + tx] * xc[(size_t)(iy + ty * q.dy) * q.W + ix + tx * q.dx];
            }
        }
        float r = sum + (beta != 0.0f ? beta * y[idx] : 0.0f);
        if (bias) r = bias[o] + r;
        y[idx] = r;
    }
}

// dx[b,c,iy,ix] = sum over connected outputs (ascending) and over the taps reaching this element + beta * dx.
__global__ __launch_bounds__(TBLOCK) void conv_f32_backward_data_kernel(ConvF32 q, const float* __restrict__ w, const float* __restrict__ dy,
                                                                        float beta, float* __restrict__ dx)
{
    const size_t total = (size_t)q.B * q.C * q.H * q.W;
    const int oxStride = q.sx * q.oW, oyStride = q.sy * q.oH;
    for (size_t idx = (size_t)blockIdx.x * TBLOCK + threadIdx.x; idx < total; idx += (size_t)gridDim.x * TBLOCK) {
        const int ix = idx % q.W, iy = (idx / q.W) % q.H;
        const int c = (idx / ((size_t)q.W * q.H)) % q.C, b = idx / ((size_t)q.W * q.H * q.C);
        const int ixPad = ix + q.pl, iyPad = iy + q.pt;
        const int sxMin = ixPad % q.sx + max(ixPad - ixPad % q.sx - oxStride + q.sx, 0);
        const int syMin = iyPad % q.sy + max(iyPad - iyPad % q.sy - oyStride + q.sy, 0);
        const int sxMax = min(q.kW, ixPad + 1), syMax = min(q.kH, iyPad + 1);
        const bool full3 = syMax - syMin == 3 && q.sy == 1 && sxMax - sxMin == 3 && q.sx == 1;
        const int o0 = q.depthwise ? c : 0, o1 = q.depthwise ? c + 1 : q.O;
        float g = 0.0f;
        for (int o = o0; o < o1; ++o) {
            const float* wo = w + ((size_t)o * q.Cw + (q.depthwise ? 0 : c)) * q.kH * q.kW;
            const float* dyo = dy + ((size_t)b * q.O + o) * q.oH * q.oW;
            if (full3) {
                const int ox = ixPad - sxMin, oy = iyPad - syMin;
#pragma unroll
                for (int t = 0; t < 9; ++t)
                    g = g + wo[(syMin + t / 3) * q.kW + sxMin + t % 3] * dyo[(size_t)(oy - t / 3) * q.oW + ox - t % 3];
            } else {
                for (int ty = syMin; ty < syMax; ty += q.sy)
                    for (int tx = sxMin; tx < sxMax; tx += q.sx)
                        g += wo[ty * q.kW + tx] * dyo[(size_t)((iyPad - ty) / q.sy) * q.oW + (ixPad - tx) / q.sx];
            }
        }
        dx[idx] = g + (beta != 0.0f ? beta * dx[idx] : 0.0f);
    }
}

// The same two sums, term for term, with the loads of the next products requested together: the chain of additions is short
// (4 cycles a term), waiting for each term's operands is what takes the time (0.14 us a term, one after the other).  A thread
// is an element of the result; the walk over (channel, tap) is the same for all and scalar, a thread only adds its own base
// and looks the tap up in its mask (bit j: column j inside, bit nj + i: row i inside).
struct WalkF32 {
    int n, ni, nj;                               // channels, tap rows, tap columns
    int xo, xi, xj, wo, wi, wj;                  // offsets per channel, row, column in the source and in the weights
    DivF32 dplane, dw, dch;                      // result: plane, row length, channels
};

constexpr int WALK = 16;                         // products in flight
__device__ __forceinline__ float walk_f32(const WalkF32& k, const float* __restrict__ x, const float* __restrict__ w, int xb, int wb, unsigned mask)
{
    float sum = 0.0f;
    const int total = k.n * k.ni * k.nj;
    int xc = 0, wc = 0, i = 0, j = 0;            // the next product's channel offsets, row, column
    for (int k0 = 0; k0 < total; k0 += WALK) {
        float xv[WALK], wv[WALK];
        unsigned ok = 0;
#pragma unroll
        for (int u = 0; u < WALK; ++u) {
            const unsigned bit = (1u << j) | (1u << (k.nj + i)) | (k0 + u < total ? 0u : 0x80000000u);       // (bit 31: never set)
            const bool v = (mask & bit) == bit;
            ok |= v ? 1u << u : 0u;
            xv[u] = x[v ? xb + xc + i * k.xi + j * k.xj : 0];
            wv[u] = w[v ? wb + wc + i * k.wi + j * k.wj : 0];
            if (++j == k.nj) {
                j = 0;
                if (++i == k.ni) { i = 0; xc += k.xo; wc += k.wo; }
            }
        }
#pragma unroll
        for (int u = 0; u < WALK; ++u) sum = ok & (1u << u) ? sum + wv[u] * xv[u] : sum;
    }
    return sum;
}
// Forward of a 3x3 kernel, CB channels at a time: a full window is summed row by row, then the rows.
template <int CB>
__device__ __forceinline__ float walk3x3_f32(const WalkF32& k, const float* __restrict__ x, const float* __restrict__ w, int xb, int wb, unsigned mask)
{
    float sum = 0.0f;
    for (int c0 = 0; c0 < k.n; c0 += CB) {
        float xv[CB][9], wv[CB][9];
#pragma unroll
        for (int c = 0; c < CB; ++c)
#pragma unroll
            for (int t = 0; t < 9; ++t) {
                const unsigned bit = (1u << t % 3) | (8u << t / 3) | (c0 + c < k.n ? 0u : 0x80000000u);
                const bool v = (mask & bit) == bit;
                xv[c][t] = x[v ? xb + (c0 + c) * k.xo + t / 3 * k.xi + t % 3 * k.xj : 0];
                wv[c][t] = w[v ? wb + (c0 + c) * k.wo + t / 3 * k.wi + t % 3 * k.wj : 0];
            }
#pragma unroll
        for (int c = 0; c < CB; ++c) {
            if (c0 + c >= k.n) break;
            const float* a = wv[c];
            const float* b = xv[c];
            const float full = sum + (a[0] * b[0] + a[1] * b[1] + a[2] * b[2]) + (a[3] * b[3] + a[4] * b[4] + a[5] * b[5])
                                   + (a[6] * b[6] + a[7] * b[7] + a[8] * b[8]);
#pragma unroll
            for (int t = 0; t < 9; ++t) {
                const unsigned bit = (1u << t % 3) | (8u << t / 3);
                sum = (mask & bit) == bit ? sum + a[t] * b[t] : sum;
            }
            sum = (mask & 63u) == 63u ? full : sum;
        }
    }
    return sum;
}

// SHAPE: 0 any kernel, 1 / 4: forward of a 3x3 kernel, channels at a time.
template <bool BWD, int SHAPE>
__global__ __launch_bounds__(64) void conv_f32_walk_kernel(ConvF32 q, WalkF32 k, const float* __restrict__ x, const float* __restrict__ w,
                                                           const float* __restrict__ bias, float beta, float* __restrict__ out, int total)
{
    const int idx = blockIdx.x * 64 + threadIdx.x;
    if (idx >= total) return;
    const int img = div_f32(idx, k.dplane);      // image and channel
    const int b = div_f32(img, k.dch), ch = img - b * (BWD ? q.C : q.O);
    const int rem = idx - img * (BWD ? q.H * q.W : q.oH * q.oW), py = div_f32(rem, k.dw), px = rem - py * (BWD ? q.W : q.oW);
    const int T = q.kH * q.kW;
    unsigned mask = 0;
    int xb, wb;
    if (BWD) {                                   // tap (ty0 + i sy, tx0 + j sx) reaches this element from output (oy0 - i, ox0 - j)
        const int iyPad = py + q.pt, ixPad = px + q.pl, oy0 = iyPad / q.sy, ox0 = ixPad / q.sx, ty0 = iyPad - oy0 * q.sy, tx0 = ixPad - ox0 * q.sx;
        for (int j = 0; j < k.nj; ++j) mask |= (unsigned)(tx0 + j * q.sx < q.kW && ox0 - j >= 0 && ox0 - j < q.oW) << j;
        for (int i = 0; i < k.ni; ++i) mask |= (unsigned)(ty0 + i * q.sy < q.kH && oy0 - i >= 0 && oy0 - i < q.oH) << (k.nj + i);
        xb = (b * q.O + (q.depthwise ? ch : 0)) * (q.oH * q.oW) + oy0 * q.oW + ox0;
        wb = ch * T + ty0 * q.kW + tx0;
    } else {
        const int iy0 = py * q.sy - q.pt, ix0 = px * q.sx - q.pl;
        for (int j = 0; j < k.nj; ++j) mask |= (unsigned)(ix0 + j >= 0 && ix0 + j < q.W) << j;
        for (int i = 0; i < k.ni; ++i) mask |= (unsigned)(iy0 + i >= 0 && iy0 + i < q.H) << (k.nj + i);
        xb = (b * q.C + (q.depthwise ? ch : 0)) * (q.H * q.W) + iy0 * q.W + ix0;
        wb = ch * q.Cw * T;
    }
    const float sum = SHAPE == 0 ? walk_f32(k, x, w, xb, wb, mask) : walk3x3_f32<SHAPE ? SHAPE : 1>(k, x, w, xb, wb, mask);
    float r = sum + (beta != 0.0f ? beta * out[idx] : 0.0f);
    if (bias) r = bias[ch] + r;
    out[idx] = r;
}

// Forward of a square kernel whose windows all lie inside the input (no padding), term for term the same sums again.  There is
// nothing to mask, so a product takes its two loads, at scalar addresses with the lane's offset, a multiplication and an
// addition (the walk above: about 14 instructions, which a wave alone on its SIMD issues one in 8 cycles), and the next
// channel's window is requested before this one's is added up.  32 x 6 x 14 x 14 -> 16 channels, 5x5: 20.1 us, now 6.0;
// 32 x 1 x 32 x 32 -> 6, 5x5: 8.6 and 4.0.
template <int KS>
__global__ __launch_bounds__(64) void conv_f32_window_kernel(ConvF32 q, WalkF32 k, const float* __restrict__ x, const float* __restrict__ w,
                                                             const float* __restrict__ bias, float beta, float* __restrict__ out, int total)
{
    constexpr int T = KS * KS;
    const int idx = blockIdx.x * 64 + threadIdx.x;
    if (idx >= total) return;
    const int img = div_f32(idx, k.dplane);      // image and channel
    const int b = div_f32(img, k.dch), ch = img - b * q.O;
    const int rem = idx - img * (q.oH * q.oW), py = div_f32(rem, k.dw), px = rem - py * q.oW;
    const unsigned xb = 4u * (unsigned)((b * q.C + (q.depthwise ? ch : 0)) * (q.H * q.W) + py * q.sy * q.W + px * q.sx), wb = 4u * (unsigned)(ch * q.Cw * T);
    struct Window { float x[T], w[T]; };
    const auto request = [&](int c, Window& v) {
        const char* const xc = (const char*)(x + (size_t)c * k.xo);
        const char* const wc = (const char*)(w + (size_t)c * T);
#pragma unroll
        for (int i = 0; i < KS; ++i)
#pragma unroll
            for (int j = 0; j < KS; ++j) {
                v.x[i * KS + j] = *(const float*)(xc + (size_t)i * q.W * 4 + 4 * j + xb);
                v.w[i * KS + j] = *(const float*)(wc + 4 * (i * KS + j) + wb);
            }
    };
    float sum = 0.0f;
    const auto add = [&](const Window& v) {
#pragma unroll
        for (int t = 0; t < T; ++t) sum = sum + v.w[t] * v.x[t];
    };
    Window even, odd;
    request(0, even);
    for (int c = 0; c < k.n; c += 2) {
        if (c + 1 < k.n) request(c + 1, odd);
        add(even);
        if (c + 1 >= k.n) break;
        if (c + 2 < k.n) request(c + 2, even);
        add(odd);
    }
    float r = sum + (beta != 0.0f ? beta * out[idx] : 0.0f);
    if (bias) r = bias[ch] + r;
    out[idx] = r;
}

// dw[o,c',ty,tx] = sum over batch and the output pixels whose tap (ty,tx) falls inside the input + beta * dw.
// One block per weight.
__global__ __launch_bounds__(TBLOCK) void conv_f32_backward_filter_kernel(ConvF32 q, const float* __restrict__ x, const float* __restrict__ dy,
                                                                          float beta, float* __restrict__ dw)
{
    const int widx = blockIdx.x;
    const int tx = widx % q.kW, ty = (widx / q.kW) % q.kH;
    const int cw = (widx / (q.kW * q.kH)) % q.Cw, o = widx / (q.kW * q.kH * q.Cw);
    const int c = q.depthwise ? o : cw;
    // ox range with 0 <= ox*sx + tx - pl < W
    const int oxMin = max((q.pl - tx + q.sx - 1) / q.sx, 0), oyMin = max((q.pt - ty + q.sy - 1) / q.sy, 0);
    const int oxMax = min((q.W + q.pl - tx + q.sx - 1) / q.sx, q.oW), oyMax = min((q.H + q.pt - ty + q.sy - 1) / q.sy, q.oH);
    const int nx = max(oxMax - oxMin, 0), ny = max(oyMax - oyMin, 0);
    const size_t total = (size_t)q.B * ny * nx;
    double acc = 0.0;
    for (size_t i = threadIdx.x; i < total; i += TBLOCK) {
        const int ox = oxMin + i % nx, oy = oyMin + (i / nx) % ny, b = i / ((size_t)nx * ny);
        const float xv = x[(((size_t)b * q.C + c) * q.H + (oy * q.sy + ty - q.pt)) * q.W + ox * q.sx + tx - q.pl];
        const float dv = dy[(((size_t)b * q.O + o) * q.oH + oy) * q.oW + ox];
        acc += (double)(xv * dv);
    }
    acc = block_sum_d(acc);
    if (threadIdx.x == 0)
        dw[widx] = (float)acc + (beta != 0.0f ? beta * dw[widx] : 0.0f);
}

// db[o] = sum over batch and pixels + beta * db.  One block per output channel.
__global__ __launch_bounds__(TBLOCK) void conv_f32_backward_bias_kernel(int B, int O, int plane, const float* __restrict__ dy, float beta,
                                                                        float* __restrict__ db)
{
    const int o = blockIdx.x;
    double acc = 0.0;
    for (size_t i = threadIdx.x; i < (size_t)B * plane; i += TBLOCK)
        acc += (double)dy[((size_t)(i / plane) * O + o) * plane + i % plane];
    acc = block_sum_d(acc);
    if (threadIdx.x == 0)
        db[o] = (float)acc + (beta != 0.0f ? beta * db[o] : 0.0f);
}

// Softmax over the channels of each pixel: exp(x - max) / sum, zeros if the sum is not positive.
// Bound by its chain of loads where there are few pixels and by reading x three times where there are many. N: channels held in
// registers, at least C, loaded once and all before the first is waited for; 0: any number, read in three loops. Measured, loops ->
// registers: 32 images of 10 classes 5.1 -> 3.4 us, 16 maps of 512 x 512 with 2 / 4 / 10 / 16 channels 21.0 -> 20.6, 39.5 -> 26.3,
// 136.5 -> 60.7, 237.5 -> 100.7 us.
template <int N>
__global__ __launch_bounds__(TBLOCK) void softmax_f32_kernel(const float* __restrict__ x, float* __restrict__ y, int B, int C, int plane)
{
    const size_t total = (size_t)B * plane;
    for (size_t idx = (size_t)blockIdx.x * TBLOCK + threadIdx.x; idx < total; idx += (size_t)gridDim.x * TBLOCK) {
        const size_t base = (idx / plane) * (size_t)C * plane + idx % plane;
        if (N) {
            float v[N ? N : 1];
#pragma unroll
            for (int c = 0; c < N; ++c) v[c] = x[base + (size_t)(c < C ? c : 0) * plane];
            float m = v[0];
#pragma unroll
            for (int c = 1; c < N; ++c) m = fmaxf(m, v[c]);                  // (past C: the first again)
            float s = 0.0f;
#pragma unroll
            for (int c = 0; c < N; ++c) {
                if (c >= C) break;
                v[c] = expf(v[c] - m);
                s += v[c];
            }
#pragma unroll
            for (int c = 0; c < N; ++c)
                if (c < C) y[base + (size_t)c * plane] = s > 0.0f ? v[c] / s : 0.0f;
            continue;
        }
        float m = x[base];
        for (int c = 1; c < C; ++c) m = fmaxf(m, x[base + (size_t)c * plane]);
        float s = 0.0f;
        for (int c = 0; c < C; ++c) s += expf(x[base + (size_t)c * plane] - m);
        for (int c = 0; c < C; ++c) y[base + (size_t)c * plane] = s > 0.0f ? expf(x[base + (size_t)c * plane] - m) / s : 0.0f;
    }
}

// diff = target - output, formed in double; partial[block] = sum of squares (double).
__global__ __launch_bounds__(TBLOCK) void loss_f32_kernel(const float* target, const float* __restrict__ out, float* diff,
                                                          size_t n, double* __restrict__ partial, double inv_batch, double* __restrict__ loss)
{
    double acc = 0.0;
    for (size_t i = (size_t)blockIdx.x * TBLOCK + threadIdx.x; i < n; i += (size_t)gridDim.x * TBLOCK) {
        const double e = (double)target[i] - (double)out[i];
        diff[i] = (float)e;
        acc += e * e;
    }
    acc = block_sum_d(acc);
    if (threadIdx.x) return;
    if (gridDim.x == 1) loss[0] = acc * inv_batch;
    else partial[blockIdx.x] = acc;
}
// Up to this many values one block goes over all of them and writes the loss itself, instead of a second launch that adds the blocks'
// partial sums: 320 / 2560 / 4096 values 3.9 / 4.0 / 4.0 us against 6.3 / 7.1 / 6.9 in two launches.
constexpr size_t LOSS_ONE_BLOCK = 4096;
__global__ __launch_bounds__(TBLOCK) void loss_finish_kernel(const double* __restrict__ partial, int nb, double inv_batch, double* __restrict__ loss)
{
    double acc = 0.0;
    for (int i = threadIdx.x; i < nb; i += TBLOCK) acc += partial[i];
    acc = block_sum_d(acc);
    if (threadIdx.x == 0) loss[0] = acc * inv_batch;
}

// The head of a learning net in one launch: softmax of few pixels, a thread each, targets - outputs and the loss from it, the
// gradient where the cell below reads it too (diff_x, or null).  The start of a launch bounds each of softmax, loss and copy: 32 images
// of 10 classes 2.9, 1.8 and 1.2 us in the kernels and as much between them, together 3.6.
template <int N>
__global__ __launch_bounds__(TBLOCK) void softmax_loss_f32_kernel(const float* __restrict__ x, const float* __restrict__ target, float* __restrict__ y,
                                                                  float* __restrict__ diff, float* __restrict__ diff_x, int total, int C, int plane, double inv_batch,
                                                                  double* __restrict__ loss)
{
    double acc = 0.0;
    for (int idx = threadIdx.x; idx < total; idx += TBLOCK) {
        const size_t base = (size_t)(idx / plane) * C * plane + idx % plane;
        float v[N], t[N];
#pragma unroll
        for (int c = 0; c < N; ++c) {
            const size_t at = base + (size_t)(c < C ? c : 0) * plane;
            v[c] = x[at];
            t[c] = target[at];
        }
        float m = v[0];
#pragma unroll
        for (int c = 1; c < N; ++c) m = fmaxf(m, v[c]);
        float s = 0.0f;
#pragma unroll
        for (int c = 0; c < N; ++c) {
            if (c >= C) break;
            v[c] = expf(v[c] - m);
            s += v[c];
        }
#pragma unroll
        for (int c = 0; c < N; ++c) {
            if (c >= C) break;
            const size_t at = base + (size_t)c * plane;
            const float o = s > 0.0f ? v[c] / s : 0.0f;
            const double e = (double)t[c] - (double)o;
            y[at] = o;
            diff[at] = (float)e;
            if (diff_x) diff_x[at] = (float)e;
            acc += e * e;
        }
    }
    acc = block_sum_d(acc);
    if (threadIdx.x == 0) loss[0] = acc * inv_batch;
}

// SGDSolver_Frame::update for one tensor.
// SGD updates of up to SGD_ITEMS tensors.  Most tensors of a net are small (scales, biases, steps), and a launch for each is
// what bounds an update; the blocks of one launch find their tensor in the table that comes with the arguments.  16 tensors
// of a small LeNet (61 k values): 16 launches of 1.7 us, now one of 3.8.  N: room in the table (2 KB of arguments for 32; a
// single tensor does not pay for them).
constexpr int SGD_ITEMS = 32;
template <int N>
struct SgdBatch {
    n2d2hip_sgd_item item[N];
    unsigned first[N + 1];                       // first block of a tensor; the grid behind the last
    int count;
};
// The update of value i by diff(i)
template <class F>
__device__ __forceinline__ void sgd_one(const n2d2hip_sgd_item& t, float* __restrict__ data, float* __restrict__ mom, size_t i, F diff)
{
    float v;
    if (mom) {
        float m = mom[i] * t.momentum;
        m += t.rate_diff * diff(i);
        if (t.decay_times_rate != 0.0f) m += -t.decay_times_rate * data[i];
        mom[i] = m;
        v = data[i] + m;
    } else {
        v = data[i] + t.rate_diff * diff(i);
    }
    data[i] = t.clamp ? fminf(fmaxf(v, t.clamp_min), t.clamp_max) : v;
}
template <int N>
__global__ __launch_bounds__(TBLOCK) void sgd_f32_kernel(SgdBatch<N> b)
{
    int k = 0;
    if (N > 1)
        while (k + 1 < b.count && blockIdx.x >= b.first[k + 1]) ++k;
    const n2d2hip_sgd_item& t = b.item[k];
    float* __restrict__ data = t.data;
    const float* __restrict__ diff = t.diff;
    float* __restrict__ mom = t.momentum_data;
    const size_t n = t.n, step = (size_t)(b.first[k + 1] - b.first[k]) * TBLOCK;
    for (size_t i = (size_t)(blockIdx.x - b.first[k]) * TBLOCK + threadIdx.x; i < n; i += step)
        sgd_one(t, data, mom, i, [=](size_t j) { return diff[j]; });
}
// With the SAT quantizers' gradients, which the update alone waits for: grad_of says which of `grad` an item's diff is, -1: it is there
// already.  A launch less at the end of every learning iteration, and one pass over the weights (240000 in six tensors, us: 4.8 + 5.2, now 6.1).
constexpr int SGD_GRADS = 16;
struct SgdSatBatch {
    SgdBatch<SGD_ITEMS> sgd;
    n2d2hip_sat_weight_grad_item grad[SGD_GRADS];
    float mode_factor[SGD_GRADS];
    signed char grad_of[SGD_ITEMS];
};
static_assert(sizeof(SgdSatBatch) <= 4096, "a launch's arguments");
__global__ __launch_bounds__(TBLOCK) void sgd_sat_f32_kernel(SgdSatBatch b)
{
    int k = 0;
    while (k + 1 < b.sgd.count && blockIdx.x >= b.sgd.first[k + 1]) ++k;
    const n2d2hip_sgd_item& t = b.sgd.item[k];
    const int from = b.grad_of[k];
    float* __restrict__ data = t.data;
    float* __restrict__ mom = t.momentum_data;
    const size_t n = t.n, step = (size_t)(b.sgd.first[k + 1] - b.sgd.first[k]) * TBLOCK;
    const size_t i0 = (size_t)(blockIdx.x - b.sgd.first[k]) * TBLOCK + threadIdx.x;
    if (from < 0) {
        const float* __restrict__ diff = t.diff;
        for (size_t i = i0; i < n; i += step) sgd_one(t, data, mom, i, [=](size_t j) { return diff[j]; });
    } else {
        const n2d2hip_sat_weight_grad_item& s = b.grad[from];
        const float inv_factor = sat_weight_inv_factor(s), mode_factor = b.mode_factor[from];
        for (size_t i = i0; i < n; i += step) {
            const float d = sat_weight_gradient(data[i], s.diff_wq[i], inv_factor, mode_factor);
            s.diff_w[i] = d;
            sgd_one(t, data, mom, i, [=](size_t) { return d; });
        }
    }
}

// Rectifier on a float tensor, in place: x > 0 ? min(x, clipping) : leak * x (clipping == 0: none).
__global__ __launch_bounds__(TBLOCK) void rectifier_f32_forward_kernel(float* __restrict__ x, size_t n, float leak, float clipping)
{
    for (size_t i = (size_t)blockIdx.x * TBLOCK + threadIdx.x; i < n; i += (size_t)gridDim.x * TBLOCK) {
        const float v = x[i];
        x[i] = v > 0.0f ? (clipping > 0.0f ? fminf(v, clipping) : v) : leak * v;
    }
}
// diff_out = diff_in * (out == clipping ? 0 : out > 0 ? 1 : leak); `out` is what the cell holds after its activation.
__global__ __launch_bounds__(TBLOCK) void rectifier_f32_backward_kernel(const float* __restrict__ out, const float* diff_in,
                                                                        float* diff_out, size_t n, float leak, float clipping)
{
    for (size_t i = (size_t)blockIdx.x * TBLOCK + threadIdx.x; i < n; i += (size_t)gridDim.x * TBLOCK) {
        const float o = out[i];
        const float f = (clipping > 0.0f && o == clipping) ? 0.0f : (o > 0.0f ? 1.0f : leak);
        diff_out[i] = diff_in[i] * f;
    }
}

// The sums over one channel of NCHW tensors.  Memory bounds them.  A block takes a range of the channel's units of V values,
// which lie in B planes: the plane and the place in it come from a 32-bit division by multiplication (the compiler's 64-bit
// one, per value, took longer than the loads), and 16-byte loads where every plane starts on such a boundary (V 4).  V 0: the
// units of V 1 counted in 64 bits, for channels of 2^31 values and more.
struct BnRange {
    int C, plane;
    int unit_plane;                              // units of a plane
    DivF32 dplane;                               // division by it
    size_t units, chunk;                         // units of the channel, and of a block
};
template <int V, class F>
__device__ __forceinline__ void bn_walk(const BnRange& q, int c, F f)
{
    const size_t u0 = (size_t)blockIdx.y * q.chunk, u1 = u0 + q.chunk < q.units ? u0 + q.chunk : q.units;
    if (V == 0) {
        for (size_t u = u0 + threadIdx.x; u < u1; u += blockDim.x)
            f(((size_t)(u / q.plane) * q.C + c) * q.plane + u % q.plane);
        return;
    }
#pragma unroll 4
    for (int u = (int)u0 + (int)threadIdx.x; u < (int)u1; u += (int)blockDim.x) {
        const int b = div_f32(u, q.dplane);
        f(((size_t)b * q.C + c) * q.plane + (size_t)(u - b * q.unit_plane) * (V ? V : 1));
    }
}
template <int V>
__device__ __forceinline__ void bn_load(float* dst, const float* __restrict__ p, size_t idx)
{
    if (V == 4) {
        const float4 v = *(const float4*)(p + idx);
        dst[0] = v.x; dst[1] = v.y; dst[2] = v.z; dst[3] = v.w;
    } else {
        dst[0] = p[idx];
    }
}
// Adds each of the N values over the block (256 or 1024 threads)
template <int N>
__device__ __forceinline__ void bn_block_sums(double* v)
{
    __shared__ double red[16][N];
#pragma unroll
    for (int k = 0; k < N; ++k) {
        v[k] = wave_sum_d(v[k]);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][k] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < N; ++k) {
        v[k] = 0.0;
        for (int i = 0; i < (int)(blockDim.x >> 6); ++i) v[k] += red[i][k];
    }
}
// Adds the partial sums of a channel's blocks (at most 64 of N values each), a lane of the wavefront for each block
template <int N>
__device__ __forceinline__ void bn_partial_sums(double* v, const double* __restrict__ p, int splits)
{
#pragma unroll
    for (int k = 0; k < N; ++k)
        v[k] = wave_sum_d((int)threadIdx.x < splits ? p[(size_t)threadIdx.x * N + k] : 0.0);
}

// Batch statistics: mean, then the mean of the squared deviations from the mean as rounded to float (the reference's two
// passes), and the running statistics' step towards them (the variance with the factor size / (size - 1)).  One pass over x:
// beside the sum of x it adds x - s and its square in double, s being the channel's first value, and moves the squares from s to
// the mean afterwards.  As s is one of the n values, (s - mean)^2 is at most n variances, so what cancels costs at most n times
// 2^-53 of the variance.  64 channels, 56 x 56, batch 64: two passes and the last step 56.8 us, now 12.4 and 4.8.
__device__ __forceinline__ void bn_stats(double n, float shift, const double* t, float* m, float* v)
{
    *m = (float)(t[0] / n);
    const double e = (double)*m - (double)shift;
    const double squares = t[2] - 2.0 * e * t[1] + n * e * e;
    *v = (float)((squares < 0.0 ? 0.0 : squares) / n);
}
__device__ __forceinline__ void bn_write_stats(int c, double n, float m, float v, float* __restrict__ mean, float* __restrict__ variance,
                                               float* __restrict__ saved_mean, float* __restrict__ saved_variance, double momentum)
{
    saved_mean[c] = m;
    saved_variance[c] = v;
    const float unbiased = v * ((float)n / ((float)n - 1.0f));
    mean[c] = (float)((double)m * momentum + (double)mean[c] * (1.0 - momentum));
    variance[c] = (float)((double)unbiased * momentum + (double)variance[c] * (1.0 - momentum));
}
// -> the shift, and in t the block's sums of x, x - shift and (x - shift)^2 over its range of channel c
template <int V>
__device__ __forceinline__ float bn_channel_sums(const BnRange& q, int c, const float* __restrict__ x, double* t)
{
    constexpr int N = V ? V : 1;
    const float shift = x[(size_t)c * q.plane];
    t[0] = t[1] = t[2] = 0.0;
    bn_walk<V>(q, c, [&](size_t idx) {
        float v[N];
        bn_load<N>(v, x, idx);
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const double d = (double)v[k] - (double)shift;
            t[0] += (double)v[k];
            t[1] += d;
            t[2] += d * d;
        }
    });
    bn_block_sums<3>(t);
    return shift;
}
template <int V>
__device__ __forceinline__ void bn_store(float* p, size_t idx, const float* v)
{
    if (V == 4) *(float4*)(p + idx) = make_float4(v[0], v[1], v[2], v[3]);
    else p[idx] = v[0];
}

// V values normalised (mean m, var the root), scaled by g, b added, and quantized
template <int V, bool SAT>
__device__ __forceinline__ void bn_apply(size_t idx, const float* __restrict__ x, float m, float var, float g, float b, const SatStore& sat, float a,
                                         float* __restrict__ y)
{
    float t[V];
    bn_load<V>(t, x, idx);
#pragma unroll
    for (int k = 0; k < V; ++k) t[k] = g * ((t[k] - m) / var) + b;
    if (SAT) {
        if (sat.fp) bn_store<V>(sat.fp, idx, t);
#pragma unroll
        for (int k = 0; k < V; ++k) t[k] = sat_quantize(t[k], sat.range, a);
    }
    bn_store<V>(y, idx, t);
}

// The 2x2 max pooling behind a normalisation and its quantizer: planes of whole windows, taken in units of two rows by VW columns.  On its own
// the pooling of a small net is a launch that lasts as long as a launch does, each way; here it comes from values that are in registers.
// us, launches one behind the other / joined: 32 x 6 x 28 x 28 forwards 4.5 + 4.8 + 3.4 / 4.6 + 5.6, backwards 3.2 + 6.1 / 5.7; 32 x 16 x 10 x 10 5.9 + 3.3 / 7.2,
// 3.2 + 6.3 / 6.6; a LeNet iteration of 32 images 167 / 154.
struct BnPool {
    BnRange units;                               // unit_plane and dplane: the units of a plane; plane: its values
    int W, row_units;                            // columns of a plane, units of two rows
    DivF32 drow;                                 // division by row_units
    float* y;
    int* argmax;
};
// f(first value of a unit, the same within its plane, its first window) over the block's range of channel c
template <int VW, class F>
__device__ __forceinline__ void bn_walk_windows(const BnPool& p, int c, F f)
{
    const BnRange& q = p.units;
    const size_t u0 = (size_t)blockIdx.y * q.chunk, u1 = u0 + q.chunk < q.units ? u0 + q.chunk : q.units;
    for (int u = (int)u0 + (int)threadIdx.x; u < (int)u1; u += (int)blockDim.x) {
        const int b = div_f32(u, q.dplane), in = u - b * q.unit_plane, row = div_f32(in, p.drow), col = in - row * p.row_units;
        const size_t plane = (size_t)b * q.C + c;
        const int first = 2 * row * p.W + col * VW;
        f(plane * q.plane + first, first, plane * (q.plane / 4) + (size_t)row * (p.W / 2) + col * (VW / 2));
    }
}
template <int VW>
__device__ __forceinline__ void bn_load_row(float* dst, const float* __restrict__ p, size_t idx)
{
    if (VW == 4) {
        bn_load<4>(dst, p, idx);
    } else {
        const float2 v = *(const float2*)(p + idx);
        dst[0] = v.x; dst[1] = v.y;
    }
}
template <int VW>
__device__ __forceinline__ void bn_store_row(float* p, size_t idx, const float* v)
{
    if (VW == 4) bn_store<4>(p, idx, v);
    else *(float2*)(p + idx) = make_float2(v[0], v[1]);
}
// A unit normalised, quantized and pooled: of a window's values the first largest in row-major order
template <int VW>
__device__ __forceinline__ void bn_apply_windows(size_t idx, int first, size_t window, const BnPool& p, const float* __restrict__ x, float m, float var,
                                                 float g, float b, const SatStore& sat, float a, float* __restrict__ y)
{
    float t[2][VW];
#pragma unroll
    for (int r = 0; r < 2; ++r) bn_load_row<VW>(t[r], x, idx + r * p.W);
#pragma unroll
    for (int r = 0; r < 2; ++r) {
#pragma unroll
        for (int k = 0; k < VW; ++k) t[r][k] = g * ((t[r][k] - m) / var) + b;
        if (sat.fp) bn_store_row<VW>(sat.fp, idx + r * p.W, t[r]);
#pragma unroll
        for (int k = 0; k < VW; ++k) t[r][k] = sat_quantize(t[r][k], sat.range, a);
        bn_store_row<VW>(y, idx + r * p.W, t[r]);
    }
#pragma unroll
    for (int w = 0; w < VW / 2; ++w) {
        float best = t[0][2 * w];
        int where = first + 2 * w;
#pragma unroll
        for (int k = 1; k < 4; ++k)
            if (t[k / 2][2 * w + k % 2] > best) {
                best = t[k / 2][2 * w + k % 2];
                where = first + (k / 2) * p.W + 2 * w + k % 2;
            }
        p.y[window + w] = best;
        p.argmax[window + w] = where;
    }
}

// A channel per blockIdx.x in gridDim.y blocks: one finishes by itself, several leave their sums in ws.  With BN_APPLY or BN_APPLY_SAT the
// one block normalises its channel too, as the kernel below does, and reads it again mostly from its cache (when, and what it gives: bn_whole()).
// BN_APPLY_SAT_POOL + VW: and pools, in units of VW columns.
enum { BN_SUMS_ONLY, BN_APPLY, BN_APPLY_SAT, BN_APPLY_SAT_POOL };
template <int V, int THEN>
__global__ __launch_bounds__(1024) void batchnorm_f32_stats_kernel(BnRange q, double n, const float* __restrict__ x, double* __restrict__ ws,
                                                                   float* __restrict__ mean, float* __restrict__ variance, float* __restrict__ saved_mean,
                                                                   float* __restrict__ saved_variance, double momentum, const float* __restrict__ scale,
                                                                   const float* __restrict__ bias, double epsilon, SatStore sat, float* __restrict__ y,
                                                                   BnPool pool)
{
    const int c = blockIdx.x;
    float g = 0.0f, b = 0.0f, a = 0.0f;          // (loaded ahead of the sums)
    if constexpr (THEN != BN_SUMS_ONLY) { g = scale[c]; b = bias[c]; }
    if constexpr (THEN >= BN_APPLY_SAT) a = fabsf(sat.alpha[0]);
    double t[3];
    const float shift = bn_channel_sums<V>(q, c, x, t);
    if (THEN == BN_SUMS_ONLY && threadIdx.x) return;
    if (THEN == BN_SUMS_ONLY && gridDim.y > 1) {
        double* o = ws + ((size_t)c * gridDim.y + blockIdx.y) * 4;
        o[0] = t[0]; o[1] = t[1]; o[2] = t[2]; o[3] = (double)shift;
        return;
    }
    float m, v;
    bn_stats(n, shift, t, &m, &v);
    if (threadIdx.x == 0) bn_write_stats(c, n, m, v, mean, variance, saved_mean, saved_variance, momentum);
    if constexpr (THEN != BN_SUMS_ONLY) {
        const float var = (float)sqrt((double)v + epsilon);
        if constexpr (THEN > BN_APPLY_SAT_POOL) {
            constexpr int VW = THEN - BN_APPLY_SAT_POOL;
            bn_walk_windows<VW>(pool, c, [&](size_t idx, int first, size_t window) { bn_apply_windows<VW>(idx, first, window, pool, x, m, var, g, b, sat, a, y); });
        } else {
            bn_walk<V>(q, c, [&](size_t idx) { bn_apply<V, THEN == BN_APPLY_SAT>(idx, x, m, var, g, b, sat, a, y); });
        }
    }
}
// The statistics of a channel from its blocks' sums, by the first wavefront of the block that asks
__device__ __forceinline__ void bn_split_stats(int c, double n, int splits, const double* __restrict__ ws, float* m, float* v)
{
    const double* p = ws + (size_t)c * splits * 4;
    double t[3];
#pragma unroll
    for (int k = 0; k < 3; ++k)
        t[k] = wave_sum_d((int)threadIdx.x < splits ? p[(size_t)threadIdx.x * 4 + k] : 0.0);
    bn_stats(n, (float)p[3], t, m, v);
}
__global__ __launch_bounds__(64) void batchnorm_f32_stats_finish_kernel(double n, int splits, const double* __restrict__ ws, float* __restrict__ mean,
                                                                        float* __restrict__ variance, float* __restrict__ saved_mean,
                                                                        float* __restrict__ saved_variance, double momentum)
{
    const int c = blockIdx.x;
    float m, v;
    bn_split_stats(c, n, splits, ws, &m, &v);
    if (threadIdx.x == 0) bn_write_stats(c, n, m, v, mean, variance, saved_mean, saved_variance, momentum);
}

// y = scale * (x - mean) / sqrt(variance + epsilon) + bias.  eps_in_float: the inference branch of the reference adds
// the epsilon in float and takes a float square root; the learning branch adds the double and rounds the root.
// A channel per blockIdx.x, in ranges of its units as the sums: what a channel needs is worked out once a block, from the sums
// of the statistics' blocks too (splits > 1), for which a launch of C blocks stood in between.  The block of a channel's first
// range writes the statistics.  The quantizer that follows a normalisation in a learning net is applied on the way out; it read
// and wrote the tensor again.  64 x 64 x 32 x 32, us: statistics, their end, this and the quantizer 5.8 + 4.8 + 6.1 + 10.5, now
// 6.0 + 12.9, of which 10 are the 50 MB.
// POOL: 0, or the columns of a unit of windows, which are pooled on the way out too (SAT only).
template <int V, bool SAT, int POOL = 0>
__global__ __launch_bounds__(TBLOCK) void batchnorm_f32_apply_kernel(BnRange q, int splits, double n, const double* __restrict__ ws, float* __restrict__ mean,
                                                                     float* __restrict__ variance, float* __restrict__ saved_mean,
                                                                     float* __restrict__ saved_variance, double momentum, int running,
                                                                     const float* __restrict__ x, const float* __restrict__ scale, const float* __restrict__ bias, double epsilon,
                                                                     SatStore sat, float* __restrict__ y, BnPool pool)
{
    const int c = blockIdx.x;
    float m, v;
    if (splits > 1) {
        __shared__ float stats[2];
        if (threadIdx.x < 64) {
            bn_split_stats(c, n, splits, ws, &m, &v);
            if (threadIdx.x == 0) {
                stats[0] = m; stats[1] = v;
                if (blockIdx.y == 0) bn_write_stats(c, n, m, v, mean, variance, saved_mean, saved_variance, momentum);
            }
        }
        __syncthreads();
        m = stats[0]; v = stats[1];
    } else {
        m = running ? mean[c] : saved_mean[c];
        v = running ? variance[c] : saved_variance[c];
    }
    const float var = running ? sqrtf(v + (float)epsilon) : (float)sqrt((double)v + epsilon);
    const float g = scale[c], b = bias[c];
    const float a = SAT ? fabsf(sat.alpha[0]) : 0.0f;
    if constexpr (POOL != 0)
        bn_walk_windows<POOL>(pool, c, [&](size_t idx, int first, size_t window) { bn_apply_windows<POOL>(idx, first, window, pool, x, m, var, g, b, sat, a, y); });
    else
        bn_walk<V>(q, c, [&](size_t idx) { bn_apply<V, SAT>(idx, x, m, var, g, b, sat, a, y); });
}

// The same for small planes, whose channels lie in pieces, and for channels past 32-bit counts: one lane per value, the
// channel found by division.
__global__ __launch_bounds__(TBLOCK) void batchnorm_f32_apply_flat_kernel(size_t total, int C, int plane, const float* __restrict__ x,
                                                                     const float* __restrict__ scale, const float* __restrict__ bias,
                                                                     const float* __restrict__ mean, const float* __restrict__ variance, double epsilon,
                                                                     int eps_in_float, SatStore sat, float* __restrict__ y)
{
    const float a = sat.alpha ? fabsf(sat.alpha[0]) : 0.0f;
    for (size_t i = (size_t)blockIdx.x * TBLOCK + threadIdx.x; i < total; i += (size_t)gridDim.x * TBLOCK) {
        const int c = (int)((i / plane) % C);
        const float var = eps_in_float ? sqrtf(variance[c] + (float)epsilon) : (float)sqrt((double)variance[c] + epsilon);
        const float normalized = (x[i] - mean[c]) / var;
        float o = scale[c] * normalized + bias[c];
        if (sat.alpha) {
            if (sat.fp) sat.fp[i] = o;
            o = sat_quantize(o, sat.range, a);
        }
        y[i] = o;
    }
}

// The sums of BatchNormCell_Frame<T>::backPropagate over one channel, and what follows from them, in blocks as above.  Its five are
// multiples of three, d the values of dy and c those of x - mean: the sums of d c, of d and of c.  Those are what the blocks add up, in
// double and the products unrounded; the factors (scale, 1 / sigma, -2) come in once a channel.  With a division and five conversions
// a value the vector units took longer than the memory.  This pass and the next, us, before / now: 64 x 64 x 32 x 32 19.7 / 15.7,
// behind a quantizer 27.7 / 23.5; 128 channels, 56 x 56, batch 32 45.6 / 42.2; 256, 14 x 14, batch 33 14.5 / 11.1; 32, 112 x 112, batch 8
// 18.7 / 13.4; 6, 28 x 28, batch 32 9.7 / 7.5.  Errors against 64 bits are the same or smaller (dx 1.1e-7 / 0.7e-7).
constexpr int BN_SUMS = 3;
struct BnGrads { float* diff_scale; float* diff_bias; float* diff_saved_mean; float* diff_saved_variance; float beta_scale, beta_bias; };
// (sigma is rounded to float, as the forward pass has it)
__device__ __forceinline__ double bn_inv_sigma(float saved_variance, double epsilon) { return 1.0 / (double)(float)sqrt((double)saved_variance + epsilon); }
// -> the reference's five: of d c / sigma, d, d scale, -2 c, d scale c
__device__ __forceinline__ void bn_five_sums(double* t, const double* s, float scale, double inv_sigma)
{
    t[0] = s[0] * inv_sigma;
    t[1] = s[1];
    t[2] = (double)scale * s[1];
    t[3] = -2.0 * s[2];
    t[4] = (double)scale * s[0];
}
__device__ __forceinline__ void bn_stats_grads(double n, const double* t, float saved_variance, double epsilon, float* dmean, float* dvariance)
{
    const float sum_mean1 = (float)t[2], sum_mean2 = (float)t[3], sum_var = (float)t[4];
    const double square = (double)saved_variance + epsilon, root = sqrt(square);
    const float var = (float)root;
    *dvariance = (float)((double)sum_var * (-1.0 / 2.0) / (square * root));      // (to the power -3/2; pow() took longer than the sums)
    *dmean = (float)((double)sum_mean1 * (-1.0 / (double)var) + (double)(*dvariance * sum_mean2 / (float)n));
}
__device__ __forceinline__ void bn_write_grads(int c, const double* t, float dmean, float dvariance, const BnGrads& o)
{
    const float sum_scale = (float)t[0], sum_bias = (float)t[1];
    o.diff_saved_variance[c] = dvariance;
    o.diff_saved_mean[c] = dmean;
    o.diff_scale[c] = sum_scale + (o.beta_scale != 0.0f ? o.beta_scale * o.diff_scale[c] : 0.0f);
    o.diff_bias[c] = sum_bias + (o.beta_bias != 0.0f ? o.beta_bias * o.diff_bias[c] : 0.0f);
}
// The SAT activation quantizer behind a normalisation, backwards: fp what went into it, alpha's gradient summed by block (partial,
// a value for each block of the sums) and finished by the launch that follows; alpha null: no quantizer
struct BnSatGrad {
    const float* fp;
    float range;
    const float* alpha;
    double* partial;
    int blocks;
    float beta;
    float* diff_alpha;
};
// (one block: the sum of the blocks' values + beta times what was there)
__device__ __forceinline__ void bn_finish_alpha(const BnSatGrad& sat)
{
    double t[1] = {};
    for (int i = threadIdx.x; i < sat.blocks; i += TBLOCK) t[0] += sat.partial[i];
    bn_block_sums<1>(t);
    if (threadIdx.x == 0) sat.diff_alpha[0] = (float)t[0] + (sat.beta != 0.0f ? sat.beta * sat.diff_alpha[0] : 0.0f);
}
__global__ __launch_bounds__(TBLOCK) void batchnorm_f32_alpha_kernel(BnSatGrad sat) { bn_finish_alpha(sat); }

// Three sums of V values of x and of the gradient in dv
template <int N>
__device__ __forceinline__ void bn_grad_terms(double* s, const float* xv, const float* dv, float m)
{
#pragma unroll
    for (int k = 0; k < N; ++k) {
        const double centred = (double)(xv[k] - m), d = (double)dv[k];
        s[0] = __fma_rn(d, centred, s[0]);
        s[1] += d;
        s[2] += centred;
    }
}
// dx = dy * scale / sigma + dVar * 2 (x - mean) / size + dMean / size.  In double, what a channel's values share worked out once a block:
// dx = kd d + kc (x - mean) + k0, where there were two divisions a value, one of them in double (figures at the sums).
struct BnData {
    float m;
    double kd, kc, k0;
    __device__ BnData(float mean, float scale, double inv_sigma, float dmean, float dvariance, float size)
        : m(mean), kd((double)scale * inv_sigma), kc((double)dvariance * 2.0 / (double)size), k0((double)(dmean / size))
    {
    }
    template <int V>
    __device__ void value(size_t idx, const float* __restrict__ x, const float* dy, float* dx) const
    {
        float xv[V], dv[V];
        bn_load<V>(xv, x, idx);
        bn_load<V>(dv, dy, idx);
#pragma unroll
        for (int k = 0; k < V; ++k) dv[k] = (float)__fma_rn(kd, (double)dv[k], __fma_rn(kc, (double)(xv[k] - m), k0));
        bn_store<V>(dx, idx, dv);
    }
};

// SAT: dy is first taken through the quantizer's gradient, in place (64 x 64 x 32 x 32, us: the quantizer's own pass 10.0, its end
// 4.6 and the sums, then 9.8; together then 19.2)
// POOL: 0, or the columns of a unit of the windows behind the quantizer: dy is not read but made from the pooled tensor's gradient (in
// pool.y), whose window chose one value each.
template <int V, bool SAT, int POOL = 0>
__global__ __launch_bounds__(1024) void batchnorm_f32_backward_sums_kernel(BnRange q, double n, const float* __restrict__ x,
                                                                           const float* __restrict__ scale, const float* __restrict__ saved_mean,
                                                                           const float* __restrict__ saved_variance, double epsilon,
                                                                           float* __restrict__ dy, double* __restrict__ ws, BnGrads grads, BnSatGrad sat,
                                                                           BnPool pool)
{
    constexpr int N = V ? V : 1;
    const int c = blockIdx.x;
    const float m = saved_mean[c], g = scale[c], variance = saved_variance[c];
    const double inv_sigma = bn_inv_sigma(variance, epsilon);
    const float a = SAT ? fabsf(sat.alpha[0]) : 0.0f;
    double s[SAT ? BN_SUMS + 1 : BN_SUMS] = {};
    if constexpr (POOL != 0) bn_walk_windows<POOL>(pool, c, [&](size_t idx, int first, size_t window) {
        float d[POOL / 2], xv[2][POOL], fp[2][POOL];
        int at[POOL / 2];
#pragma unroll
        for (int w = 0; w < POOL / 2; ++w) { d[w] = pool.y[window + w]; at[w] = pool.argmax[window + w] - first; }
#pragma unroll
        for (int r = 0; r < 2; ++r) { bn_load_row<POOL>(xv[r], x, idx + r * pool.W); bn_load_row<POOL>(fp[r], sat.fp, idx + r * pool.W); }
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            float dv[POOL];
#pragma unroll
            for (int k = 0; k < POOL; ++k) {
                dv[k] = at[k / 2] == r * pool.W + k ? d[k / 2] : 0.0f;
                s[BN_SUMS] += (double)__fmul_rn(sat_alpha_slope(fp[r][k], sat.range, a), dv[k]);
                dv[k] = __fmul_rn(sat_input_slope(fp[r][k], a), dv[k]);
            }
            bn_store_row<POOL>(dy, idx + r * pool.W, dv);
            bn_grad_terms<POOL>(s, xv[r], dv, m);
        }
    });
    else bn_walk<V>(q, c, [&](size_t idx) {
        float xv[N], dv[N];
        bn_load<N>(xv, x, idx);
        bn_load<N>(dv, dy, idx);
        if constexpr (SAT) {
            float fp[N];
            bn_load<N>(fp, sat.fp, idx);
#pragma unroll
            for (int k = 0; k < N; ++k) {
                s[BN_SUMS] += (double)__fmul_rn(sat_alpha_slope(fp[k], sat.range, a), dv[k]);
                dv[k] = __fmul_rn(sat_input_slope(fp[k], a), dv[k]);
            }
            bn_store<N>(dy, idx, dv);
        }
        bn_grad_terms<N>(s, xv, dv, m);
    });
    bn_block_sums<SAT ? BN_SUMS + 1 : BN_SUMS>(s);
    if (threadIdx.x) return;
    if constexpr (SAT) sat.partial[(size_t)c * gridDim.y + blockIdx.y] = s[BN_SUMS];
    if (gridDim.y == 1) {
        double t[5];
        float dmean, dvariance;
        bn_five_sums(t, s, g, inv_sigma);
        bn_stats_grads(n, t, variance, epsilon, &dmean, &dvariance);
        bn_write_grads(c, t, dmean, dvariance, grads);
    } else {
        double* o = ws + ((size_t)c * gridDim.y + blockIdx.y) * BN_SUMS;
        o[0] = s[0]; o[1] = s[1]; o[2] = s[2];
    }
}
__global__ __launch_bounds__(64) void batchnorm_f32_backward_finish_kernel(double n, int splits, const double* __restrict__ ws, const float* __restrict__ scale,
                                                                           const float* __restrict__ saved_variance, double epsilon, BnGrads grads)
{
    const int c = blockIdx.x;
    double s[BN_SUMS], t[5];
    bn_partial_sums<BN_SUMS>(s, ws + (size_t)c * splits * BN_SUMS, splits);
    if (threadIdx.x) return;
    bn_five_sums(t, s, scale[c], bn_inv_sigma(saved_variance[c], epsilon));
    float dmean, dvariance;
    bn_stats_grads(n, t, saved_variance[c], epsilon, &dmean, &dvariance);
    bn_write_grads(c, t, dmean, dvariance, grads);
}

// Sums and values of channels that one block adds up, in one launch (when, and what it gives: bn_whole()).  dx may be dy.
template <int V>
__global__ __launch_bounds__(1024) void batchnorm_f32_backward_whole_kernel(BnRange q, double n, float size, const float* __restrict__ x,
                                                                            const float* __restrict__ scale, const float* __restrict__ saved_mean,
                                                                            const float* __restrict__ saved_variance, double epsilon, const float* dy,
                                                                            BnGrads grads, float* dx)
{
    const int c = blockIdx.x;
    const float m = saved_mean[c], g = scale[c], variance = saved_variance[c];
    double s[BN_SUMS] = {}, t[5];
    bn_walk<V>(q, c, [&](size_t idx) {
        float xv[V], dv[V];
        bn_load<V>(xv, x, idx);
        bn_load<V>(dv, dy, idx);
        bn_grad_terms<V>(s, xv, dv, m);
    });
    const double inv_sigma = bn_inv_sigma(variance, epsilon);
    bn_block_sums<BN_SUMS>(s);
    float dmean, dvariance;
    bn_five_sums(t, s, g, inv_sigma);
    bn_stats_grads(n, t, variance, epsilon, &dmean, &dvariance);
    if (threadIdx.x == 0) bn_write_grads(c, t, dmean, dvariance, grads);
    const BnData data(m, g, inv_sigma, dmean, dvariance, size);
    bn_walk<V>(q, c, [&](size_t idx) { data.value<V>(idx, x, dy, dx); });
}

// The values (BnData), in ranges of a channel as the apply kernel, the end of the sums before it with it.
template <int V>
__global__ __launch_bounds__(TBLOCK) void batchnorm_f32_backward_data_kernel(BnRange q, int splits, double n, const double* __restrict__ ws, float size,
                                                                            const float* __restrict__ x, const float* __restrict__ scale,
                                                                            const float* __restrict__ saved_mean, const float* __restrict__ saved_variance,
                                                                            double epsilon, const float* dy, BnGrads grads, BnSatGrad sat, float* dx)
{
    const int c = blockIdx.x;
    if (sat.alpha && blockIdx.x == 0 && blockIdx.y == gridDim.y - 1) {
        bn_finish_alpha(sat);
        __syncthreads();
    }
    const float m = saved_mean[c], g = scale[c], variance = saved_variance[c];
    const double inv_sigma = bn_inv_sigma(variance, epsilon);
    float dmean, dvariance;
    if (splits > 1) {
        __shared__ float of_stats[2];
        if (threadIdx.x < 64) {
            double s[BN_SUMS], t[5];
            bn_partial_sums<BN_SUMS>(s, ws + (size_t)c * splits * BN_SUMS, splits);
            if (threadIdx.x == 0) {
                bn_five_sums(t, s, g, inv_sigma);
                bn_stats_grads(n, t, variance, epsilon, &dmean, &dvariance);
                of_stats[0] = dmean; of_stats[1] = dvariance;
                if (blockIdx.y == 0) bn_write_grads(c, t, dmean, dvariance, grads);
            }
        }
        __syncthreads();
        dmean = of_stats[0]; dvariance = of_stats[1];
    } else {
        dmean = grads.diff_saved_mean[c];
        dvariance = grads.diff_saved_variance[c];
    }
    const BnData data(m, g, inv_sigma, dmean, dvariance, size);
    bn_walk<V>(q, c, [&](size_t idx) { data.value<V>(idx, x, dy, dx); });
}

// The same for small planes: one lane per value.
__global__ __launch_bounds__(TBLOCK) void batchnorm_f32_backward_data_flat_kernel(size_t total, int C, int plane, float size, const float* __restrict__ x,
                                                                            const float* __restrict__ scale, const float* __restrict__ saved_mean,
                                                                            const float* __restrict__ saved_variance, double epsilon, const float* dy,
                                                                            const float* __restrict__ diff_saved_mean,
                                                                            const float* __restrict__ diff_saved_variance, BnSatGrad sat, float* dx)
{
    if (sat.alpha && blockIdx.x == 0) bn_finish_alpha(sat);
    for (size_t i = (size_t)blockIdx.x * TBLOCK + threadIdx.x; i < total; i += (size_t)gridDim.x * TBLOCK) {
        const int c = (int)((i / plane) % C);
        const BnData data(saved_mean[c], scale[c], bn_inv_sigma(saved_variance[c], epsilon), diff_saved_mean[c], diff_saved_variance[c], size);
        data.value<1>(i, x, dy, dx);
    }
}

struct PoolF32 {
    int B, C, H, W, oH, oW, pw, ph, sx, sy, px, py;
    DivF32 dw, dh, dow, doh, dsx, dsy;           // division by W, H, oW, oH, sx, sy
};
// Row, column and plane of element i of planes of h x w.  SMALL: the tensor has less than 2^31 elements, and the divisions are
// multiplications (the compiler's 64-bit ones, two a value and two more a window, were most of the time: 64 x 64 x 32 x 32, 2x2:
// backward 22.2 us, now 13.9).
template <bool SMALL>
__device__ __forceinline__ void pool_place(size_t i, int w, int h, DivF32 dw, DivF32 dh, int* ix, int* iy, size_t* plane)
{
    if (SMALL) {
        const int row = div_f32((int)i, dw), bc = div_f32(row, dh);
        *ix = (int)i - row * w;
        *iy = row - bc * h;
        *plane = bc;
    } else {
        *ix = (int)(i % w);
        *iy = (int)((i / w) % h);
        *plane = i / ((size_t)w * h);
    }
}

// Max pooling of float NCHW with the unit mapping; argmax keeps iy * W + ix of the first largest element of the
// window in row-major order (-1: empty window, output 0).
template <bool SMALL>
__global__ __launch_bounds__(TBLOCK) void pool_max_f32_forward_kernel(PoolF32 q, const float* __restrict__ x, float* __restrict__ y, int* __restrict__ argmax)
{
    const size_t total = (size_t)q.B * q.C * q.oH * q.oW;
    for (size_t i = (size_t)blockIdx.x * TBLOCK + threadIdx.x; i < total; i += (size_t)gridDim.x * TBLOCK) {
        int ox, oy;
        size_t bc;
        pool_place<SMALL>(i, q.oW, q.oH, q.dow, q.doh, &ox, &oy, &bc);
        const float* in = x + bc * (size_t)q.H * q.W;
        const int x0 = ox * q.sx - q.px, y0 = oy * q.sy - q.py;
        const int sx_min = max(-x0, 0), sy_min = max(-y0, 0);
        const int sx_max = min(max(q.W - x0, 0), q.pw), sy_max = min(max(q.H - y0, 0), q.ph);
        float best = 0.0f;
        int where = -1;
        for (int sy = sy_min; sy < sy_max; ++sy)
            for (int sx = sx_min; sx < sx_max; ++sx) {
                const float v = in[(size_t)(y0 + sy) * q.W + x0 + sx];
                if (where < 0 || v > best) {
                    best = v;
                    where = (y0 + sy) * q.W + x0 + sx;
                }
            }
        y[i] = best;
        argmax[i] = where;
    }
}

// Every input collects the gradients of the outputs that chose it, in the reference's order (window rows, then columns,
// from the input's own residue modulo the stride upwards).
template <bool SMALL>
__global__ __launch_bounds__(TBLOCK) void pool_max_f32_backward_kernel(PoolF32 q, const float* __restrict__ dy, const int* __restrict__ argmax, float beta,
                                                                       float* __restrict__ dx)
{
    const size_t total = (size_t)q.B * q.C * q.H * q.W;
    for (size_t i = (size_t)blockIdx.x * TBLOCK + threadIdx.x; i < total; i += (size_t)gridDim.x * TBLOCK) {
        int ix, iy;
        size_t bc;
        pool_place<SMALL>(i, q.W, q.H, q.dw, q.dh, &ix, &iy, &bc);
        const int ix_pad = ix + q.px, iy_pad = iy + q.py;
        // the last output row and column whose window begins at or before this input, and the input's place in it
        const int oy0 = div_f32(iy_pad, q.dsy), ox0 = div_f32(ix_pad, q.dsx);
        const int sy0 = iy_pad - oy0 * q.sy, sx0 = ix_pad - ox0 * q.sx;
        float acc = 0.0f;
        for (int oy = oy0, sy = sy0; sy < q.ph && oy >= 0; sy += q.sy, --oy) {
            if (oy >= q.oH)
                continue;
            for (int ox = ox0, sx = sx0; sx < q.pw && ox >= 0; sx += q.sx, --ox) {
                if (ox >= q.oW)
                    continue;
                const size_t o = (bc * q.oH + oy) * q.oW + ox;
                if (argmax[o] == iy * q.W + ix)
                    acc += dy[o];
            }
        }
        dx[i] = acc + (beta != 0.0f ? beta * dx[i] : 0.0f);
    }
}

// The same for rows of whole quads: a lane takes four inputs of a row and goes through the windows that hold one of them, so that a
// window's two loads and the places are worked out once for the four.  (Of the same windows an input adds the same values in the same
// order.)  us, an input / a quad a lane: 64 x 64 x 32 x 32, 2x2 11.6 / 6.6 (42 MB); 32 x 64 x 112 x 112, 3x3 at 2 123 / 45; 32 x 64 x 56 x 56, 3x3
// at 1 72 / 57; 16 x 32 x 64 x 64, 7x7 at 7 7.7 / 4.3; 2 x 8 x 8 x 8 4.0 / 3.8.
__global__ __launch_bounds__(TBLOCK) void pool_max_f32_backward_quads_kernel(PoolF32 q, DivF32 dquads, const float* __restrict__ dy, const int* __restrict__ argmax,
                                                                             float beta, float* __restrict__ dx)
{
    const int quads = q.W / 4, total = q.B * q.C * q.H * quads;
    for (int i = (int)(blockIdx.x * TBLOCK + threadIdx.x); i < total; i += (int)gridDim.x * TBLOCK) {
        const int row = div_f32(i, dquads), ix = (i - row * quads) * 4, bc = div_f32(row, q.dh), iy = row - bc * q.H;
        // windows that begin at or before the last of the four, and end behind the first
        const int iy_pad = iy + q.py, oy0 = div_f32(iy_pad, q.dsy), ox0 = min(div_f32(ix + 3 + q.px, q.dsx), q.oW - 1);
        const int place = iy * q.W + ix;
        float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int oy = oy0, sy = iy_pad - oy0 * q.sy; sy < q.ph && oy >= 0; sy += q.sy, --oy) {
            if (oy >= q.oH) continue;
            const int base = (bc * q.oH + oy) * q.oW;
            for (int ox = ox0; ox >= 0 && ox * q.sx + q.pw > ix + q.px; --ox) {
                const int at = argmax[base + ox] - place;
                const float d = dy[base + ox];
#pragma unroll
                for (int u = 0; u < 4; ++u) acc[u] = at == u ? acc[u] + d : acc[u];
            }
        }
        float4* const out = (float4*)dx + i;
        if (beta != 0.0f) {
            const float4 o = *out;
            acc[0] += beta * o.x; acc[1] += beta * o.y; acc[2] += beta * o.z; acc[3] += beta * o.w;
        }
        *out = make_float4(acc[0], acc[1], acc[2], acc[3]);
    }
}

static int grid_for(size_t total)
{
    const size_t blocks = (total + TBLOCK - 1) / TBLOCK;
    return (int)std::min<size_t>(std::max<size_t>(blocks, 1), 256 * 32);
}

static int make_conv(const n2d2hip_conv_desc* d, int B, int H, int W, bool backward, ConvF32* q, const char* who)
{
    N2D2HIP_REQUIRE(d != nullptr, N2D2HIP_ERR_INVALID, "%s: null descriptor", who);
    N2D2HIP_REQUIRE(B > 0 && H > 0 && W > 0 && d->C > 0 && d->O > 0 && d->kW > 0 && d->kH > 0 && d->strideX > 0 && d->strideY > 0
                        && d->dilX > 0 && d->dilY > 0 && d->padL >= 0 && d->padT >= 0 && d->padR >= 0 && d->padB >= 0,
                    N2D2HIP_ERR_INVALID, "%s: bad shape", who);
    N2D2HIP_REQUIRE(d->groups == 1 || (d->groups == d->C && d->C == d->O), N2D2HIP_ERR_UNSUPPORTED,
                    "%s: groups=%d (C=%d, O=%d): only ungrouped and depthwise convolutions", who, d->groups, d->C, d->O);
    N2D2HIP_REQUIRE(!backward || (d->dilX == 1 && d->dilY == 1), N2D2HIP_ERR_UNSUPPORTED,
                    "%s: the reference's backward kernels do not read the dilation", who);
    int oH = 0, oW = 0;
    const int st = n2d2hip_conv_out_dims(d, H, W, &oH, &oW);
    if (st != N2D2HIP_OK) return st;
    N2D2HIP_REQUIRE(oH > 0 && oW > 0, N2D2HIP_ERR_INVALID, "%s: empty output", who);
    N2D2HIP_REQUIRE((size_t)B * std::max(d->C, d->O) * std::max((size_t)H * W, (size_t)oH * oW) < ((size_t)1 << 40), N2D2HIP_ERR_INVALID,
                    "%s: tensor too large", who);
    *q = ConvF32{B, d->C, H, W, d->O, oH, oW, d->kW, d->kH, d->C / d->groups, d->strideX, d->strideY,
                 d->padL, d->padT, d->padR, d->padB, d->dilX, d->dilY, d->groups > 1 ? 1 : 0, d->kernel_choice};
    return N2D2HIP_OK;
}

static int ceil_div_i(long a, long b) { return (int)((a + b - 1) / b); }

static bool spans_input(const ConvF32& q)
{
    return q.kH == q.H && q.kW == q.W && q.oH == 1 && q.oW == 1 && q.pl == 0 && q.pt == 0 && q.pr == 0 && q.pb == 0;
}

enum { PASS_FWD = 0, PASS_BWD_DATA = 1, PASS_BWD_FILTER = 2 };
enum { F32_PATH_DIRECT, F32_PATH_GEMM, F32_PATH_SMALL, F32_PATH_SMALL_DATA };

// More than the pixel kernels have lanes and the filter kernel has mask bits for
static bool many_taps(const ConvF32& q) { return (long)q.kH * q.kW > 64; }

// Largest second dimension of a grid.  Layers of more outputs or images than it covers take kernels with those in the first.
constexpr long GRID_Y = 65535;

// The kernels of a pass.  The matrix cores serve ungrouped convolutions without dilation; the direct kernels keep the rest
// (depthwise, dilated) and the forward sums below 2e7 flops or of kernels over 64 taps, which stay in the reference's order
// of terms (quantizers turn the last bit of a sum into a level now and then).  Backward-filter below 2e7 flops, and of a
// spanning kernel over 64 taps, and small data gradients add in double (F32_PATH_SMALL, _SMALL_DATA).  The descriptor's kernel_choice (N2D2HIP_KERNEL_F32_DIRECT /
// _GEMM) overrides the size rules.
static int f32_path(const ConvF32& q, int pass)
{
    if (q.depthwise || q.dx != 1 || q.dy != 1 || (q.choice & N2D2HIP_KERNEL_F32_DIRECT))
        return F32_PATH_DIRECT;
    // 32-bit byte offsets from a base moved back by the padding
    const size_t most = (size_t)1 << 29, rows = (size_t)q.pt + q.kH, cols = (size_t)q.W + q.oW + q.pl + q.kW;
    if (rows >= most || cols >= most || rows * cols >= most)
        return F32_PATH_DIRECT;
    const size_t lim = most - rows * cols;
    if ((size_t)q.B * q.C * q.H * q.W >= lim || (size_t)q.B * q.O * q.oH * q.oW >= lim || (size_t)q.O * q.C * q.kH * q.kW >= lim
        || (many_taps(q) && !spans_input(q)))
        return F32_PATH_DIRECT;
    if (pass == PASS_BWD_FILTER && many_taps(q)) return q.O <= 16 * GRID_Y ? F32_PATH_SMALL : F32_PATH_DIRECT;
    if (pass == PASS_BWD_FILTER && q.O > 64 * GRID_Y && !spans_input(q)) return F32_PATH_DIRECT;
    const double flops = 2.0 * q.B * q.O * q.oH * q.oW * q.C * q.kH * q.kW;
    const bool forced = q.choice & N2D2HIP_KERNEL_F32_GEMM, small = flops < 2.0e7;
    // As a convolution the K of a spanning layer's backward-data runs over all taps of an output, one of which is not zero: few
    // terms to a range.  As a product it has as many terms as outputs, so it adds in double up to 5e8 flops (64 images,
    // 64 x 4 x 4 <- 256: 2.5e-8 from 64 bits and 10 us; convolution 7.7e-8, 41 us; product in float 2.9e-7, 14 us) and beyond
    // has float sums as short as the convolution's (128 images, 512 x 2 x 2 <- 1000: 1.5e-7 and 22 us; in double 36; convolution
    // 1.5e-7, 64; 64 images, 512 x 7 x 7 <- 4096: 177 us, in double 1019, convolution 9566).
    if (pass == PASS_BWD_DATA && (forced || !small) && flops < 5.0e8 && !many_taps(q) && q.kH * q.kW > 1 && q.B <= 16 * GRID_Y && spans_input(q))
        return F32_PATH_SMALL;
    if (forced) return F32_PATH_GEMM;
    // Small data gradients add in double.  Spanning layers below 2e7 flops (us, product in float / this): 16 x 5 x 5 <- 120, batch 32 8.4 / 4.2;
    // 120 <- 84, batch 32 8.5 / 4.2; 512 x 1 x 1 <- 64, batch 2 7.7 / 3.9; 64 <- 10, batch 96 5.5 / 4.0.  Others by the rounds of loads
    // of all blocks and of one (data_small_tile has the times).  (Of 90 drawn strided layers with products from
    // 0.9e5, 76 are faster than the sums in float, down to 0.6 of their time; most of K from 1340 and of over 2000 tiles take 1.0 to 1.4 times as long,
    // 4 us at most.)
    if (pass == PASS_BWD_DATA && !many_taps(q)) {
        if (spans_input(q)) {
            if (small && q.B <= 16 * GRID_Y) return F32_PATH_SMALL;
        } else {
            const long K = (long)q.O * q.kH * q.kW;
            if (K <= 2304 && (double)ceil_div_i((long)q.B * q.H * q.W, 16) * ceil_div_i(q.C, 16) * K <= 2.3e5) return F32_PATH_SMALL_DATA;
        }
    }
    if (pass == PASS_FWD) return small || many_taps(q) ? F32_PATH_DIRECT : F32_PATH_GEMM;
    if (small && pass == PASS_BWD_FILTER) return q.O <= 16 * GRID_Y ? F32_PATH_SMALL : F32_PATH_DIRECT;
    return F32_PATH_GEMM;
}

static DivF32 div_of(int d)
{
    DivF32 r;
    magic_div((unsigned)d, &r.mul, &r.sh);
    return r;
}

// The strip kernels of depthwise layers (depthwise_f32.hpp): square kernels of 3 or 5 at one stride of 1 or 2, 32-bit offsets
// (with room for a window past the end).  All forms that qualify are faster so: 128
// channels, 3x3, 56 x 56, batch 32: backward-data 167.5 -> 19.4 us, backward-filter 407.8 -> 49.7.
static bool depthwise_strips(const ConvF32& q)
{
    const size_t lim = ((size_t)1 << 31) - 4096;
    return q.depthwise && q.dx == 1 && q.dy == 1 && q.kH == q.kW && (q.kH == 3 || q.kH == 5) && q.sx == q.sy && q.sx <= 2 && q.C <= 65535
           && (size_t)q.B * q.C * (q.H + q.kH) * (q.W + q.kW + q.pl + 8) < lim && (size_t)q.B * q.C * (q.oH + q.kH) * (q.oW + q.pl + 8) < lim
           && (size_t)q.pl + q.pt + q.pr + q.pb < 4096;
}
static unsigned reduce_grid(size_t n) { return (unsigned)std::min<size_t>((n + 63) / 64, 16384); }

// Short sums: a block per channel and tap row (of so many threads; 0: none), whose blocks find each other's strips in the caches.
// Ahead of ranges of all taps, whose K * K sums take a block as long to add up as some hundred strips, and of the launch
// that adds the ranges, until the strips are many or, with many channels, the tensors no longer lie in the L2.  us, a block of 256 /
// 512 / 1024 per tap row / ranges:
//   3x3, channels, strips: 8, 224 4.0 / 4.0 / 4.2 / 5.6; 8, 3136 9.3 / 6.7 / 6.2 / 11.0; 48, 6400 14.3 / 9.7 / 8.7 / 11.2; 128, 480 4.8 / 4.9 / 6.1 / 6.9;
//     128, 12544 37.3 / 29.8 / 34.2 / 28.2; 256, 3200 12.2 / 11.1 / 11.6 / 13.6; 256, 12544 41.8 / 39.2 / 41.6 / 29.7; 512, 784 8.8 / 9.9 / 13.9 / 10.4;
//     512, 3136 31.7 / 40.5 / 40.5 / 26.5; 1024, 448 9.1 / 13.1 / 22.6 / 9.7; 1024, 1568 21.1 / 25.1 / 28.7 / 19.9
//   5x5: 8, 200 4.2 / 4.3 / 5.3 / 9.9; 8, 12800 29.1 / 19.8 / 17.3 / 20.1; 8, 25088 53.2 / 35.0 / 30.2 / 21.2; 128, 784 6.9 / 7.7 / 11.1 / 14.7;
//     128, 12800 50.5 / 45.6 / 42.5 / 41.9; 512, 1568 20.5 / 21.4 / 31.6 / 25.3; 512, 6272 77.0 / 75.7 / 75.9 / 62.0; 1024, 1600 38.0 / 41.6 / 62.3 / 43.4;
//     stride 2, 1024, 512 40.7 / 44.1 / 57.8 / 24.8
static int depthwise_row_threads(const ConvF32& q)
{
    const long items = (long)q.B * q.oH * ceil_div_i(q.oW, 4), blocks = (long)q.C * q.kH;
    if (items > (q.kH == 3 ? 8192 : 12800) || items * q.C > 1600000 / q.sx / (blocks > 2560 ? 2 : 1)) return 0;
    if (items > 2048 && blocks <= 1024) return 1024;
    return items > 512 && blocks <= 512 ? 512 : 256;
}
// Ranges the strips of a channel are split into for its filter gradient: enough for eight blocks of 256 on every compute unit,
// but no fewer than six strips a thread.  us, at 2 / 3 / 6 / 12 strips: 128 channels, 56 x 56, batch 32 30.8 / 31.4 / 31.1 / 32.6;
// 512, 14 x 14, batch 64 20.0 / 20.2 / 20.0 / 20.3; 8, 56 x 56, batch 32 10.3 / 10.0 / 11.9 / 15.4; 96, 5x5, 56 x 56, batch 16
// 41.8 / 37.0 / 33.9 / 33.1 (a block per channel and tap row: 48.6, 27.6, 25.4, 36.2).
// The workspace query answers for them; with few channels (blocks for less than half of the chip) also where a block per tap row
// takes the sum without, as a batch that is a little larger will need it.
static int depthwise_filter_ranges(const ConvF32& q)
{
    const int items = q.B * q.oH * ceil_div_i(q.oW, 4);
    return depthwise_row_threads(q) && 2 * q.C * q.kH >= num_cus() ? 1 : std::max(1, std::min(ceil_div_i(items, 6 * 256), ceil_div_i(8 * num_cus(), q.C)));
}
static size_t depthwise_filter_bytes(const ConvF32& q, int ranges) { return ranges > 1 ? (size_t)ranges * q.C * q.kH * q.kW * sizeof(double) : 0; }

static int run_depthwise(const ConvF32& q, int pass, const float* a, const float* b, const float* bias, float beta, float* out, void* workspace,
                         size_t workspace_bytes, hipStream_t st)
{
    const int rows = pass == PASS_BWD_DATA ? q.H : q.oH, cols = pass == PASS_BWD_DATA ? q.W : q.oW, strips = ceil_div_i(cols, 4);
    const DepthwiseF32 k = {q.C, q.H, q.W, q.oH, q.oW, q.pl, q.pt, q.B * rows * strips, strips, q.B * q.C * q.H * q.W, q.B * q.C * q.oH * q.oW,
                            div_of(strips), div_of(rows),
                            q.oW % 4 == 0 && q.pl <= q.kW / 2 && (q.oW - 1) * q.sx - q.pl + q.kW - 1 < q.W + q.kW / 2};
    const dim3 grid(ceil_div_i(k.items, 256), q.C);
    const auto run = [&](auto K_, auto S_) {
        constexpr int K = decltype(K_)::value, S = decltype(S_)::value;
        if (pass == PASS_FWD) hipLaunchKernelGGL((depthwise_f32_forward_kernel<K, S>), grid, dim3(256), 0, st, k, a, b, bias, beta, out);
        else if (pass == PASS_BWD_FILTER) {
            // (without the workspace that the query names, or with one that holds no doubles: one range)
            const int row_threads = depthwise_row_threads(q);
            int ranges = row_threads ? 1 : depthwise_filter_ranges(q);
            if (workspace_bytes < depthwise_filter_bytes(q, ranges) || (size_t)workspace % sizeof(double)) ranges = 1;
            const int per_range = ceil_div_i(k.items, ranges);
            ranges = ceil_div_i(k.items, per_range);
            constexpr int WIDE = K == 3 ? 1024 : 512;
            const auto by_rows = [&](auto T) {
                constexpr int THREADS = decltype(T)::value;
                N2D2HIP_LAUNCH_T(depthwise_f32_filter_kernel, (K, S, THREADS, 1), dim3(q.C, 1, K), dim3(THREADS), 0, st, k, per_range, a, b, beta, out, (double*)nullptr);
            };
            if (row_threads == 1024) by_rows(std::integral_constant<int, 1024>{});
            else if (row_threads == 512) by_rows(std::integral_constant<int, 512>{});
            else if (row_threads == 256) by_rows(std::integral_constant<int, 256>{});
            else if (ranges == 1 && k.items > 6 * 256)
                N2D2HIP_LAUNCH_T(depthwise_f32_filter_kernel, (K, S, WIDE, K), dim3(q.C), dim3(WIDE), 0, st, k, per_range, a, b, beta, out, (double*)nullptr);
            else
                N2D2HIP_LAUNCH_T(depthwise_f32_filter_kernel, (K, S, 256, K), dim3(q.C, ranges), dim3(256), 0, st, k, per_range, a, b, beta, out, (double*)workspace);
            const size_t n = (size_t)q.C * K * K;
            if (ranges > 1)
                hipLaunchKernelGGL(conv_f32_reduce_partials_kernel<double>, dim3(reduce_grid(n)), dim3(256), 0, st, (const double*)workspace, ranges, n, beta, out,
                                   (const float*)nullptr, 1, 1);
        }
        else if (S == 2 && (q.pl & 1)) hipLaunchKernelGGL((depthwise_f32_data_kernel<K, S, S == 2>), grid, dim3(256), 0, st, k, b, a, beta, out);
        else hipLaunchKernelGGL((depthwise_f32_data_kernel<K, S, 0>), grid, dim3(256), 0, st, k, b, a, beta, out);
    };
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;
    using I5 = std::integral_constant<int, 5>;
    if (q.kH == 3) q.sx == 1 ? run(I3{}, I1{}) : run(I3{}, I2{});
    else q.sx == 1 ? run(I5{}, I1{}) : run(I5{}, I2{});
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

// The direct kernel of forward and backward-data: the walk with 32-bit offsets and one mask bit per tap row and column, or
// (dilated, larger) one load after the other.
// (sat: done by the kernels of a spanning layer, which say so)
static int run_direct(const ConvF32& q, int pass, const float* x, const float* w, const float* bias, float beta, float* out, hipStream_t st, const SatStore& sat = {},
                      bool* sat_done = nullptr)
{
    if (depthwise_strips(q)) return run_depthwise(q, pass, x, w, bias, beta, out, nullptr, 0, st);
    const bool bwd = pass == PASS_BWD_DATA;
    const size_t lim = (size_t)1 << 31, total = (size_t)q.B * (bwd ? (size_t)q.C * q.H * q.W : (size_t)q.O * q.oH * q.oW);
    const size_t source = (size_t)q.B * (bwd ? (size_t)q.O * q.oH * q.oW : (size_t)q.C * q.H * q.W);
    const int T = q.kH * q.kW;
    const long K = (long)q.C * T;
    // (a kernel of 3x3 has an order of its own; 16-byte loads)
    if (!bwd && !q.depthwise && q.dx == 1 && q.dy == 1 && spans_input(q) && (q.kH != 3 || q.kW != 3) && K % 4 == 0 && K < (1 << 22) && q.O <= 8 * GRID_Y
        && (((size_t)x | (size_t)w) & 15) == 0) {
        const dim3 grid(ceil_div_i(q.B, 8), ceil_div_i(q.O, 8));
        // (the first up to two of its waves a SIMD; a unit holds one block of the second, and three of the third; measured at the kernels)
        const dim3 small(ceil_div_i(q.B, 2), ceil_div_i(q.O, 2));
        if ((size_t)small.x * small.y <= 8 * (size_t)num_cus())
            N2D2HIP_LAUNCH(conv_f32_chain_kernel<4>, small, dim3(64), 0, st, q.B, q.O, (int)K, x, w, bias, beta, sat, out);
        else if ((size_t)grid.x * grid.y <= (size_t)num_cus())
            N2D2HIP_LAUNCH(conv_f32_chain_kernel<64>, grid, dim3(192), 0, st, q.B, q.O, (int)K, x, w, bias, beta, sat, out);
        else
            N2D2HIP_LAUNCH(conv_f32_chain_wave_kernel, grid, dim3(64), 0, st, q.B, q.O, (int)K, x, w, bias, beta, sat, out);
        if (sat_done) *sat_done = true;
        N2D2HIP_HIP_CHECK(hipGetLastError());
        return N2D2HIP_OK;
    }
    if (q.dx != 1 || q.dy != 1 || total >= lim - 64 || source >= lim || (size_t)q.O * q.Cw * T >= lim || q.kH + q.kW > 31) {
        if (bwd) hipLaunchKernelGGL(conv_f32_backward_data_kernel, dim3(grid_for(total)), dim3(TBLOCK), 0, st, q, w, x, beta, out);
        else hipLaunchKernelGGL(conv_f32_forward_kernel, dim3(grid_for(total)), dim3(TBLOCK), 0, st, q, x, w, bias, beta, out);
        N2D2HIP_HIP_CHECK(hipGetLastError());
        return N2D2HIP_OK;
    }
    WalkF32 k = {};
    if (bwd) {
        k = {q.depthwise ? 1 : q.O, ceil_div_i(q.kH, q.sy), ceil_div_i(q.kW, q.sx), q.oH * q.oW, -q.oW, -1, q.Cw * T, q.sy * q.kW, q.sx,
             div_of(q.H * q.W), div_of(q.W), div_of(q.C)};
        hipLaunchKernelGGL((conv_f32_walk_kernel<true, 0>), dim3((unsigned)((total + 63) / 64)), dim3(64), 0, st, q, k, x, w, bias, beta, out, (int)total);
    } else {
        k = {q.depthwise ? 1 : q.C, q.kH, q.kW, q.H * q.W, q.W, 1, T, q.kW, 1, div_of(q.oH * q.oW), div_of(q.oW), div_of(q.O)};
        const dim3 grid((unsigned)((total + 63) / 64));
        // (windows inside the input, byte offsets of 32 bits; kernels of 4 to 7, whose windows the registers hold twice)
        const bool inside = q.pt == 0 && q.pl == 0 && (q.oH - 1) * q.sy + q.kH <= q.H && (q.oW - 1) * q.sx + q.kW <= q.W && source < lim / 2
            && (size_t)q.O * q.Cw * T < lim / 2;
        if (inside && q.kH == q.kW && q.kH >= 4 && q.kH <= 7) {
            const auto kernel = q.kH == 4 ? conv_f32_window_kernel<4> : q.kH == 5 ? conv_f32_window_kernel<5> : q.kH == 6 ? conv_f32_window_kernel<6>
                                                                                                                      : conv_f32_window_kernel<7>;
            hipLaunchKernelGGL(kernel, grid, dim3(64), 0, st, q, k, x, w, bias, beta, out, (int)total);
        } else if (q.kH != 3 || q.kW != 3) hipLaunchKernelGGL((conv_f32_walk_kernel<false, 0>), grid, dim3(64), 0, st, q, k, x, w, bias, beta, out, (int)total);
        else if (k.n == 1) hipLaunchKernelGGL((conv_f32_walk_kernel<false, 1>), grid, dim3(64), 0, st, q, k, x, w, bias, beta, out, (int)total);
        else hipLaunchKernelGGL((conv_f32_walk_kernel<false, 4>), grid, dim3(64), 0, st, q, k, x, w, bias, beta, out, (int)total);
    }
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

// K ranges of P pixels x Q channels over K terms, from the sizes alone, as if tiles were 128 x 128: 768 blocks, none below 256
// terms.
static int pass_ranges(long P, int Q, long K)
{
    const long tiles = ((P + 127) / 128) * (Q <= 64 ? 1 : ceil_div_i(Q, 128));
    return (int)std::min<long>(tiles >= 384 ? 1 : std::max(1L, 768 / tiles), std::max(1L, K / (16 * GK)));
}

// A kernel that spans its input (an FcCell) makes of each pass a plain matrix product, which is a 1x1 convolution with the
// roles of the tensors exchanged so that the long contiguous dimension is the one the kernels read contiguously:
//   forward          y[b][o] = sum_k x[b][k] w[o][k]     the filter pass of pixels k between "channels" w[o] and "outputs" x[b]
//   backward data    dx[b][k] = sum_o dy[b][o] w[o][k]   the forward pass over one "image" w of O channels and K pixels
//   backward filter  dw[o][k] = sum_b dy[b][o] x[b][k]   the data pass over one "image" x of B channels and K pixels
// Forward and backward data have no longer float sums than the convolution itself would.
static ConvF32 product_of(const ConvF32& q, int pass, int* as_pass)
{
    const int K = q.C * q.H * q.W, T = q.H * q.W;
    const int ranges = pass == PASS_FWD ? pass_ranges(q.B, q.O, K) : pass == PASS_BWD_DATA && T > 1 && T <= 64 ? pass_ranges((long)q.B * T, q.C, (long)q.O * T) : 0;
    *as_pass = pass == PASS_FWD ? PASS_BWD_FILTER : pass == PASS_BWD_DATA ? PASS_FWD : PASS_BWD_DATA;
    return ConvF32{1, q.O, 1, K, q.B, 1, K, 1, 1, q.O, 1, 1, 0, 0, 0, 0, 1, 1, 0, q.choice, ranges};
}

// ---- forward and backward-data: tile shape and K ranges of a launch
struct PatchShape {
    int wq, wp, mq, np;        // a tile: 16 wq mq rows of q x 16 wp np pixels
    int nu;                    // units of 128 source positions that hold what a tile's taps read; 0: more than the kernel takes
    int pixels() const { return 16 * np * wp; }
    int rows() const { return 16 * wq * mq; }
};
struct PixelPlan {
    bool small_q;              // tiles of 32 q x 128 pixels instead of 64 x 64
    int splits;                // K ranges that leave partial results
    int kind;                  // PIXELS_*
    PatchShape patch;          // (PIXELS_PATCH, PIXELS_PARTS)
    bool chunks;               // (PIXELS_PARTS) a step is channels at one tap
    bool many;                 // a class has more tap rows and columns than a mask of 31 bits
    PixelGemm g;
};

// Classes of pixels of one launch (backward-data of a strided convolution: s * s residue classes, those with the most taps
// first).  Returns how many launches of up to PIXEL_CLASSES classes the pass takes.
static std::vector<PixelClass> pixel_classes(const ConvF32& q, int pass)
{
    std::vector<PixelClass> v;
    if (pass == PASS_FWD) {
        PixelClass c = {};
        c.gW = q.oW; c.gHW = q.oH * q.oW; c.P = q.B * c.gHW;
        c.nx = q.kW; c.nT = q.kH * q.kW;
        c.y0 = -q.pt; c.x0 = -q.pl;
        c.stepy = q.W; c.stepx = 1;
        c.bias = q.pt * q.W + q.pl; c.soff0 = 0;
        v.push_back(c);
    } else {
        for (int ry = 0; ry < std::min(q.sy, q.H); ++ry)
            for (int rx = 0; rx < std::min(q.sx, q.W); ++rx) {
                PixelClass c = {};
                c.gW = (q.W - rx + q.sx - 1) / q.sx;
                c.gHW = ((q.H - ry + q.sy - 1) / q.sy) * c.gW;
                c.P = q.B * c.gHW;
                c.ty0 = (ry + q.pt) % q.sy; c.tx0 = (rx + q.pl) % q.sx;
                const int ny = c.ty0 < q.kH ? (q.kH - 1 - c.ty0) / q.sy + 1 : 0;
                c.nx = c.tx0 < q.kW ? (q.kW - 1 - c.tx0) / q.sx + 1 : 0;
                c.nT = ny * c.nx;
                c.y0 = (ry + q.pt) / q.sy; c.x0 = (rx + q.pl) / q.sx;
                c.stepy = -q.oW; c.stepx = -1;
                c.ry = ry; c.rx = rx;
                const int first = c.y0 * q.oW + c.x0, last = first - std::max(ny - 1, 0) * q.oW - std::max(c.nx - 1, 0);
                c.bias = std::max(0, -last);
                c.soff0 = first + c.bias;
                v.push_back(c);
            }
        std::stable_sort(v.begin(), v.end(), [](const PixelClass& a, const PixelClass& b) { return a.nT > b.nT; });
    }
    for (PixelClass& c : v) {
        c.ghw = div_of(c.gHW); c.gw = div_of(c.gW); c.nt = div_of(c.nT); c.nxd = div_of(c.nx);
    }
    return v;
}

enum { PIXELS_TAPS, PIXELS_CHUNK, PIXELS_3X3, PIXELS_PATCH, PIXELS_PARTS };
// Units of 128 source positions that hold what the taps of any `pixels` consecutive pixels of the class read: every step to the
// next pixel is at least 0 and at most one of a row's, a row's end's and an image's end's.  0: a step back.
static int patch_units(const ConvF32& q, int pass, const PixelClass& c, int pixels)
{
    const long sy = pass == PASS_FWD ? q.sy : 1, sx = pass == PASS_FWD ? q.sx : 1;
    const long Hs = pass == PASS_FWD ? q.H : q.oH, Ws = pass == PASS_FWD ? q.W : q.oW, gH = c.gHW / c.gW, ny = c.nT / c.nx;
    const long row = sy * Ws - c.gW * sx, image = Hs * Ws - gH * sy * Ws;        // beyond a step of sx; beyond that and `row`
    if (sx + row < 0 || sx + row + image < 0) return 0;
    const long n = pixels - 1;
    const long span = n * sx + (n / c.gW + 1) * std::max(0L, row) + (n / c.gHW + 1) * std::max(0L, image) + (ny - 1) * Ws + c.nx;
    return span <= 128 * 3 ? ceil_div_i(span, 128) : 0;
}
// Chunks of a class after which a float sum of the patch kernel is added to the one in double: where it has been rounded as often as
// the longest float sum of the other kernels.  Theirs round once a term, this one 5 times in 32.
static int patch_fold(const ConvF32& q, int pass, const PixelClass& c)
{
    const bool fwd = pass == PASS_FWD;
    const long K = (long)(fwd ? q.C : q.O) * q.kH * q.kW;
    const long ranges = pass_ranges((long)q.B * (fwd ? q.oH * q.oW : q.H * q.W), fwd ? q.O : q.C, K);
    const long T = fwd ? (long)c.nT : (long)ceil_div_i(q.kH, q.sy) * ceil_div_i(q.kW, q.sx);     // taps of the longest sum
    return (int)std::max(4 * (K / ranges) / (PK * T), 1L);
}
// Backward-data of a 3x3 kernel at stride 2 as one class whose every place is four pixels
static bool patch_fours(const ConvF32& q, int pass) { return pass == PASS_BWD_DATA && q.kH == 3 && q.kW == 3 && q.sx == 2 && q.sy == 2; }
static PixelClass fours_class(const ConvF32& q)
{
    PixelClass c = {};
    c.gW = (q.W + 1) / 2; c.gHW = (q.H + 1) / 2 * c.gW; c.P = q.B * c.gHW;
    c.nx = 3; c.nT = 9;
    c.ry = q.pt & 1; c.rx = q.pl & 1;            // the pixel of taps 0 and 2
    c.y0 = (c.ry + q.pt) / 2; c.x0 = (c.rx + q.pl) / 2;
    c.ghw = div_of(c.gHW); c.gw = div_of(c.gW); c.nt = div_of(c.nT); c.nxd = div_of(c.nx);
    return c;
}
// Tiles of 64 rows x 128 pixels where they fill three quarters of the chip's two blocks to a CU and need no sums in double (whose
// registers they lack); else of 64 x 64.  us, 64 x 128 / 64 x 64, forward: 64 -> 64, 56 x 56, batch 64 (1568 of the larger tiles)
// 90 / 105; 64 -> 64, 32 x 32, batch 64 (512) 34 / 38; 256 -> 256, 14 x 14, batch 32 (196) 65 / 60; 48 -> 96, 5x5, 30 x 30, batch
// 16 (226) 54 / 42.  No shape for runs of more than 384 positions, which would leave one block to a CU: 64 -> 128, stride 2, 56 x
// 56, batch 16 (456) 40 against 31 of the chunk kernel.  (All counts of tiles are for 256 CUs, wherever they run: the order of a sum's
// additions follows from the sizes alone.)
static PatchShape patch_shape(const ConvF32& q, int pass, const PixelClass& c)
{
    const int Q = pass == PASS_FWD ? q.O : q.C, chunks = ceil_div_i(pass == PASS_FWD ? q.C : q.O, PK);
    auto fit = [&](PatchShape s) {
        s.nu = c.nx + c.nT / c.nx > 31 ? 0 : patch_units(q, pass, c, s.pixels());
        return s;
    };
    if (patch_fours(q, pass)) {
        // No sums in double (the float ones take the registers).  Where the tiles give every CU a block, or are so few that the chunk
        // kernel's longest class leaves most of the chip idle; between, partial results of two ranges cost more than it saves.
        // us, chunk kernel / this: 64 <- 64, 56 x 56, batch 128 (1568 tiles) 98 / 74; 256 <- 512, 14 x 14, batch 128 (392) 145 / 106; 64 <- 128,
        // 32 x 32, batch 64 (256) 34.4 / 29.1; 128 <- 256, 27 x 27, batch 33 (202) 52.3 / 54.7; 64 <- 128, 56 x 56, batch 16 (196) 32.5 / 47.7; 320 <- 384,
        // 13 x 13, batch 33 (130 of 12 chunks) 62 / 54; 128 <- 256, 16 x 16, batch 64 (128 of 8) 42.5 / 43.1; 256 <- 512, 28 x 28, batch 8 (100 of
        // 16) 75 / 54; half of a tile padding: 40 <- 48, 48 x 48, batch 64 33.3 / 34.1.
        PatchShape s = fit(PatchShape{2, 2, 2, 2, 0});
        const long tiles = (long)ceil_div_i(c.P, 64) * ceil_div_i(Q, 64);
        if (s.nu > 2 || Q <= 32 || patch_fold(q, pass, c) < chunks || (tiles < 256 && !(tiles <= 160 && chunks >= 12))
            || 2L * Q * q.O < (long)ceil_div_i(Q, 64) * 64 * chunks * PK)
            s.nu = 0;
        return s;
    }
    if (Q <= 32) return fit(PatchShape{1, 4, 2, 2, 0});
    if (patch_fold(q, pass, c) >= chunks && (long)ceil_div_i(c.P, 128) * ceil_div_i(Q, 64) >= 384) {
        const PatchShape s = fit(PatchShape{2, 2, 2, 4, 0});
        if (s.nu) return s;
    }
    return fit(PatchShape{2, 2, 2, 2, 0});
}
// conv_f32_taps_kernel: whether a step is 32 channels at one tap, and the steps of a class
static bool taps_chunks(const ConvF32& q, int pass) { const int ch = pass == PASS_FWD ? q.C : q.O; return round_up(ch, PK) * 5 <= ch * 6; }
static int taps_steps(const ConvF32& q, int pass, const PixelClass& c)
{
    const int ch = pass == PASS_FWD ? q.C : q.O;
    return taps_chunks(q, pass) ? ceil_div_i(ch, PK) * c.nT : ceil_div_i((long)ch * c.nT, PK);
}
// Steps after which its float sums go to those in double: as patch_fold
static int taps_fold(const ConvF32& q, int pass)
{
    const bool fwd = pass == PASS_FWD;
    const long K = (long)(fwd ? q.C : q.O) * q.kH * q.kW;
    return (int)std::max(4 * (K / pass_ranges((long)q.B * (fwd ? q.oH * q.oW : q.H * q.W), fwd ? q.O : q.C, K)) / PK, 1L);
}
// Tiles of 128 rows x 64 pixels, whose waves read each weight once and take each value of the source apart for twice as many products, where they fill
// 128 rows and give every CU a block or K is long enough to be split; of 64 x 64 else, and where several classes of different length share
// the chip.  us, 128 / 64 rows: forward 164 -> 377, 5x5 stride 2, 9 x 85, batch 16 (162 blocks of 128 rows, K 4100) 99 / 124; 64 -> 256, 1x1, 56 x 56,
// batch 64 (6272) 87 / 95; 1024 -> 256, 1x1, 14 x 14, batch 32 (196, K 1024) 45 / 40; 512 -> 2048, 7 x 7, batch 16 (208, K 512) 39 / 31; data 128 <- 256, 3x3
// stride 2, 27 x 27, batch 33, four classes 48.6 / 46.6.
static PatchShape taps_shape(const ConvF32& q, int pass, const std::vector<PixelClass>& cls)
{
    const int Q = pass == PASS_FWD ? q.O : q.C;
    if (Q <= 16) return PatchShape{1, 4, 1, 2, 0};
    if (Q <= 32) return PatchShape{1, 4, 2, 2, 0};
    const long blocks = (long)ceil_div_i(cls[0].P, 64) * ceil_div_i(Q, 128), K = (long)(pass == PASS_FWD ? q.C : q.O) * cls[0].nT;
    return cls.size() == 1 && round_up(Q, 128) * 8 <= round_up(Q, 64) * 9 && (blocks >= 256 || K >= 2048) ? PatchShape{4, 1, 2, 4, 0} : PatchShape{2, 2, 2, 2, 0};
}
static PixelPlan plan_pixels(const ConvF32& q, int pass, std::vector<PixelClass> cls, int kind)
{
    PixelPlan pl = {};
    PixelGemm& g = pl.g;
    const bool fwd = pass == PASS_FWD;
    g.Q = fwd ? q.O : q.C;
    g.Ch = fwd ? q.C : q.O;
    g.sy = fwd ? q.sy : 1; g.sx = fwd ? q.sx : 1;
    g.d = fwd ? 1 : -1;
    g.Hs = fwd ? q.H : q.oH; g.Ws = fwd ? q.W : q.oW; g.planeS = g.Hs * g.Ws;
    const int T = q.kH * q.kW;
    g.qs = fwd ? q.C * T : T; g.chs = fwd ? T : q.C * T; g.kW = q.kW; g.osy = fwd ? 1 : q.sy; g.osx = fwd ? 1 : q.sx;
    g.planeO = fwd ? q.oH * q.oW : q.H * q.W; g.Wo = fwd ? q.oW : q.W;
    g.bytesX = (unsigned)(4 * (size_t)q.B * g.Ch * g.planeS);
    g.bytesW = (unsigned)(4 * (size_t)q.O * q.C * T);
    // tile shape
    long P = 0, kmax = 0;
    const int nchunks = ceil_div_i(g.Ch, GK);
    const int kch = kind == PIXELS_PATCH ? round_up(g.Ch, PK) : kind == PIXELS_CHUNK && (!fwd || T > 1) ? nchunks * GK : g.Ch;
    for (const PixelClass& c : cls) { P += c.P; kmax = std::max(kmax, (long)kch * c.nT); }
    // (64 x 64 tiles, four to a CU, lost at most 4 % to the best of 32 x 128, 64 x 128 and 128 x 128 on every shape with Q
    // over 32 that was timed, and gained up to 70 % where the larger tiles are few)
    pl.small_q = g.Q <= 32;
    if (kind == PIXELS_PATCH) pl.patch = patch_shape(q, pass, cls[0]);
    if (kind == PIXELS_PARTS) pl.patch = taps_shape(q, pass, cls);
    const bool parts = kind == PIXELS_PATCH || kind == PIXELS_PARTS;
    const int PT = parts ? pl.patch.pixels() : pl.small_q ? 128 : 64, QT = parts ? pl.patch.rows() : pl.small_q ? 32 : 64;
    g.qtiles = ceil_div_i(g.Q, QT);
    pl.kind = kind;
    g.T = T;
    g.qpad = kind == PIXELS_PATCH ? round_up(g.Q, 128) : g.qtiles * QT;
    g.npos = q.B * g.planeS;
    g.bytesO = (unsigned)(4 * (size_t)q.B * g.Q * g.planeO);
    g.dplane = div_of(g.planeS);
    long tiles = 0;
    g.nclass = (int)cls.size();
    for (int i = 0; i < g.nclass; ++i) {
        cls[i].tile0 = (int)tiles;
        pl.many = pl.many || cls[i].nx + (cls[i].nT > 0 ? cls[i].nT / cls[i].nx : 0) > 31;
        tiles += ceil_div_i(cls[i].P, PT);
    }
    g.ptiles = (int)tiles;
    g.ptiles8 = ceil_div_i(tiles, 8);
    const long blocks = tiles * g.qtiles;
    g.nz = 1;
    if (kind == PIXELS_PATCH) {
        // ranges (of chunks) where the tiles alone would not give each of 256 CUs a block
        const int chunks = ceil_div_i(g.Ch, PK);
        const int each = ceil_div_i(chunks, blocks >= 256 ? 1 : std::min<long>(chunks, std::max(1L, 512 / std::max(blocks, 1L))));
        pl.splits = ceil_div_i(chunks, each);
        const int fold = patch_fold(q, pass, cls[0]);
        g.c[0] = cls[0];
        g.c[0].kchunk = each;
        g.c[0].fold = fold < each ? fold : 0;
        return pl;
    }
    if (kind == PIXELS_PARTS) {
        int most = 1, w0 = 0;
        for (const PixelClass& c : cls) most = std::max(most, taps_steps(q, pass, c));
        const int fold = taps_fold(q, pass);
        pl.chunks = taps_chunks(q, pass);
        // (ranges of four steps at least, where the tiles alone would not give each of 256 CUs a block)
        const int splits = blocks >= 256 ? 1 : (int)std::max(1L, std::min<long>(512 / std::max(blocks, 1L), most / 4));
        const int each = ceil_div_i(most, splits);
        pl.splits = ceil_div_i(most, each);
        for (int i = 0; i < g.nclass; ++i) {
            g.c[i] = cls[i];
            g.c[i].w0 = w0;
            const int steps = taps_steps(q, pass, cls[i]);
            w0 += steps;
            g.c[i].kchunk = std::max(ceil_div_i(steps, pl.splits), 1);
            g.c[i].fold = fold < each ? fold : 0;
        }
        return pl;
    }
    long splits, least = q.ranges;
    if (fwd) {
        // The ranges of a forward sum follow from its sizes alone: with another order of additions the quantizer behind it would
        // give another level now and then.  With a block for every CU it takes all of them (long kernels: with two; 64 -> 64,
        // 1 x 31, 256 tiles: 102 us with one, 82 with partial results).
        splits = pass_ranges(P, g.Q, kmax);
    } else {
        // where the tiles do not fill the chip twice; none below four steps.  And no float sum longer than over all taps at 128 x
        // 128 tiles: the longer, the more it loses (256 -> 256, 3x3, 14 x 14, batch 32: one sum 8.3e-7 from 64 bits and 89 us,
        // seven added in double as the steps go 3.1e-7 and 91, as ranges that each fill the ring anew 97).
        splits = blocks >= 512 ? 1 : std::max(1L, 768 / blocks);
        splits = std::min<long>(splits, std::max(1L, kmax / (4 * GK)));
        least = pass_ranges((long)q.B * q.H * q.W, q.C, (long)q.O * T);
    }
    const int step = kind == PIXELS_3X3 ? K33 : GK;
    pl.splits = 1;
    for (int i = 0; i < g.nclass; ++i) {         // (the ranges of a class of fewer taps are as many, and shorter)
        const long K = (long)kch * cls[i].nT;
        const bool ranges = fwd && kind == PIXELS_TAPS && least > splits;        // (the forward pixel kernel does not fold)
        cls[i].kchunk = std::max(ranges ? (int)(K / least) / GK * GK : round_up((int)((K + splits - 1) / splits), GK), GK);
        cls[i].fold = least > splits && !ranges ? std::max((int)(K / least) / step, 1) : 0;
        pl.splits = std::max(pl.splits, ceil_div_i(K, cls[i].kchunk));
        if (kind == PIXELS_CHUNK) cls[i].kchunk /= GK;
        g.c[i] = cls[i];
    }
    if (fwd && blocks >= (pl.many ? 512 : 256)) {
        g.nz = pl.splits;
        pl.splits = 1;
    }
    return pl;
}

// Blocks of the patch kernel: those of all items, or two to a CU that stay for several (a multiple of 8, one to each XCD)
static unsigned patch_blocks(unsigned items) { return std::min(items, (unsigned)std::max(2 * num_cus() / 8, 1) * 8); }
template <int WQ, int WP, int MQ, int NP, bool FOLDS>
static void launch_patch(const PixelPlan& pl, dim3 grid, const float* x, const float* w, const float* wt, const float* bias, float beta, float* out, size_t partial,
                         hipStream_t st)
{
    grid.x = patch_blocks(grid.x);
    const auto run = [&](auto nu_, auto nt_, auto fold_) {
        constexpr int PB = 2 * decltype(nu_)::value, NT = decltype(nt_)::value;
        constexpr bool FOLD = decltype(fold_)::value;
        N2D2HIP_LAUNCH_T(conv_f32_patch_kernel, (WQ, WP, MQ, NP, PB, NT, FOLD), grid, dim3(256), 0, st, pl.g, x, w, (const v4u*)wt, bias, beta, out, partial);
    };
    const auto taps = [&](auto nu_, auto fold_) {
        pl.g.c[0].nT == 9 && pl.g.c[0].nx == 3 ? run(nu_, std::integral_constant<int, 9>{}, fold_) : run(nu_, std::integral_constant<int, 0>{}, fold_);
    };
    const auto units = [&](auto fold_) {
        pl.patch.nu <= 2 ? taps(std::integral_constant<int, 2>{}, fold_) : taps(std::integral_constant<int, 3>{}, fold_);
    };
    if constexpr (FOLDS) {
        if (pl.g.c[0].fold) return units(std::true_type{});
    }
    units(std::false_type{});
}

template <bool BWD>
static void launch_pixels(PixelPlan& pl, int splits, const float* x, const float* w, const float* wt, const float* bias, float beta, float* out, size_t partial,
                          hipStream_t st)
{
    const dim3 grid(pl.g.ptiles8 * 8 * pl.g.qtiles, 1, splits);
    if (pl.kind == PIXELS_PATCH) {
        if (BWD && pl.g.osx == 2) {
            const dim3 most(patch_blocks(grid.x), 1, grid.z);
            if (pl.patch.nu == 1)
                N2D2HIP_LAUNCH_T(conv_f32_patch_kernel, (2, 2, 2, 2, 2, 9, false, 4), most, dim3(256), 0, st, pl.g, x, w, (const v4u*)wt, bias, beta, out, partial);
            else
                N2D2HIP_LAUNCH_T(conv_f32_patch_kernel, (2, 2, 2, 2, 4, 9, false, 4), most, dim3(256), 0, st, pl.g, x, w, (const v4u*)wt, bias, beta, out, partial);
        } else if (pl.patch.wq == 1) launch_patch<1, 4, 2, 2, true>(pl, grid, x, w, wt, bias, beta, out, partial, st);
        else if (pl.patch.np == 2) launch_patch<2, 2, 2, 2, true>(pl, grid, x, w, wt, bias, beta, out, partial, st);
        else launch_patch<2, 2, 2, 4, false>(pl, grid, x, w, wt, bias, beta, out, partial, st);
        return;
    }
    if (pl.kind == PIXELS_PARTS) {
        const auto run = [&](auto wq_, auto mq_, auto np_, auto chunk_, auto fold_) {
            constexpr int WQ = decltype(wq_)::value, MQ = decltype(mq_)::value, NP = decltype(np_)::value;
            constexpr bool CHUNK = decltype(chunk_)::value, FOLD = decltype(fold_)::value;
            N2D2HIP_LAUNCH_T(conv_f32_taps_kernel, (WQ, 4 / WQ, MQ, NP, CHUNK, FOLD), grid, dim3(256), 0, st, pl.g, x, w, (const v4u*)wt, bias, beta, out, partial);
        };
        using I1 = std::integral_constant<int, 1>;
        using I2 = std::integral_constant<int, 2>;
        using I4 = std::integral_constant<int, 4>;
        const auto shape = [&](auto chunk_, auto fold_) {
            if (pl.patch.wq == 4) run(I4{}, I2{}, I4{}, chunk_, fold_);
            else if (pl.patch.wq == 1 && pl.patch.mq == 1) run(I1{}, I1{}, I2{}, chunk_, fold_);
            else if (pl.patch.wq == 1) run(I1{}, I2{}, I2{}, chunk_, fold_);
            else run(I2{}, I2{}, I2{}, chunk_, fold_);
        };
        const auto folds = [&](auto chunk_) {
            if (pl.g.c[0].fold) shape(chunk_, std::true_type{});
            else shape(chunk_, std::false_type{});
        };
        pl.chunks ? folds(std::true_type{}) : folds(std::false_type{});
        return;
    }
    if (pl.kind != PIXELS_TAPS) w = wt;
    if (pl.kind == PIXELS_3X3) {
        if (pl.small_q) hipLaunchKernelGGL((conv_f32_3x3_kernel<1, 4>), grid, dim3(256), 0, st, pl.g, x, w, bias, beta, out, partial);
        else hipLaunchKernelGGL((conv_f32_3x3_kernel<2, 2>), grid, dim3(256), 0, st, pl.g, x, w, bias, beta, out, partial);
        return;
    }
    const auto run = [&](auto long_) {
        constexpr bool LONG = decltype(long_)::value;
        if (pl.kind == PIXELS_CHUNK) {
            if (pl.small_q) hipLaunchKernelGGL((conv_f32_chunk_kernel<1, 4, 3, LONG>), grid, dim3(256), 0, st, pl.g, x, w, bias, beta, out, partial);
            else hipLaunchKernelGGL((conv_f32_chunk_kernel<2, 2, 3, LONG>), grid, dim3(256), 0, st, pl.g, x, w, bias, beta, out, partial);
            return;
        }
        if (pl.small_q) hipLaunchKernelGGL((conv_f32_pixel_kernel<BWD, 1, 4, 3, LONG>), grid, dim3(256), 0, st, pl.g, x, w, bias, beta, out, partial);
        else hipLaunchKernelGGL((conv_f32_pixel_kernel<BWD, 2, 2, 3, LONG>), grid, dim3(256), 0, st, pl.g, x, w, bias, beta, out, partial);
    };
    pl.many ? run(std::true_type{}) : run(std::false_type{});
}


// ---- backward-filter
struct FilterPlan {
    bool small_q;              // tiles of 32 q x 128 columns instead of 64 x 64
    int splits;
    FilterGemm g;
};
static FilterGemm filter_gemm(const ConvF32& q)
{
    FilterGemm g = {};
    g.P = q.C * q.kH * q.kW; g.Q = q.O; g.K = q.B * q.oH * q.oW;
    g.C = q.C; g.H = q.H; g.W = q.W; g.kW = q.kW; g.kH = q.kH;
    g.s_y = q.sy; g.s_x = q.sx; g.pt = q.pt; g.pl = q.pl;
    g.oW = q.oW; g.plane = q.oH * q.oW;
    g.imgX = q.C * q.H * q.W; g.imgY = q.O * g.plane; g.rowY = g.plane;
    g.bytesX = (unsigned)(4 * (size_t)q.B * g.imgX); g.bytesY = (unsigned)(4 * (size_t)q.B * g.imgY);
    g.dplane = div_of(g.plane); g.dow = div_of(g.oW);
    return g;
}
static FilterPlan plan_filter(const ConvF32& q)
{
    FilterPlan pl = {};
    FilterGemm& g = pl.g;
    g = filter_gemm(q);
    pl.small_q = g.Q <= 32;
    const long tiles = (long)ceil_div_i(g.P, pl.small_q ? 128 : 64) * ceil_div_i(g.Q, pl.small_q ? 32 : 64);
    // (few tiles: four blocks per CU, two of the wide ones, beyond which the partial results cost more than the last round of
    // blocks; many: three blocks per tile or six per CU)
    long splits = tiles <= 256 ? (pl.small_q ? 512 : 1024) / tiles : std::max(1L, (1535 + tiles) / tiles);
    splits = std::min<long>(splits, std::max(1, g.K / (4 * FK)));
    // No float sum longer than the ranges that 128 x 128 tiles would take, none of those below 512 pixels: the longer, the more
    // it loses (256 -> 256, 3x3, 14 x 14, batch 32: sums of 896 pixels 5.1e-7 from 64 bits and 89 us, of 512 3.7e-7 and 90, with
    // as many partial results 95).
    const long tiles128 = (long)ceil_div_i(g.P, 128) * (g.Q <= 64 ? 1 : ceil_div_i(g.Q, 128));
    const long least = q.ranges ? q.ranges : std::min<long>(std::max(1L, 1024 / tiles128), std::max(1, g.K / (16 * FK)));
    g.kchunk = round_up((int)((g.K + splits - 1) / splits), FK);
    g.fold = least > splits ? std::max((int)(g.K / least) / FK, 1) : 0;
    pl.splits = ceil_div_i(g.K, g.kchunk);
    return pl;
}
// ---- backward-filter of 3x3 kernels on the bf16 matrix cores
struct RowsPlan {
    int nol;                   // log2 of a step's octets of a row; -1: not this kernel
    int qtiles, ctiles, splits;
    FilterRows g;
    size_t values() const { return (size_t)qtiles * ctiles * ROWS_TILE; }
};
static RowsPlan plan_rows(const ConvF32& q)
{
    RowsPlan pl = {};
    pl.nol = -1;
    if (q.kH != 3 || q.kW != 3 || q.sx != q.sy || q.sx > 2 || q.pl != 1 || q.pt > 2 || q.ranges) return pl;
    FilterRows& g = pl.g;
    g.B = q.B; g.C = q.C; g.Q = q.O; g.H = q.H; g.W = q.W; g.oH = q.oH; g.oW = q.oW; g.pt = q.pt;
    // an image's rows of x, the padding above the next one's, and all that the last output row reads
    g.D = std::max(ceil_div_i(q.H + q.pt, q.sy), ceil_div_i((q.oH - 1) * q.sy - q.pt + 3, q.sy));
    const int octets = ceil_div_i(q.oW, 8);
    pl.qtiles = ceil_div_i(q.O, ROWS_Q); pl.ctiles = ceil_div_i(q.C, ROWS_C);
    // Where the layer is large and fills the tiles and octets (us, fp32 kernel / this one): 64 <- 64, 28 x 28, batch 8, 4.6e8 flops 17 / 22;
    // 128 <- 128, 56 x 56, 9.2e8 25 / 26; 64 <- 32, 112 x 112, batch 4, 1.8e9 34 / 28; 71 <- 37 channels, 113 x 75, batch 5, 0.3 filled
    // 52 / 54; 100 <- 48, 56 x 56, batch 16, 0.59 filled 69 / 61.
    const double flops = 2.0 * q.B * q.O * q.oH * q.oW * q.C * 9;
    if (flops < 1.5e9 || (double)q.O * q.C * q.oW < 0.4 * pl.qtiles * ROWS_Q * (double)pl.ctiles * ROWS_C * octets * 8) return pl;
    // a step has 8 octets (4 at stride 2): as many of a row as leave the fewest beyond its end; rows that follow each other share theirs of x
    int best = 1 << 30;
    for (int nol = q.sx == 1 ? 3 : 2; nol >= 0; --nol)
        if (round_up(octets, 1 << nol) < best) {
            best = round_up(octets, 1 << nol);
            pl.nol = nol;
        }
    const int rows = (q.sx == 1 ? 8 : 4) >> pl.nol;
    g.pieces = best >> pl.nol;
    g.chunks = ceil_div_i((long)q.B * g.D, rows) * g.pieces;
    pl.splits = (int)std::min<long>(std::max(256L / ((long)pl.qtiles * pl.ctiles), 1L), ceil_div_i(g.chunks, 4));
    g.per = ceil_div_i(g.chunks, pl.splits);
    pl.splits = ceil_div_i(g.chunks, g.per);
    g.masked = q.oW % 8 != 0 || q.W % (8 * q.sx) != 0;
    g.bytesX = (unsigned)(4 * (size_t)q.B * q.C * q.H * q.W); g.bytesY = (unsigned)(4 * (size_t)q.B * q.O * q.oH * q.oW);
    g.dD = div_of(g.D); g.dSD = div_of(q.sx * g.D); g.dpieces = div_of(g.pieces);
    return pl;
}
static void launch_rows(const RowsPlan& pl, int s, const float* x, const float* dy, float beta, float* dw, float* ws, hipStream_t st)
{
    const dim3 grid(pl.ctiles, pl.qtiles, pl.splits);
    const auto run = [&](auto s_, auto nol_) {
        constexpr int S = decltype(s_)::value, NOL = decltype(nol_)::value;
        N2D2HIP_LAUNCH_T(conv_f32_filter_rows_kernel, (S, NOL), grid, dim3(512), 0, st, pl.g, x, dy, ws);
    };
    const auto octets = [&](auto s_) {
        if (pl.nol == 0) run(s_, std::integral_constant<int, 0>{});
        else if (pl.nol == 1) run(s_, std::integral_constant<int, 1>{});
        else if (pl.nol == 2) run(s_, std::integral_constant<int, 2>{});
        else if constexpr (decltype(s_)::value == 1) run(s_, std::integral_constant<int, 3>{});
    };
    s == 1 ? octets(std::integral_constant<int, 1>{}) : octets(std::integral_constant<int, 2>{});
    N2D2HIP_LAUNCH(conv_f32_reduce_rows_kernel, dim3((unsigned)(pl.values() / 64)), dim3(256), 0, st, (const float*)ws, pl.splits, pl.ctiles, pl.values(), pl.g.Q,
                   pl.g.C, beta, dw);
}
// What the small filter kernel runs of a pass: backward-filter, or backward-data of a spanning kernel as a sum over "pixels" o,
// dx[b][k] = sum_o dy[b][o] w[o][k], with the images as rows of q and the weights of an output as columns of p.
static FilterGemm small_gemm(const ConvF32& q, int pass)
{
    if (pass == PASS_BWD_FILTER) return filter_gemm(q);
    FilterGemm g = {};
    g.P = q.C * q.kH * q.kW; g.Q = q.B; g.K = q.O;
    g.C = g.P; g.H = g.W = g.kW = g.kH = g.s_y = g.s_x = g.oW = g.plane = 1;
    g.imgX = g.P; g.imgY = 1; g.rowY = q.O;
    g.dplane = div_of(1); g.dow = div_of(1);
    return g;
}
// The small kernel: enough ranges for two blocks per CU, none below 128 pixels (two rounds of a wave's loads).
static int small_filter_splits(const FilterGemm& g)
{
    const long tiles = (long)ceil_div_i(g.P, 16) * ceil_div_i(g.Q, 16);
    return (int)std::max(1L, std::min<long>(512 / tiles, g.K / 128));
}
// -> ranges, and their length in g (a workspace too small for the partial results: one range)
static int small_filter_ranges(FilterGemm& g, size_t n, const double* ws, size_t ws_bytes)
{
    int splits = small_filter_splits(g);
    if (splits * n * sizeof(double) > ws_bytes || ((size_t)ws & 7)) splits = 1;
    g.kchunk = round_up(ceil_div_i(g.K, splits), 64);
    return ceil_div_i(g.K, g.kchunk);
}
static int run_small_filter(FilterGemm g, const float* x, const float* dy, float beta, float* out, double* ws, size_t ws_bytes, hipStream_t st)
{
    const size_t n = (size_t)g.Q * g.P;
    const int splits = small_filter_ranges(g, n, ws, ws_bytes);
    hipLaunchKernelGGL(conv_f32_filter_small_kernel, dim3(ceil_div_i(g.P, 16), ceil_div_i(g.Q, 16), splits), dim3(256), 0, st, g, x, dy,
                       splits > 1 ? ws : (double*)nullptr, beta, out);
    if (splits > 1)
        hipLaunchKernelGGL(conv_f32_reduce_partials_kernel<double>, dim3(reduce_grid(n)), dim3(256), 0, st, (const double*)ws, splits, n, beta, out,
                           (const float*)nullptr, 1, 1);
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}
static void launch_filter(const FilterPlan& pl, const float* x, const float* dy, float* out, hipStream_t st)
{
    const dim3 grid(ceil_div_i(pl.g.P, pl.small_q ? 128 : 64), ceil_div_i(pl.g.Q, pl.small_q ? 32 : 64), pl.splits);
    const auto run = [&](auto long_, auto fold_) {
        constexpr bool LONG = decltype(long_)::value, FOLD = decltype(fold_)::value;
        if (pl.small_q) hipLaunchKernelGGL((conv_f32_filter_kernel<1, 4, 2, LONG, FOLD>), grid, dim3(256), 0, st, pl.g, x, dy, out);
        else hipLaunchKernelGGL((conv_f32_filter_kernel<2, 2, 2, LONG, FOLD>), grid, dim3(256), 0, st, pl.g, x, dy, out);
    };
    const auto pick = [&](auto long_) { pl.g.fold ? run(long_, std::true_type{}) : run(long_, std::false_type{}); };
    pl.g.kH + pl.g.kW > 31 ? pick(std::true_type{}) : pick(std::false_type{});
}

// The kernel and its order of K.  Kernels of several taps whose tiles read runs of source pixels that fit its LDS, with less than 2 / 5
// of padding to 32 channels: the patch kernel, on the bf16 matrix cores.  Else 3x3 kernels, forward or at stride 1: four channels with their taps at a time.  Chunks of 16 channels at one
// tap: 1x1 kernels, kernels of more than 31 rows and columns (1 x 64, 128 -> 128: 138 -> 113 us) and backward-data, where padding
// the channels to them costs less than testing every load (about a fifth).  Both lay the weights out first (a launch of 3 us: even at 3 to 7e8 flops).
static int pixels_kind(const ConvF32& q, int pass)
{
    const int ch = pass == PASS_FWD ? q.C : q.O, T = q.kH * q.kW;
    if (2.0 * q.B * q.O * q.oH * q.oW * q.C * T < 5.0e8 || (size_t)(q.O + 64) * (q.C + 64) * (T + 2) >= ((size_t)1 << 28))
        return PIXELS_TAPS;
    if (T > 1 && round_up(ch, PK) * 5 <= ch * 7 && !(pass == PASS_FWD && (q.choice & N2D2HIP_KERNEL_F32_TERMS))) {
        // (backward-data at other strides and kernels: the classes are few taps to a step each; 128 <- 256, stride 2, 27 x 27, batch 33, a class a
        // launch: 58 us against 53)
        if (patch_fours(q, pass) ? patch_shape(q, pass, fours_class(q)).nu
            : (pass == PASS_FWD || (q.sx == 1 && q.sy == 1)) && patch_shape(q, pass, pixel_classes(q, pass)[0]).nu) return PIXELS_PATCH;
    }
    // The other large ones whose K is more than a few steps: conv_f32_taps_kernel, but where a third of a tile's rows is empty (17 <- 253, 5x5: 149 us, pixel
    // kernel 140).  us, fp32 kernels / this: below the rule 33 -> 79, 3x3, 55 x 72, batch 6, 1.1e9 flops 23.7 / 27.4; 16 -> 54, 3x3, 97 x 27, batch 14, 5.7e8
    // 15.4 / 22; 64 -> 64, 1x1, 56 x 56, batch 64, K 64 31.2 / 31; others at the kernel.
    const int rows = pass == PASS_FWD ? q.O : q.C;
    if (!(pass == PASS_FWD && (q.choice & N2D2HIP_KERNEL_F32_TERMS)) && q.kH + q.kW <= 31 && !q.ranges && q.sx * q.sy <= PIXEL_CLASSES
        && 2.0 * q.B * q.O * q.oH * q.oW * q.C * T >= 1.5e9 && (long)ch * T >= 200 && (rows <= 16 || rows >= 22))
        return PIXELS_PARTS;
    if (q.kH == 3 && q.kW == 3 && (pass == PASS_FWD || (q.sx == 1 && q.sy == 1)) && round_up(ch, 4) * 5 <= ch * 7)
        return PIXELS_3X3;
    return (pass == PASS_BWD_DATA || T == 1 || q.kH + q.kW > 31) && round_up(ch, GK) * 5 <= ch * 6 ? PIXELS_CHUNK : PIXELS_TAPS;
}
static std::vector<PixelClass> launch_classes(const ConvF32& q, int pass, int kind)
{
    return kind == PIXELS_PATCH && patch_fours(q, pass) ? std::vector<PixelClass>{fours_class(q)} : pixel_classes(q, pass);
}
static size_t laid_weights(const ConvF32& q, int pass, int kind)
{
    const int ch = pass == PASS_FWD ? q.C : q.O, rows = pass == PASS_FWD ? q.O : q.C, qpad = round_up(rows, rows <= 32 ? 32 : 64);
    if (kind == PIXELS_TAPS) return 0;
    if (kind == PIXELS_PARTS) {
        const std::vector<PixelClass> cls = pixel_classes(q, pass);
        size_t steps = 0;
        for (const PixelClass& c : cls) steps += taps_steps(q, pass, c);
        return steps * (round_up(rows, taps_shape(q, pass, cls).rows()) / 16) * (PATCH_FRAG / 4);
    }
    if (kind == PIXELS_PATCH) return (size_t)ceil_div_i(ch, PK) * q.kH * q.kW * (round_up(rows, 128) / 16) * (PATCH_FRAG / 4);
    return kind == PIXELS_3X3 ? (size_t)(ch + 3) / 4 * qpad * W33 : (size_t)round_up(ch, GK) * q.kH * q.kW * qpad;
}

// Floats of workspace a pass takes when it may split its K
static size_t pass_workspace(const ConvF32& q, int pass)
{
    if (pass == PASS_BWD_FILTER) {
        const RowsPlan rows = plan_rows(q);
        if (rows.nol >= 0) return rows.splits * rows.values();
        const FilterPlan pl = plan_filter(q);
        return (size_t)pl.splits * pl.g.Q * pl.g.P;
    }
    const int kind = pixels_kind(q, pass);
    const std::vector<PixelClass> cls = launch_classes(q, pass, kind);
    const size_t n = (size_t)q.B * (pass == PASS_FWD ? (size_t)q.O * q.oH * q.oW : (size_t)q.C * q.H * q.W);
    int splits = 1;
    for (size_t i = 0; i < cls.size(); i += PIXEL_CLASSES)
        splits = std::max(splits, plan_pixels(q, pass, std::vector<PixelClass>(cls.begin() + i, cls.begin() + std::min(cls.size(), i + PIXEL_CLASSES)), kind).splits);
    return (splits > 1 ? splits * n : 0) + laid_weights(q, pass, kind);
}

// Runs one pass of q (which qualifies for the matrix cores): out = pass(x, w) + beta * out (+ bias[channel] forward).
// The tensors are the pass's own operands: forward (x, w), backward-data (dy, w), backward-filter (x, dy).
static int run_pass(const ConvF32& q, int pass, const float* a, const float* b, const float* bias, int bias_plane, int bias_channels, float beta,
                    float* out, float* ws, size_t ws_floats, hipStream_t st)
{
    if (pass == PASS_BWD_FILTER) {
        const RowsPlan rows = plan_rows(q);
        if (rows.nol >= 0 && rows.splits * rows.values() <= ws_floats) {
            launch_rows(rows, q.sx, a, b, beta, out, ws, st);
            N2D2HIP_HIP_CHECK(hipGetLastError());
            return N2D2HIP_OK;
        }
        FilterPlan pl = plan_filter(q);
        const size_t n = (size_t)pl.g.Q * pl.g.P;
        bool direct = false;
        if (pl.splits * n > ws_floats) {
            pl.splits = 1;
            pl.g.kchunk = round_up(pl.g.K, FK);
        }
        direct = pl.splits == 1 && beta == 0.0f && !bias;
        N2D2HIP_REQUIRE(direct || pl.splits * n <= ws_floats, N2D2HIP_ERR_WORKSPACE, "convolution: workspace of %zu bytes, %zu needed", 4 * ws_floats,
                        4 * pl.splits * n);
        launch_filter(pl, a, b, direct ? out : ws, st);
        if (!direct)
            hipLaunchKernelGGL(conv_f32_reduce_partials_kernel<float>, dim3(reduce_grid(n)), dim3(256), 0, st, (const float*)ws, pl.splits, n, beta, out, bias,
                               bias_plane, bias_channels);
        N2D2HIP_HIP_CHECK(hipGetLastError());
        return N2D2HIP_OK;
    }
    const size_t n = (size_t)q.B * (pass == PASS_FWD ? (size_t)q.O * q.oH * q.oW : (size_t)q.C * q.H * q.W);
    // (the weights laid out come first in the workspace; without room for them, K tap by tap)
    int kind = pixels_kind(q, pass);
    const size_t nlaid = laid_weights(q, pass, kind);
    if (nlaid > ws_floats || ((size_t)ws & 15)) kind = PIXELS_TAPS;
    const std::vector<PixelClass> cls = launch_classes(q, pass, kind);
    std::vector<PixelPlan> plans;
    int splits = 1;
    for (size_t i = 0; i < cls.size(); i += PIXEL_CLASSES) {
        plans.push_back(plan_pixels(q, pass, std::vector<PixelClass>(cls.begin() + i, cls.begin() + std::min(cls.size(), i + PIXEL_CLASSES)), kind));
        splits = std::max(splits, plans.back().splits);
    }
    const float* wt = ws;
    if (kind != PIXELS_TAPS) {
        const PixelGemm& g = plans[0].g;
        const int total = (int)(kind == PIXELS_3X3 ? nlaid : kind == PIXELS_PATCH || kind == PIXELS_PARTS ? nlaid / 12 : nlaid / 4);
        const dim3 grid(std::min((total + 255) / 256, 4096));
        if (kind == PIXELS_3X3) hipLaunchKernelGGL(conv_f32_lay_weights3x3_kernel, grid, dim3(256), 0, st, b, ws, total, g.Q, g.qpad, g.Ch, g.qs, g.chs);
        else if (kind == PIXELS_PATCH)
            N2D2HIP_LAUNCH(conv_f32_lay_parts_kernel, dim3(std::min(ceil_div_i(total, LAY_THREADS), 16384)), dim3(LAY_THREADS), 0, st, b, (v4u*)ws, total, g.Q, g.qpad / 16, g.Ch, g.T, g.qs, g.chs);
        else if (kind == PIXELS_PARTS) {
            if (plans[0].chunks) N2D2HIP_LAUNCH_T(conv_f32_lay_taps_kernel, (true), grid, dim3(256), 0, st, g, b, (v4u*)ws, total);
            else N2D2HIP_LAUNCH_T(conv_f32_lay_taps_kernel, (false), grid, dim3(256), 0, st, g, b, (v4u*)ws, total);
        } else hipLaunchKernelGGL(conv_f32_lay_weights_kernel, grid, dim3(256), 0, st, b, ws, total, g.Q, g.qpad, g.Ch, g.T, g.qs, g.chs);
        ws += nlaid;
        ws_floats -= nlaid;
    }
    if (splits * n > ws_floats) {                           // no room for partial results: a block takes all ranges
        for (PixelPlan& pl : plans) {
            if (kind == PIXELS_PATCH) {          // (whose ranges are not walked one by one: a single one of all chunks)
                const int fold = patch_fold(q, pass, cls[0]), chunks = ceil_div_i(pl.g.Ch, PK);
                pl.g.c[0].kchunk = chunks;
                pl.g.c[0].fold = fold < chunks ? fold : 0;
            } else if (kind == PIXELS_PARTS) {
                const int fold = taps_fold(q, pass);
                int most = 0;
                for (int i = 0; i < pl.g.nclass; ++i) {
                    pl.g.c[i].kchunk = taps_steps(q, pass, pl.g.c[i]);
                    most = std::max(most, pl.g.c[i].kchunk);
                }
                for (int i = 0; i < pl.g.nclass; ++i) pl.g.c[i].fold = fold < most ? fold : 0;
            } else {
                pl.g.nz *= pl.splits;
            }
        }
        splits = 1;
    }
    for (PixelPlan& pl : plans) {
        float* dst = splits > 1 ? ws : out;
        // (every launch runs the ranges of the pass, so that each partial result is complete)
        if (pass == PASS_FWD) launch_pixels<false>(pl, splits, a, b, wt, splits > 1 ? nullptr : bias, splits > 1 ? 0.0f : beta, dst, splits > 1 ? n : 0, st);
        else launch_pixels<true>(pl, splits, a, b, wt, nullptr, splits > 1 ? 0.0f : beta, dst, splits > 1 ? n : 0, st);
    }
    if (splits > 1)
        hipLaunchKernelGGL(conv_f32_reduce_partials_kernel<float>, dim3(reduce_grid(n)), dim3(256), 0, st, (const float*)ws, splits, n, beta, out, bias,
                           bias_plane, bias_channels);
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

static DataSmall small_data(const ConvF32& q)
{
    const int T = q.kH * q.kW;
    return DataSmall{q.B * q.H * q.W, q.C, q.O, T, q.O * T, q.kW, q.H * q.W, q.W, q.oH, q.oW, q.sy, q.sx, q.pt, q.pl,
                     (unsigned)(4 * (size_t)q.O * q.C * T), (unsigned)(4 * (size_t)q.B * q.O * q.oH * q.oW),
                     div_of(q.H * q.W), div_of(q.W), div_of(T), div_of(q.kW), div_of(q.sy), div_of(q.sx)};
}
// Waves of a block, and tiles: of the block, or one of each wave: where the tiles are more than the chip holds blocks, and a wave's share of K
// is short.  us, all of a block / one of a wave (tiles, K): 804, 14 4.0 / 4.0; 1296, 64 4.5 / 5.8; 1674, 128 7.6 / 8.3; 1785, 36 5.1 / 4.9; 1890, 28
// 4.8 / 4.6; 2232, 53 6.1 / 6.7; 2444, 16 5.5 / 4.0; 2366, 91 8.8 / 8.4; 4200, 9 7.1 / 4.6; 23674, 9 28.2 / 14.3.
struct SmallDataShape {
    int waves, tiles, across;
    unsigned blocks;                             // (2.3e5 / K at most)
};
static SmallDataShape small_data_shape(const DataSmall& g)
{
    const int dtiles = ceil_div_i(g.P, 16), ctiles = ceil_div_i(g.C, 16);
    SmallDataShape s = {};
    s.waves = g.K <= 256 ? 4 : g.K <= 1024 ? 8 : 16;
    s.tiles = s.waves == 4 && (long)dtiles * ctiles > 1792 && g.K <= 112 ? 4 : 1;
    s.across = ceil_div_i(dtiles, s.tiles);
    s.blocks = (unsigned)(s.across * ctiles);
    return s;
}
template <class F>
static void small_data_kernel(const SmallDataShape& s, F&& f)
{
    if (s.tiles == 4) f(std::integral_constant<int, 4>{}, std::integral_constant<int, 4>{});
    else if (s.waves == 4) f(std::integral_constant<int, 4>{}, std::integral_constant<int, 1>{});
    else if (s.waves == 8) f(std::integral_constant<int, 8>{}, std::integral_constant<int, 1>{});
    else f(std::integral_constant<int, 16>{}, std::integral_constant<int, 1>{});
}

} // namespace n2d2hip

using namespace n2d2hip;

extern "C" {

static int conv_forward(const char* who, const n2d2hip_conv_desc* desc, int B, int H, int W, const float* x, const float* w, const float* bias, float beta, float* y,
                        const SatStore& sat, void* workspace, size_t workspace_bytes, n2d2hip_stream_t stream)
{
    ConvF32 q;
    int st = make_conv(desc, B, H, W, false, &q, who);
    if (st != N2D2HIP_OK) return st;
    N2D2HIP_REQUIRE(x && w && y, N2D2HIP_ERR_INVALID, "%s: null pointer", who);
    bool sat_done = false;
    const auto forward = [&] {
        if (f32_path(q, PASS_FWD) == F32_PATH_GEMM) {
            float* ws = (float*)workspace;
            const size_t nws = workspace ? workspace_bytes / sizeof(float) : 0;
            if (spans_input(q)) {
                int pass;
                const ConvF32 m = product_of(q, PASS_FWD, &pass);
                // (without a workspace that holds its partial results: the convolution as it stands, whose kernels keep a tap in each
                // of a wave's 64 lanes, or the direct kernels)
                if (q.B <= 64 * GRID_Y && pass_workspace(m, pass) <= nws)
                    return run_pass(m, pass, w, x, bias, 1, q.O, beta, y, ws, nws, (hipStream_t)stream);
                if (many_taps(q)) return run_direct(q, PASS_FWD, x, w, bias, beta, y, (hipStream_t)stream, sat, &sat_done);
            }
            return run_pass(q, PASS_FWD, x, w, bias, q.oH * q.oW, q.O, beta, y, ws, nws, (hipStream_t)stream);
        }
        return run_direct(q, PASS_FWD, x, w, bias, beta, y, (hipStream_t)stream, sat, &sat_done);
    };
    st = forward();
    if (st != N2D2HIP_OK || !sat.alpha || sat_done) return st;
    return n2d2hip_sat_act_forward(y, sat.fp, (size_t)q.B * q.O * q.oH * q.oW, sat.range, sat.alpha, stream);
}

int n2d2hip_conv2d_f32_forward(const n2d2hip_conv_desc* desc, int B, int H, int W, const float* x, const float* w, const float* bias,
                               float beta, float* y, void* workspace, size_t workspace_bytes, n2d2hip_stream_t stream)
{
    return conv_forward("n2d2hip_conv2d_f32_forward", desc, B, H, W, x, w, bias, beta, y, SatStore{}, workspace, workspace_bytes, stream);
}

int n2d2hip_conv2d_f32_forward_sat(const n2d2hip_conv_desc* desc, int B, int H, int W, const float* x, const float* w, const float* bias, float* y,
                                   float* full_precision, float range, const float* alpha, void* workspace, size_t workspace_bytes, n2d2hip_stream_t stream)
{
    N2D2HIP_REQUIRE(alpha && full_precision != y, N2D2HIP_ERR_INVALID, "n2d2hip_conv2d_f32_forward_sat: bad argument");
    return conv_forward("n2d2hip_conv2d_f32_forward_sat", desc, B, H, W, x, w, bias, 0.0f, y, SatStore{full_precision, range, alpha}, workspace, workspace_bytes,
                        stream);
}

int n2d2hip_conv2d_f32_backward_data(const n2d2hip_conv_desc* desc, int B, int H, int W, const float* w, const float* diff_y, float beta,
                                     float* diff_x, void* workspace, size_t workspace_bytes, n2d2hip_stream_t stream)
{
    ConvF32 q;
    const int st = make_conv(desc, B, H, W, true, &q, "n2d2hip_conv2d_f32_backward_data");
    if (st != N2D2HIP_OK) return st;
    N2D2HIP_REQUIRE(w && diff_y && diff_x, N2D2HIP_ERR_INVALID, "n2d2hip_conv2d_f32_backward_data: null pointer");
    const int path = f32_path(q, PASS_BWD_DATA);
    if (path == F32_PATH_SMALL)
        return run_small_filter(small_gemm(q, PASS_BWD_DATA), w, diff_y, beta, diff_x, (double*)workspace, workspace ? workspace_bytes : 0, (hipStream_t)stream);
    if (path == F32_PATH_SMALL_DATA) {
        const DataSmall g = small_data(q);
        const SmallDataShape shape = small_data_shape(g);
        small_data_kernel(shape, [&](auto waves_, auto tiles_) {
            constexpr int WAVES = decltype(waves_)::value, TILES = decltype(tiles_)::value;
            N2D2HIP_LAUNCH_T(conv_f32_data_small_kernel, (WAVES, TILES), dim3(shape.blocks), dim3(64 * WAVES), 0, (hipStream_t)stream, g, shape.across, w, diff_y, beta,
                             diff_x);
        });
        N2D2HIP_HIP_CHECK(hipGetLastError());
        return N2D2HIP_OK;
    }
    if (path == F32_PATH_GEMM) {
        float* ws = (float*)workspace;
        const size_t nws = workspace ? workspace_bytes / sizeof(float) : 0;
        if (spans_input(q)) {
            int pass;
            const ConvF32 m = product_of(q, PASS_BWD_DATA, &pass);
            return run_pass(m, pass, w, diff_y, nullptr, 1, 1, beta, diff_x, ws, nws, (hipStream_t)stream);
        }
        return run_pass(q, PASS_BWD_DATA, diff_y, w, nullptr, 1, 1, beta, diff_x, ws, nws, (hipStream_t)stream);
    }
    return run_direct(q, PASS_BWD_DATA, diff_y, w, nullptr, beta, diff_x, (hipStream_t)stream);
}

size_t n2d2hip_conv2d_f32_workspace_bytes(const n2d2hip_conv_desc* desc, int B, int H, int W)
{
    ConvF32 q;
    if (make_conv(desc, B, H, W, true, &q, "n2d2hip_conv2d_f32_workspace_bytes") != N2D2HIP_OK)
        return 0;
    size_t need = 0;
    for (int pass : {PASS_FWD, PASS_BWD_DATA, PASS_BWD_FILTER}) {
        const int path = f32_path(q, pass);
        if (path == F32_PATH_SMALL) {
            const FilterGemm g = small_gemm(q, pass);
            const int splits = small_filter_splits(g);
            need = std::max(need, splits > 1 ? splits * (size_t)g.Q * g.P * 2 : 0);
        } else if (path == F32_PATH_GEMM) {
            int as = pass;
            const ConvF32 m = spans_input(q) ? product_of(q, pass, &as) : q;
            need = std::max(need, pass_workspace(m, as));
            if (pass == PASS_BWD_FILTER) need = std::max(need, (size_t)q.O * q.C * q.kH * q.kW);     // (always has one)
        }
    }
    if (depthwise_strips(q) && f32_path(q, PASS_BWD_FILTER) == F32_PATH_DIRECT)
        need = std::max(need, depthwise_filter_bytes(q, depthwise_filter_ranges(q)) / sizeof(float));
    return need * sizeof(float);
}

int n2d2hip_conv2d_f32_backward_filter(const n2d2hip_conv_desc* desc, int B, int H, int W, const float* x, const float* diff_y, float beta,
                                       float* diff_w, void* workspace, size_t workspace_bytes, n2d2hip_stream_t stream)
{
    ConvF32 q;
    const int st = make_conv(desc, B, H, W, true, &q, "n2d2hip_conv2d_f32_backward_filter");
    if (st != N2D2HIP_OK) return st;
    N2D2HIP_REQUIRE(x && diff_y && diff_w, N2D2HIP_ERR_INVALID, "n2d2hip_conv2d_f32_backward_filter: null pointer");
    const size_t nw = (size_t)q.O * q.Cw * q.kH * q.kW;
    N2D2HIP_REQUIRE(nw < ((size_t)1 << 31), N2D2HIP_ERR_INVALID, "n2d2hip_conv2d_f32_backward_filter: too many weights");
    const int path = f32_path(q, PASS_BWD_FILTER);
    if (path == F32_PATH_SMALL)
        return run_small_filter(small_gemm(q, PASS_BWD_FILTER), x, diff_y, beta, diff_w, (double*)workspace, workspace ? workspace_bytes : 0, (hipStream_t)stream);
    if (path == F32_PATH_GEMM) {
        int pass = PASS_BWD_FILTER;
        const bool fc = spans_input(q);
        const ConvF32 m = fc ? product_of(q, PASS_BWD_FILTER, &pass) : q;
        const size_t need = std::max(nw, pass_workspace(m, pass)) * sizeof(float);
        N2D2HIP_REQUIRE(workspace && workspace_bytes >= need, N2D2HIP_ERR_WORKSPACE,
                        "n2d2hip_conv2d_f32_backward_filter: workspace of %zu bytes, %zu needed (n2d2hip_conv2d_f32_workspace_bytes)",
                        workspace_bytes, need);
        return run_pass(m, pass, x, diff_y, nullptr, 1, 1, beta, diff_w, (float*)workspace, workspace_bytes / sizeof(float), (hipStream_t)stream);
    }
    if (depthwise_strips(q))
        return run_depthwise(q, PASS_BWD_FILTER, x, diff_y, nullptr, beta, diff_w, workspace, workspace ? workspace_bytes : 0, (hipStream_t)stream);
    hipLaunchKernelGGL(conv_f32_backward_filter_kernel, dim3((unsigned)nw), dim3(TBLOCK), 0, (hipStream_t)stream, q, x, diff_y, beta, diff_w);
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

// (neither product in ranges, whose partial results a second launch adds up; 2^30 tiles at most)
static bool small_pair(const ConvF32& q, SmallPair* a, long* blocks)
{
    if (f32_path(q, PASS_BWD_FILTER) != F32_PATH_SMALL || f32_path(q, PASS_BWD_DATA) != F32_PATH_SMALL) return false;
    *blocks = 0;
    for (int k = 0; k < 2; ++k) {
        SmallProduct& s = a->of[k];
        s.g = small_gemm(q, k ? PASS_BWD_DATA : PASS_BWD_FILTER);
        if (small_filter_splits(s.g) > 1) return false;
        s.g.kchunk = round_up(s.g.K, 64);
        s.ptiles = ceil_div_i(s.g.P, 16);
        if (k) a->first = (unsigned)*blocks;
        *blocks += (long)s.ptiles * ceil_div_i(s.g.Q, 16);
        if (*blocks >= 1L << 30) return false;
    }
    return true;
}
int n2d2hip_conv2d_f32_backward(const n2d2hip_conv_desc* desc, int B, int H, int W, const float* x, const float* w, const float* diff_y, float beta_w,
                                float* diff_w, float beta_x, float* diff_x, void* workspace, size_t workspace_bytes, n2d2hip_stream_t stream)
{
    ConvF32 q;
    const int st = make_conv(desc, B, H, W, true, &q, "n2d2hip_conv2d_f32_backward");
    if (st != N2D2HIP_OK) return st;
    N2D2HIP_REQUIRE(x && w && diff_y && diff_w && diff_x, N2D2HIP_ERR_INVALID, "n2d2hip_conv2d_f32_backward: null pointer");
    const size_t nx = (size_t)q.B * q.C * q.H * q.W, nw = (size_t)q.O * q.Cw * q.kH * q.kW, ny = (size_t)q.B * q.O * q.oH * q.oW;
    const auto disjoint = [](const float* a, size_t na, const float* b, size_t nb) { return a + na <= b || b + nb <= a; };
    // (results over the operands, as the two passes one behind the other allow: in that order)
    const bool apart = disjoint(diff_w, nw, x, nx) && disjoint(diff_w, nw, w, nw) && disjoint(diff_w, nw, diff_y, ny) && disjoint(diff_x, nx, x, nx)
                       && disjoint(diff_x, nx, w, nw) && disjoint(diff_x, nx, diff_y, ny) && disjoint(diff_x, nx, diff_w, nw);
    SmallPair a;
    long blocks;
    if (apart && small_pair(q, &a, &blocks)) {
        a.of[0].srcX = x; a.of[0].srcY = diff_y; a.of[0].beta = beta_w; a.of[0].out = diff_w;
        a.of[1].srcX = w; a.of[1].srcY = diff_y; a.of[1].beta = beta_x; a.of[1].out = diff_x;
        N2D2HIP_LAUNCH(conv_f32_small_pair_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, a);
        N2D2HIP_HIP_CHECK(hipGetLastError());
        return N2D2HIP_OK;
    }
    if (apart && f32_path(q, PASS_BWD_FILTER) == F32_PATH_SMALL && f32_path(q, PASS_BWD_DATA) == F32_PATH_SMALL_DATA) {
        SmallBoth b = {};
        b.data = small_data(q);
        const SmallDataShape shape = small_data_shape(b.data);
        b.across = shape.across;
        b.first = shape.blocks;
        b.filter.g = small_gemm(q, PASS_BWD_FILTER);
        const size_t n = (size_t)b.filter.g.Q * b.filter.g.P;
        const int ranges = small_filter_ranges(b.filter.g, n, (const double*)workspace, workspace ? workspace_bytes : 0);
        b.filter.ptiles = ceil_div_i(b.filter.g.P, 16);
        const long ftiles = (long)b.filter.ptiles * ceil_div_i(b.filter.g.Q, 16);
        if (ftiles * ranges < 1L << 30) {
            b.ftiles = (int)ftiles;
            b.filter.srcX = x; b.filter.srcY = diff_y; b.filter.beta = beta_w; b.filter.out = diff_w;
            b.w = w; b.dy = diff_y; b.beta = beta_x; b.dx = diff_x;
            b.partial = ranges > 1 ? (double*)workspace : nullptr;
            const dim3 grid(b.first + (unsigned)(ftiles * ranges));
            small_data_kernel(shape, [&](auto waves_, auto tiles_) {
                constexpr int WAVES = decltype(waves_)::value, TILES = decltype(tiles_)::value;
                N2D2HIP_LAUNCH_T(conv_f32_small_both_kernel, (WAVES, TILES), grid, dim3(64 * WAVES), 0, (hipStream_t)stream, b);
            });
            if (ranges > 1)
                hipLaunchKernelGGL(conv_f32_reduce_partials_kernel<double>, dim3(reduce_grid(n)), dim3(256), 0, (hipStream_t)stream, (const double*)workspace,
                                   ranges, n, beta_w, diff_w, (const float*)nullptr, 1, 1);
            N2D2HIP_HIP_CHECK(hipGetLastError());
            return N2D2HIP_OK;
        }
    }
    const int rc = n2d2hip_conv2d_f32_backward_filter(desc, B, H, W, x, diff_y, beta_w, diff_w, workspace, workspace_bytes, stream);
    return rc != N2D2HIP_OK ? rc : n2d2hip_conv2d_f32_backward_data(desc, B, H, W, w, diff_y, beta_x, diff_x, workspace, workspace_bytes, stream);
}

int n2d2hip_conv2d_f32_backward_bias(int B, int O, int oH, int oW, const float* diff_y, float beta, float* diff_bias, n2d2hip_stream_t stream)
{
    N2D2HIP_REQUIRE(B > 0 && O > 0 && oH > 0 && oW > 0 && diff_y && diff_bias, N2D2HIP_ERR_INVALID, "n2d2hip_conv2d_f32_backward_bias: bad argument");
    hipLaunchKernelGGL(conv_f32_backward_bias_kernel, dim3(O), dim3(TBLOCK), 0, (hipStream_t)stream, B, O, oH * oW, diff_y, beta, diff_bias);
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

int n2d2hip_softmax_f32_forward(const float* x, float* y, int B, int C, int H, int W, n2d2hip_stream_t stream)
{
    N2D2HIP_REQUIRE(B > 0 && C > 0 && H > 0 && W > 0 && x && y, N2D2HIP_ERR_INVALID, "n2d2hip_softmax_f32_forward: bad argument");
    hipLaunchKernelGGL(C <= 16 ? softmax_f32_kernel<16> : softmax_f32_kernel<0>, dim3(grid_for((size_t)B * H * W)), dim3(TBLOCK), 0, (hipStream_t)stream, x, y, B, C, H * W);
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

int n2d2hip_rectifier_f32_forward(float* x, size_t n, float leak_slope, float clipping, n2d2hip_stream_t stream)
{
    N2D2HIP_REQUIRE(x && n > 0 && clipping >= 0.0f, N2D2HIP_ERR_INVALID, "n2d2hip_rectifier_f32_forward: bad argument");
    hipLaunchKernelGGL(rectifier_f32_forward_kernel, dim3(grid_for(n)), dim3(TBLOCK), 0, (hipStream_t)stream, x, n, leak_slope, clipping);
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

int n2d2hip_rectifier_f32_backward(const float* output, const float* diff_in, float* diff_out, size_t n, float leak_slope, float clipping,
                                   n2d2hip_stream_t stream)
{
    N2D2HIP_REQUIRE(output && diff_in && diff_out && n > 0 && clipping >= 0.0f, N2D2HIP_ERR_INVALID, "n2d2hip_rectifier_f32_backward: bad argument");
    hipLaunchKernelGGL(rectifier_f32_backward_kernel, dim3(grid_for(n)), dim3(TBLOCK), 0, (hipStream_t)stream, output, diff_in, diff_out, n,
                       leak_slope, clipping);
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

// Planes below 64 values (a channel's values of one image are less than a cache line or two) are written value by value, others
// channel by channel, with the sums' end
constexpr int BN_WALK_PLANE = 64;
// Blocks per channel for the sums over batch and pixels: one below 8192 values; then about 1024 blocks in all, at most 64, of at
// least 1024 values each, or 4096 where their end is a launch of its own.
static int bn_splits(int B, int C, int H, int W)
{
    const size_t n = (size_t)B * H * W;
    const size_t by_size = n < 8192 ? 1 : n / ((size_t)H * W >= BN_WALK_PLANE ? 1024 : 4096);
    const size_t by_grid = (size_t)std::max(1024 / C, 1);
    return (int)std::max<size_t>(1, std::min<size_t>(std::min(by_size, by_grid), 64));
}

// Units of 16 bytes where the planes allow it.  One block a channel: 1024 threads where 256 would go round more than four times, and
// 512 where they would more than twice and the channels leave every block a compute unit of its own.  us, forward / backward /
// backward with the quantizer's gradient, 513 to 1024 units: 16 channels with 256 threads 7.4 / 8.5 / 11.0, 512 7.1 / 7.9 / 9.7, 1024
// 8.3 / 10.4 / 12.3; 256 channels 8.1 / 9.5 / 12.1, 7.8 / 8.9 / 10.8, 9.0 / 11.4 / 13.5; 512 channels 9.0 / 11.0 / 14.6, 9.8 / 12.1 /
// 14.9, 12.7 / 17.3 / 21.6; 2048 channels 16.7 / 24.2 / 32.3, 21.3 / 31.1 / 39.2, 34.7 / 53.3 / 67.6.
struct BnLaunch {
    BnRange q;
    int V, block;
};
static BnLaunch bn_launch(int B, int C, int plane, int splits, uintptr_t pointers)
{
    BnLaunch l;
    const size_t n = (size_t)B * plane;
    l.V = plane % 4 == 0 && pointers % 16 == 0 ? 4 : 1;
    if (n / l.V >= ((size_t)1 << 30)) l.V = 0;
    const int v = l.V ? l.V : 1;
    l.q = {C, plane, plane / v, div_of(plane / v), n / v, (n / v + splits - 1) / splits};
    l.block = splits > 1 || l.q.units <= 2 * TBLOCK ? TBLOCK : l.q.units > 4 * TBLOCK ? 1024 : C <= num_cus() ? 512 : TBLOCK;
    return l;
}

size_t n2d2hip_batchnorm_f32_workspace_bytes(int B, int C, int H, int W)
{
    if (B <= 0 || C <= 0 || H <= 0 || W <= 0)
        return 0;
    return (size_t)C * bn_splits(B, C, H, W) * 5 * sizeof(double);
}

// Blocks a channel for the passes that write a tensor: about 2048 in all, none for less than a value or quad a thread
static int bn_ranges(int B, int C, int plane, int V)
{
    const size_t blocks = ((size_t)B * plane / std::max(V, 1) + TBLOCK - 1) / TBLOCK;
    return (int)std::min<size_t>(std::max(2048 / C, 1), blocks);
}

// Whether one block takes each channel, statistics and normalisation in one launch.  The second launch, and the statistics on their way
// to it, take longer than what one block has to do while a channel is short, or while there are blocks for every compute unit; until the tensors
// (three with a quantizer) outgrow the 256 MB of the last cache, where the many blocks of two launches keep the memory busier.  Single values
// and pieces of a few a plane it would write line by line with other blocks: only where they are few in all.  us, two launches / one,
// batch x channels x plane: 32 x 16 x 10^2 6.8 / 5.1, 33 x 256 x 14^2 10.1 / 7.8, 128 x 512 x 7^2 22.3 / 14.9, 64 x 512 x 14^2 22.0 / 17.1,
// 32 x 512 x 28^2 29.2 / 25.6, with the quantizer 38.7 / 34.3, 256 x 2048 x 7^2 with it 114 / 126; 256 x 512 x 1 7.2 / 6.1, 256 x 2048 x 1 11.1 / 11.6.
// Backwards (three tensors): 32 x 16 x 10^2 6.5 / 4.7, 33 x 256 x 14^2 10.7 / 8.1, 128 x 512 x 7^2 27.5 / 17.9, 64 x 512 x 14^2 27.9 / 22.3, 32 x 512 x 28^2
// 43.5 / 37.9.  (Behind a SAT quantizer alpha's gradient waits for every channel, so those stay two launches.)
static bool bn_whole(int B, int C, int plane, int tensors)
{
    const size_t n = (size_t)B * plane;
    return (n < 8192 || (C >= num_cus() && n < 65536)) && n * C * tensors <= ((size_t)64 << 20) && (plane >= 16 || n * C <= 128 * 1024);
}

// Windows that tile planes of even sides, from and to memory that the loads of `columns` allow: 4 or 2, 0: neither
static int bn_pool_columns(int B, int H, int W, uintptr_t pointers)
{
    if (H % 2 || W % 2 || (size_t)B * H * W >= ((size_t)1 << 31)) return 0;
    return W % 4 == 0 && pointers % 16 == 0 ? 4 : pointers % 8 == 0 ? 2 : 0;
}
static BnPool bn_pool(int B, int C, int H, int W, int columns, int blocks, float* y, int* argmax)
{
    BnPool p;
    const int row = W / columns, plane = H / 2 * row;
    p.units = {C, H * W, plane, div_of(plane), (size_t)B * plane, ((size_t)B * plane + blocks - 1) / blocks};
    p.W = W; p.row_units = row; p.drow = div_of(row); p.y = y; p.argmax = argmax;
    return p;
}

static int batchnorm_forward(const char* who, int B, int C, int H, int W, const float* x, const float* scale, const float* bias, float* mean, float* variance,
                             float* saved_mean, float* saved_variance, double epsilon, double moving_average_momentum, int use_running, float* y,
                             const SatStore& sat, void* workspace, size_t workspace_bytes, hipStream_t stream, int columns = 0, float* pooled = nullptr,
                             int* argmax = nullptr)
{
    N2D2HIP_REQUIRE(B > 0 && C > 0 && H > 0 && W > 0 && x && scale && bias && mean && variance && y && epsilon > 0.0, N2D2HIP_ERR_INVALID,
                    "%s: bad argument", who);
    N2D2HIP_REQUIRE((size_t)B * C < ((size_t)1 << 31) && (size_t)H * W < ((size_t)1 << 31), N2D2HIP_ERR_INVALID, "%s: tensor too large", who);
    const bool running = use_running || moving_average_momentum == 0.0;
    const double n = (double)B * H * W;
    const int plane = H * W;
    const int V = bn_launch(B, C, plane, 1, (uintptr_t)x | (uintptr_t)y | (uintptr_t)sat.fp).V;
    const bool walk = plane >= BN_WALK_PLANE && V != 0;
    int splits = 1;
    if (!running) {
        N2D2HIP_REQUIRE(saved_mean && saved_variance, N2D2HIP_ERR_INVALID, "%s: the learning pass needs saved_mean and saved_variance", who);
        N2D2HIP_REQUIRE((size_t)B * H * W > 1, N2D2HIP_ERR_INVALID, "%s: batch statistics need more than one value per channel", who);
        splits = workspace && workspace_bytes >= n2d2hip_batchnorm_f32_workspace_bytes(B, C, H, W) ? bn_splits(B, C, H, W) : 1;
        const bool whole = bn_whole(B, C, plane, sat.fp ? 3 : 2);
        if (whole) splits = 1;
        const BnLaunch l = bn_launch(B, C, plane, splits, (uintptr_t)x | (whole ? (uintptr_t)y | (uintptr_t)sat.fp : 0));
        const auto stats = [&](auto W, auto then) {
            N2D2HIP_LAUNCH_T(batchnorm_f32_stats_kernel, (decltype(W)::value, decltype(then)::value), dim3(C, splits), dim3(l.block), 0, stream, l.q, n, x,
                             (double*)workspace, mean, variance, saved_mean, saved_variance, moving_average_momentum, scale, bias, epsilon, sat, y,
                             columns ? bn_pool(B, C, H, plane / H, columns, 1, pooled, argmax) : BnPool{});
        };
        const auto then = [&](auto W) {
            if (!whole) stats(W, std::integral_constant<int, BN_SUMS_ONLY>{});
            else if (columns == 4) stats(W, std::integral_constant<int, BN_APPLY_SAT_POOL + 4>{});
            else if (columns == 2) stats(W, std::integral_constant<int, BN_APPLY_SAT_POOL + 2>{});
            else if (sat.alpha) stats(W, std::integral_constant<int, BN_APPLY_SAT>{});
            else stats(W, std::integral_constant<int, BN_APPLY>{});
        };
        if (l.V == 4) then(std::integral_constant<int, 4>{});
        else if (l.V == 1) then(std::integral_constant<int, 1>{});
        else stats(std::integral_constant<int, 0>{}, std::integral_constant<int, BN_SUMS_ONLY>{});       // (2^30 values a channel: never whole)
        if (whole) {
            N2D2HIP_HIP_CHECK(hipGetLastError());
            return N2D2HIP_OK;
        }
        if (splits > 1 && !walk)
            hipLaunchKernelGGL(batchnorm_f32_stats_finish_kernel, dim3(C), dim3(64), 0, stream, n, splits, (const double*)workspace, mean, variance,
                               saved_mean, saved_variance, moving_average_momentum);
    }
    if (walk) {
        const int ranges = bn_ranges(B, C, plane, V);
        const BnLaunch l = bn_launch(B, C, plane, ranges, (uintptr_t)x | (uintptr_t)y | (uintptr_t)sat.fp);
        const auto kernel = columns == 4 ? batchnorm_f32_apply_kernel<1, true, 4> : columns == 2 ? batchnorm_f32_apply_kernel<1, true, 2>
                            : V == 4 ? (sat.alpha ? batchnorm_f32_apply_kernel<4, true> : batchnorm_f32_apply_kernel<4, false>)
                                     : (sat.alpha ? batchnorm_f32_apply_kernel<1, true> : batchnorm_f32_apply_kernel<1, false>);
        hipLaunchKernelGGL(kernel, dim3(C, ranges), dim3(TBLOCK), 0, stream, l.q, splits, n, (const double*)workspace, mean, variance, saved_mean,
                           saved_variance, moving_average_momentum, running ? 1 : 0, x, scale, bias, epsilon, sat, y,
                           columns ? bn_pool(B, C, H, W, columns, ranges, pooled, argmax) : BnPool{});
    } else {
        hipLaunchKernelGGL(batchnorm_f32_apply_flat_kernel, dim3(grid_for((size_t)B * C * plane)), dim3(TBLOCK), 0, stream, (size_t)B * C * plane, C, plane, x,
                           scale, bias, running ? (const float*)mean : (const float*)saved_mean, running ? (const float*)variance : (const float*)saved_variance,
                           epsilon, running ? 1 : 0, sat, y);
    }
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

int n2d2hip_batchnorm_f32_forward(int B, int C, int H, int W, const float* x, const float* scale, const float* bias, float* mean,
                                  float* variance, float* saved_mean, float* saved_variance, double epsilon, double moving_average_momentum,
                                  int use_running, float* y, void* workspace, size_t workspace_bytes, n2d2hip_stream_t stream)
{
    return batchnorm_forward("n2d2hip_batchnorm_f32_forward", B, C, H, W, x, scale, bias, mean, variance, saved_mean, saved_variance, epsilon,
                             moving_average_momentum, use_running, y, SatStore{nullptr, 0.0f, nullptr}, workspace, workspace_bytes, (hipStream_t)stream);
}

int n2d2hip_batchnorm_f32_forward_sat(int B, int C, int H, int W, const float* x, const float* scale, const float* bias, float* mean,
                                      float* variance, float* saved_mean, float* saved_variance, double epsilon, double moving_average_momentum,
                                      int use_running, float* y, float* full_precision, float range, const float* alpha, void* workspace,
                                      size_t workspace_bytes, n2d2hip_stream_t stream)
{
    N2D2HIP_REQUIRE(alpha && range >= 1.0f && full_precision != y, N2D2HIP_ERR_INVALID, "n2d2hip_batchnorm_f32_forward_sat: bad argument");
    return batchnorm_forward("n2d2hip_batchnorm_f32_forward_sat", B, C, H, W, x, scale, bias, mean, variance, saved_mean, saved_variance, epsilon,
                             moving_average_momentum, use_running, y, SatStore{full_precision, range, alpha}, workspace, workspace_bytes, (hipStream_t)stream);
}

int n2d2hip_batchnorm_f32_forward_sat_pool(int B, int C, int H, int W, const float* x, const float* scale, const float* bias, float* mean,
                                           float* variance, float* saved_mean, float* saved_variance, double epsilon, double moving_average_momentum,
                                           int use_running, float* y, float* full_precision, float range, const float* alpha, float* pooled, int* argmax,
                                           void* workspace, size_t workspace_bytes, n2d2hip_stream_t stream)
{
    const char* who = "n2d2hip_batchnorm_f32_forward_sat_pool";
    N2D2HIP_REQUIRE(alpha && range >= 1.0f && full_precision != y && pooled && argmax, N2D2HIP_ERR_INVALID, "%s: bad argument", who);
    N2D2HIP_REQUIRE(B > 0 && C > 0 && H > 1 && W > 1 && H % 2 == 0 && W % 2 == 0, N2D2HIP_ERR_INVALID, "%s: planes of whole 2x2 windows expected", who);
    const uintptr_t pointers = (uintptr_t)x | (uintptr_t)y | (uintptr_t)full_precision;
    const int V = bn_launch(B, C, H * W, 1, pointers).V, columns = bn_pool_columns(B, H, W, pointers);
    // (in one pass where the values are written channel by channel)
    const bool learns = !use_running && moving_average_momentum != 0.0;
    if (columns && V != 0 && (H * W >= BN_WALK_PLANE || (learns && bn_whole(B, C, H * W, full_precision ? 3 : 2))))
        return batchnorm_forward(who, B, C, H, W, x, scale, bias, mean, variance, saved_mean, saved_variance, epsilon, moving_average_momentum, use_running, y,
                                 SatStore{full_precision, range, alpha}, workspace, workspace_bytes, (hipStream_t)stream, columns, pooled, argmax);
    const int rc = n2d2hip_batchnorm_f32_forward_sat(B, C, H, W, x, scale, bias, mean, variance, saved_mean, saved_variance, epsilon, moving_average_momentum,
                                                     use_running, y, full_precision, range, alpha, workspace, workspace_bytes, stream);
    return rc == N2D2HIP_OK ? n2d2hip_pool_max_f32_forward(B, C, H, W, 2, 2, 2, 2, 0, 0, y, pooled, argmax, stream) : rc;
}

size_t n2d2hip_batchnorm_f32_backward_sat_workspace_bytes(int B, int C, int H, int W)
{
    if (B <= 0 || C <= 0 || H <= 0 || W <= 0)
        return 0;
    return (size_t)C * bn_splits(B, C, H, W) * 6 * sizeof(double);
}

static int batchnorm_backward(const char* who, int B, int C, int H, int W, const float* x, const float* scale, const float* saved_mean,
                              const float* saved_variance, double epsilon, BnSatGrad sat, float* diff_y, const BnGrads& grads, float* diff_x,
                              void* workspace, int splits, hipStream_t stream, int columns = 0, const float* diff_pooled = nullptr,
                              const int* argmax = nullptr)
{
    N2D2HIP_REQUIRE(B > 0 && C > 0 && H > 0 && W > 0 && x && scale && saved_mean && saved_variance && diff_y && grads.diff_scale && grads.diff_bias
                        && grads.diff_saved_mean && grads.diff_saved_variance && epsilon > 0.0,
                    N2D2HIP_ERR_INVALID, "%s: bad argument", who);
    N2D2HIP_REQUIRE((size_t)B * C < ((size_t)1 << 31) && (size_t)H * W < ((size_t)1 << 31), N2D2HIP_ERR_INVALID, "%s: tensor too large", who);
    const double n = (double)B * H * W;
    const int plane = H * W;
    const uintptr_t in = (uintptr_t)x | (uintptr_t)diff_y;
    if (!sat.alpha && diff_x && bn_whole(B, C, plane, 3)) {
        const BnLaunch w = bn_launch(B, C, plane, 1, in | (uintptr_t)diff_x);
        hipLaunchKernelGGL(w.V == 4 ? batchnorm_f32_backward_whole_kernel<4> : batchnorm_f32_backward_whole_kernel<1>, dim3(C), dim3(w.block), 0, stream, w.q,
                           n, (float)((size_t)B * H * W), x, scale, saved_mean, saved_variance, epsilon, (const float*)diff_y, grads, diff_x);
        N2D2HIP_HIP_CHECK(hipGetLastError());
        return N2D2HIP_OK;
    }
    const BnLaunch l = bn_launch(B, C, plane, splits, in | (uintptr_t)sat.fp);
    sat.partial = (double*)workspace + (size_t)C * splits * BN_SUMS;
    sat.blocks = C * splits;
    const auto kernel = columns == 4 ? batchnorm_f32_backward_sums_kernel<1, true, 4> : columns == 2 ? batchnorm_f32_backward_sums_kernel<1, true, 2>
                        : sat.alpha ? (l.V == 4 ? batchnorm_f32_backward_sums_kernel<4, true> : l.V == 1 ? batchnorm_f32_backward_sums_kernel<1, true>
                                                                                                : batchnorm_f32_backward_sums_kernel<0, true>)
                                  : (l.V == 4 ? batchnorm_f32_backward_sums_kernel<4, false> : l.V == 1 ? batchnorm_f32_backward_sums_kernel<1, false>
                                                                                                 : batchnorm_f32_backward_sums_kernel<0, false>);
    hipLaunchKernelGGL(kernel, dim3(C, splits), dim3(l.block), 0, stream, l.q, n, x, scale, saved_mean, saved_variance, epsilon, diff_y, (double*)workspace,
                       grads, sat, columns ? bn_pool(B, C, H, W, columns, splits, const_cast<float*>(diff_pooled), const_cast<int*>(argmax)) : BnPool{});
    const int V = bn_launch(B, C, plane, 1, in | (uintptr_t)diff_x).V;
    const bool walk = diff_x && plane >= BN_WALK_PLANE && V != 0;
    if (splits > 1 && !walk)
        hipLaunchKernelGGL(batchnorm_f32_backward_finish_kernel, dim3(C), dim3(64), 0, stream, n, splits, (const double*)workspace, scale, saved_variance, epsilon,
                           grads);
    if (walk) {
        const int ranges = bn_ranges(B, C, plane, V);
        const BnLaunch d = bn_launch(B, C, plane, ranges, in | (uintptr_t)diff_x);
        hipLaunchKernelGGL(V == 4 ? batchnorm_f32_backward_data_kernel<4> : batchnorm_f32_backward_data_kernel<1>, dim3(C, ranges), dim3(TBLOCK), 0, stream,
                           d.q, splits, n, (const double*)workspace, (float)((size_t)B * H * W), x, scale, saved_mean, saved_variance, epsilon, diff_y, grads,
                           sat, diff_x);
    } else if (diff_x)
        hipLaunchKernelGGL(batchnorm_f32_backward_data_flat_kernel, dim3(grid_for((size_t)B * C * plane)), dim3(TBLOCK), 0, stream, (size_t)B * C * plane, C,
                           plane, (float)((size_t)B * H * W), x, scale, saved_mean, saved_variance, epsilon, diff_y, (const float*)grads.diff_saved_mean,
                           (const float*)grads.diff_saved_variance, sat, diff_x);
    else if (sat.alpha)
        hipLaunchKernelGGL(batchnorm_f32_alpha_kernel, dim3(1), dim3(TBLOCK), 0, stream, sat);
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

int n2d2hip_batchnorm_f32_backward(int B, int C, int H, int W, const float* x, const float* scale, const float* saved_mean,
                                   const float* saved_variance, double epsilon, const float* diff_y, float beta_scale, float* diff_scale,
                                   float beta_bias, float* diff_bias, float* diff_saved_mean, float* diff_saved_variance, float* diff_x,
                                   void* workspace, size_t workspace_bytes, n2d2hip_stream_t stream)
{
    const int splits = B > 0 && C > 0 && H > 0 && W > 0 && workspace && workspace_bytes >= n2d2hip_batchnorm_f32_workspace_bytes(B, C, H, W)
                           ? bn_splits(B, C, H, W) : 1;
    const BnGrads grads = {diff_scale, diff_bias, diff_saved_mean, diff_saved_variance, beta_scale, beta_bias};
    // (without a quantizer diff_y is only read)
    return batchnorm_backward("n2d2hip_batchnorm_f32_backward", B, C, H, W, x, scale, saved_mean, saved_variance, epsilon, BnSatGrad{},
                              const_cast<float*>(diff_y), grads, diff_x, workspace, splits, (hipStream_t)stream);
}

int n2d2hip_batchnorm_f32_backward_sat(int B, int C, int H, int W, const float* x, const float* scale, const float* saved_mean,
                                       const float* saved_variance, double epsilon, const float* full_precision, float range, const float* alpha,
                                       float beta_alpha, float* diff_alpha, float* diff_y, float beta_scale, float* diff_scale, float beta_bias,
                                       float* diff_bias, float* diff_saved_mean, float* diff_saved_variance, float* diff_x, void* workspace,
                                       size_t workspace_bytes, n2d2hip_stream_t stream)
{
    N2D2HIP_REQUIRE(full_precision && alpha && diff_alpha && full_precision != diff_y && full_precision != diff_x, N2D2HIP_ERR_INVALID,
                    "n2d2hip_batchnorm_f32_backward_sat: bad argument");
    const size_t need = n2d2hip_batchnorm_f32_backward_sat_workspace_bytes(B, C, H, W);
    N2D2HIP_REQUIRE(workspace && workspace_bytes >= need, N2D2HIP_ERR_WORKSPACE, "n2d2hip_batchnorm_f32_backward_sat: workspace of %zu bytes needed", need);
    const BnGrads grads = {diff_scale, diff_bias, diff_saved_mean, diff_saved_variance, beta_scale, beta_bias};
    return batchnorm_backward("n2d2hip_batchnorm_f32_backward_sat", B, C, H, W, x, scale, saved_mean, saved_variance, epsilon,
                              BnSatGrad{full_precision, range, alpha, nullptr, 0, beta_alpha, diff_alpha}, diff_y, grads, diff_x, workspace,
                              need ? bn_splits(B, C, H, W) : 1, (hipStream_t)stream);
}

int n2d2hip_batchnorm_f32_backward_sat_pool(int B, int C, int H, int W, const float* x, const float* scale, const float* saved_mean,
                                            const float* saved_variance, double epsilon, const float* full_precision, float range, const float* alpha,
                                            float beta_alpha, float* diff_alpha, const float* diff_pooled, const int* argmax, float* diff_y, float beta_scale,
                                            float* diff_scale, float beta_bias, float* diff_bias, float* diff_saved_mean, float* diff_saved_variance,
                                            float* diff_x, void* workspace, size_t workspace_bytes, n2d2hip_stream_t stream)
{
    const char* who = "n2d2hip_batchnorm_f32_backward_sat_pool";
    N2D2HIP_REQUIRE(full_precision && alpha && diff_alpha && full_precision != diff_y && full_precision != diff_x && diff_pooled && argmax && diff_y,
                    N2D2HIP_ERR_INVALID, "%s: bad argument", who);
    N2D2HIP_REQUIRE(B > 0 && C > 0 && H > 1 && W > 1 && H % 2 == 0 && W % 2 == 0, N2D2HIP_ERR_INVALID, "%s: planes of whole 2x2 windows expected", who);
    const size_t need = n2d2hip_batchnorm_f32_backward_sat_workspace_bytes(B, C, H, W);
    N2D2HIP_REQUIRE(workspace && workspace_bytes >= need, N2D2HIP_ERR_WORKSPACE, "%s: workspace of %zu bytes needed", who, need);
    const int columns = bn_pool_columns(B, H, W, (uintptr_t)x | (uintptr_t)full_precision | (uintptr_t)diff_y);
    if (!columns) {
        const int rc = n2d2hip_pool_max_f32_backward(B, C, H, W, 2, 2, 2, 2, 0, 0, diff_pooled, argmax, 0.0f, diff_y, stream);
        return rc == N2D2HIP_OK ? n2d2hip_batchnorm_f32_backward_sat(B, C, H, W, x, scale, saved_mean, saved_variance, epsilon, full_precision, range, alpha,
                                                                     beta_alpha, diff_alpha, diff_y, beta_scale, diff_scale, beta_bias, diff_bias,
                                                                     diff_saved_mean, diff_saved_variance, diff_x, workspace, workspace_bytes, stream) : rc;
    }
    const BnGrads grads = {diff_scale, diff_bias, diff_saved_mean, diff_saved_variance, beta_scale, beta_bias};
    return batchnorm_backward(who, B, C, H, W, x, scale, saved_mean, saved_variance, epsilon,
                              BnSatGrad{full_precision, range, alpha, nullptr, 0, beta_alpha, diff_alpha}, diff_y, grads, diff_x, workspace,
                              bn_splits(B, C, H, W), (hipStream_t)stream, columns, diff_pooled, argmax);
}

static bool pool_small(const PoolF32& q) { return (size_t)q.B * q.C * std::max((size_t)q.H * q.W, (size_t)q.oH * q.oW) < ((size_t)1 << 31) - TBLOCK; }
static int make_pool(int B, int C, int H, int W, int pool_w, int pool_h, int stride_x, int stride_y, int pad_x, int pad_y, PoolF32* q, const char* who)
{
    N2D2HIP_REQUIRE(B > 0 && C > 0 && H > 0 && W > 0 && pool_w > 0 && pool_h > 0 && stride_x > 0 && stride_y > 0 && pad_x >= 0 && pad_y >= 0,
                    N2D2HIP_ERR_INVALID, "%s: bad argument", who);
    N2D2HIP_REQUIRE(pad_x < pool_w && pad_y < pool_h, N2D2HIP_ERR_INVALID, "%s: padding must be smaller than the window", who);
    q->B = B; q->C = C; q->H = H; q->W = W;
    q->pw = pool_w; q->ph = pool_h; q->sx = stride_x; q->sy = stride_y; q->px = pad_x; q->py = pad_y;
    // PoolCell::setOutputsDims (src/Cell/PoolCell.cpp:219-240)
    q->oW = (int)((W + 2 * pad_x - pool_w + stride_x) / (double)stride_x);
    q->oH = (int)((H + 2 * pad_y - pool_h + stride_y) / (double)stride_y);
    N2D2HIP_REQUIRE(q->oW > 0 && q->oH > 0, N2D2HIP_ERR_INVALID, "%s: the window does not fit the input", who);
    q->dw = div_of(W); q->dh = div_of(H); q->dow = div_of(q->oW); q->doh = div_of(q->oH); q->dsx = div_of(stride_x); q->dsy = div_of(stride_y);
    N2D2HIP_REQUIRE((size_t)H * W < ((size_t)1 << 31) && (size_t)B * C * H * W < ((size_t)1 << 40), N2D2HIP_ERR_INVALID, "%s: tensor too large", who);
    return N2D2HIP_OK;
}

int n2d2hip_pool_max_f32_forward(int B, int C, int H, int W, int pool_w, int pool_h, int stride_x, int stride_y, int pad_x, int pad_y,
                                 const float* x, float* y, int* argmax, n2d2hip_stream_t stream)
{
    PoolF32 q;
    const int rc = make_pool(B, C, H, W, pool_w, pool_h, stride_x, stride_y, pad_x, pad_y, &q, "n2d2hip_pool_max_f32_forward");
    if (rc != N2D2HIP_OK) return rc;
    N2D2HIP_REQUIRE(x && y && argmax, N2D2HIP_ERR_INVALID, "n2d2hip_pool_max_f32_forward: null pointer");
    hipLaunchKernelGGL(pool_small(q) ? pool_max_f32_forward_kernel<true> : pool_max_f32_forward_kernel<false>, dim3(grid_for((size_t)B * C * q.oH * q.oW)), dim3(TBLOCK), 0, (hipStream_t)stream, q, x, y, argmax);
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

int n2d2hip_pool_max_f32_backward(int B, int C, int H, int W, int pool_w, int pool_h, int stride_x, int stride_y, int pad_x, int pad_y,
                                  const float* diff_y, const int* argmax, float beta, float* diff_x, n2d2hip_stream_t stream)
{
    PoolF32 q;
    const int rc = make_pool(B, C, H, W, pool_w, pool_h, stride_x, stride_y, pad_x, pad_y, &q, "n2d2hip_pool_max_f32_backward");
    if (rc != N2D2HIP_OK) return rc;
    N2D2HIP_REQUIRE(diff_y && argmax && diff_x, N2D2HIP_ERR_INVALID, "n2d2hip_pool_max_f32_backward: null pointer");
    if (pool_small(q) && W % 4 == 0 && ((size_t)diff_x & 15) == 0) {
        hipLaunchKernelGGL(pool_max_f32_backward_quads_kernel, dim3(grid_for((size_t)B * C * H * W / 4)), dim3(TBLOCK), 0, (hipStream_t)stream, q, div_of(W / 4), diff_y,
                           argmax, beta, diff_x);
        N2D2HIP_HIP_CHECK(hipGetLastError());
        return N2D2HIP_OK;
    }
    hipLaunchKernelGGL(pool_small(q) ? pool_max_f32_backward_kernel<true> : pool_max_f32_backward_kernel<false>, dim3(grid_for((size_t)B * C * H * W)),
                       dim3(TBLOCK), 0, (hipStream_t)stream, q, diff_y, argmax, beta, diff_x);
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

}  // extern "C"

// Average pooling of float NCHW with the unit mapping: the window's values are added in row-major order and divided
// by the window's size (count_include_padding) or by the number of values inside the input.
__global__ __launch_bounds__(TBLOCK) void pool_average_f32_forward_kernel(PoolF32 q, int count_include_padding, const float* __restrict__ x,
                                                                          float* __restrict__ y)
{
    const size_t total = (size_t)q.B * q.C * q.oH * q.oW;
    for (size_t i = (size_t)blockIdx.x * TBLOCK + threadIdx.x; i < total; i += (size_t)gridDim.x * TBLOCK) {
        const int ox = (int)(i % q.oW), oy = (int)((i / q.oW) % q.oH);
        const size_t bc = i / ((size_t)q.oW * q.oH);
        const float* in = x + bc * (size_t)q.H * q.W;
        const int x0 = ox * q.sx - q.px, y0 = oy * q.sy - q.py;
        const int sx_min = max(-x0, 0), sy_min = max(-y0, 0);
        const int sx_max = min(max(q.W - x0, 0), q.pw), sy_max = min(max(q.H - y0, 0), q.ph);
        float acc = 0.0f;
        for (int sy = sy_min; sy < sy_max; ++sy)
            for (int sx = sx_min; sx < sx_max; ++sx)
                acc += in[(size_t)(y0 + sy) * q.W + x0 + sx];
        const int inside = max(sx_max - sx_min, 0) * max(sy_max - sy_min, 0);
        const unsigned count = count_include_padding ? (unsigned)(q.pw * q.ph) : (unsigned)inside;
        y[i] = count > 0 ? acc / (float)count : 0.0f;
    }
}

// Every input collects the gradients of the windows it lies in, in the reference's order (window rows, then columns,
// from the input's own residue modulo the stride upwards); the sum is divided by the window's size.
__global__ __launch_bounds__(TBLOCK) void pool_average_f32_backward_kernel(PoolF32 q, const float* __restrict__ dy, float beta, float* __restrict__ dx)
{
    const size_t total = (size_t)q.B * q.C * q.H * q.W;
    const float count = (float)(unsigned)(q.pw * q.ph);
    for (size_t i = (size_t)blockIdx.x * TBLOCK + threadIdx.x; i < total; i += (size_t)gridDim.x * TBLOCK) {
        const int ix = (int)(i % q.W), iy = (int)((i / q.W) % q.H);
        const size_t bc = i / ((size_t)q.W * q.H);
        const int ix_pad = ix + q.px, iy_pad = iy + q.py;
        const int sx_max = min(q.pw, ix_pad + 1), sy_max = min(q.ph, iy_pad + 1);
        float acc = 0.0f;
        for (int sy = iy_pad % q.sy; sy < sy_max; sy += q.sy) {
            if (iy_pad >= q.sy * q.oH + sy)
                continue;
            const int oy = (iy_pad - sy) / q.sy;
            for (int sx = ix_pad % q.sx; sx < sx_max; sx += q.sx) {
                if (ix_pad >= q.sx * q.oW + sx)
                    continue;
                const int ox = (ix_pad - sx) / q.sx;
                acc += dy[(bc * q.oH + oy) * q.oW + ox];
            }
        }
        const float g = acc / count;
        dx[i] = beta != 0.0f ? __fadd_rn(g, __fmul_rn(beta, dx[i])) : g;
    }
}

extern "C" {

int n2d2hip_pool_average_f32_forward(int B, int C, int H, int W, int pool_w, int pool_h, int stride_x, int stride_y, int pad_x, int pad_y,
                                     int count_include_padding, const float* x, float* y, n2d2hip_stream_t stream)
{
    PoolF32 q;
    const int rc = make_pool(B, C, H, W, pool_w, pool_h, stride_x, stride_y, pad_x, pad_y, &q, "n2d2hip_pool_average_f32_forward");
    if (rc != N2D2HIP_OK) return rc;
    N2D2HIP_REQUIRE(x && y, N2D2HIP_ERR_INVALID, "n2d2hip_pool_average_f32_forward: null pointer");
    hipLaunchKernelGGL(pool_average_f32_forward_kernel, dim3(grid_for((size_t)B * C * q.oH * q.oW)), dim3(TBLOCK), 0, (hipStream_t)stream, q,
                       count_include_padding ? 1 : 0, x, y);
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

int n2d2hip_pool_average_f32_backward(int B, int C, int H, int W, int pool_w, int pool_h, int stride_x, int stride_y, int pad_x, int pad_y,
                                      int count_include_padding, const float* diff_y, float beta, float* diff_x, n2d2hip_stream_t stream)
{
    PoolF32 q;
    const int rc = make_pool(B, C, H, W, pool_w, pool_h, stride_x, stride_y, pad_x, pad_y, &q, "n2d2hip_pool_average_f32_backward");
    if (rc != N2D2HIP_OK) return rc;
    // the reference throws for the other case (src/Cell/PoolCell_Frame_Kernels.cpp:210-213)
    N2D2HIP_REQUIRE(count_include_padding, N2D2HIP_ERR_UNSUPPORTED, "n2d2hip_pool_average_f32_backward: exclude padding not implemented");
    N2D2HIP_REQUIRE(diff_y && diff_x, N2D2HIP_ERR_INVALID, "n2d2hip_pool_average_f32_backward: null pointer");
    hipLaunchKernelGGL(pool_average_f32_backward_kernel, dim3(grid_for((size_t)B * C * H * W)), dim3(TBLOCK), 0, (hipStream_t)stream, q, diff_y, beta,
                       diff_x);
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

}  // extern "C"

// Weighted sum of up to N2D2HIP_ELEMWISE_F32_MAX_INPUTS float tensors of one shape: products and sums are rounded one
// by one, in the order of the inputs, as the reference's scalar loop does.
struct ElemWiseF32 {
    const float* x[N2D2HIP_ELEMWISE_F32_MAX_INPUTS];
    float w[N2D2HIP_ELEMWISE_F32_MAX_INPUTS], s[N2D2HIP_ELEMWISE_F32_MAX_INPUTS];
    int n;
};

__device__ __forceinline__ float elemwise_sum_one(const ElemWiseF32& e, const float* v)
{
    float acc = __fadd_rn(__fmul_rn(e.w[0], v[0]), e.s[0]);
#pragma unroll
    for (int k = 1; k < N2D2HIP_ELEMWISE_F32_MAX_INPUTS; ++k)
        if (k < e.n)
            acc = __fadd_rn(acc, __fadd_rn(__fmul_rn(e.w[k], v[k]), e.s[k]));
    return acc;
}

// Memory bounds it.  SAT: the quantizer that follows the sum in a learning net is applied on the way out; its own pass read and wrote the
// tensor again (64 x 64 x 32 x 32, two inputs, us: sum and quantizer 10.4 + 11.9, now 15.0).
template <int VEC, bool SAT>
__global__ __launch_bounds__(TBLOCK) void elemwise_sum_f32_forward_kernel(ElemWiseF32 e, size_t total, SatStore sat, float* __restrict__ y)
{
    const float alpha = SAT ? fabsf(sat.alpha[0]) : 0.0f;
    for (size_t i = (size_t)blockIdx.x * TBLOCK + threadIdx.x; i < total / VEC; i += (size_t)gridDim.x * TBLOCK) {
        if (VEC == 4) {
            float4 v[N2D2HIP_ELEMWISE_F32_MAX_INPUTS];
#pragma unroll
            for (int k = 0; k < N2D2HIP_ELEMWISE_F32_MAX_INPUTS; ++k)
                if (k < e.n)
                    v[k] = ((const float4*)e.x[k])[i];
            float a[N2D2HIP_ELEMWISE_F32_MAX_INPUTS], b[N2D2HIP_ELEMWISE_F32_MAX_INPUTS], c[N2D2HIP_ELEMWISE_F32_MAX_INPUTS],
                d[N2D2HIP_ELEMWISE_F32_MAX_INPUTS];
#pragma unroll
            for (int k = 0; k < N2D2HIP_ELEMWISE_F32_MAX_INPUTS; ++k)
                if (k < e.n) {
                    a[k] = v[k].x; b[k] = v[k].y; c[k] = v[k].z; d[k] = v[k].w;
                }
            float4 o;
            o.x = elemwise_sum_one(e, a);
            o.y = elemwise_sum_one(e, b);
            o.z = elemwise_sum_one(e, c);
            o.w = elemwise_sum_one(e, d);
            if (SAT) {
                if (sat.fp) ((float4*)sat.fp)[i] = o;
                o = make_float4(sat_quantize(o.x, sat.range, alpha), sat_quantize(o.y, sat.range, alpha), sat_quantize(o.z, sat.range, alpha),
                                sat_quantize(o.w, sat.range, alpha));
            }
            ((float4*)y)[i] = o;
        } else {
            float a[N2D2HIP_ELEMWISE_F32_MAX_INPUTS];
#pragma unroll
            for (int k = 0; k < N2D2HIP_ELEMWISE_F32_MAX_INPUTS; ++k)
                if (k < e.n)
                    a[k] = e.x[k][i];
            float o = elemwise_sum_one(e, a);
            if (SAT) {
                if (sat.fp) sat.fp[i] = o;
                o = sat_quantize(o, sat.range, alpha);
            }
            y[i] = o;
        }
    }
}

// diff_x = weight * diff_y + beta * diff_x
template <int VEC>
__global__ __launch_bounds__(TBLOCK) void elemwise_sum_f32_backward_kernel(size_t total, float weight, const float* __restrict__ dy, float beta, float* dx)
{
    for (size_t i = (size_t)blockIdx.x * TBLOCK + threadIdx.x; i < total / VEC; i += (size_t)gridDim.x * TBLOCK) {
        if (VEC == 4) {
            const float4 d = ((const float4*)dy)[i];
            float4 o = make_float4(__fmul_rn(weight, d.x), __fmul_rn(weight, d.y), __fmul_rn(weight, d.z), __fmul_rn(weight, d.w));
            if (beta != 0.0f) {
                const float4 p = ((const float4*)dx)[i];
                o.x = __fadd_rn(o.x, __fmul_rn(beta, p.x));
                o.y = __fadd_rn(o.y, __fmul_rn(beta, p.y));
                o.z = __fadd_rn(o.z, __fmul_rn(beta, p.z));
                o.w = __fadd_rn(o.w, __fmul_rn(beta, p.w));
            }
            ((float4*)dx)[i] = o;
        } else {
            const float g = __fmul_rn(weight, dy[i]);
            dx[i] = beta != 0.0f ? __fadd_rn(g, __fmul_rn(beta, dx[i])) : g;
        }
    }
}

template <int N>
static SgdBatch<N> sgd_batch(const n2d2hip_sgd_item* item, int count)
{
    SgdBatch<N> b = {};
    b.count = count;
    for (int i = 0; i < count; ++i) {
        b.item[i] = item[i];
        b.first[i + 1] = b.first[i] + (unsigned)grid_for(item[i].n);
    }
    return b;
}

extern "C" {

static int elemwise_sum_forward(const char* who, int nb_inputs, const float* const* inputs, size_t n, const float* weights, const float* shifts, float* y,
                                const SatStore& sat, n2d2hip_stream_t stream)
{
    N2D2HIP_REQUIRE(nb_inputs > 0 && inputs && weights && shifts && y && n > 0, N2D2HIP_ERR_INVALID, "%s: bad argument", who);
    N2D2HIP_REQUIRE(nb_inputs <= N2D2HIP_ELEMWISE_F32_MAX_INPUTS, N2D2HIP_ERR_UNSUPPORTED, "%s: at most %d inputs", who, N2D2HIP_ELEMWISE_F32_MAX_INPUTS);
    ElemWiseF32 e = {};
    e.n = nb_inputs;
    uintptr_t align = (uintptr_t)y | (uintptr_t)sat.fp;
    for (int k = 0; k < nb_inputs; ++k) {
        N2D2HIP_REQUIRE(inputs[k], N2D2HIP_ERR_INVALID, "%s: input %d is null", who, k);
        e.x[k] = inputs[k];
        e.w[k] = weights[k];
        e.s[k] = shifts[k];
        align |= (uintptr_t)inputs[k];
    }
    const int vec = n % 4 == 0 && align % 16 == 0 ? 4 : 1;
    const auto kernel = vec == 4 ? (sat.alpha ? elemwise_sum_f32_forward_kernel<4, true> : elemwise_sum_f32_forward_kernel<4, false>)
                                 : (sat.alpha ? elemwise_sum_f32_forward_kernel<1, true> : elemwise_sum_f32_forward_kernel<1, false>);
    hipLaunchKernelGGL(kernel, dim3(grid_for(n / vec)), dim3(TBLOCK), 0, (hipStream_t)stream, e, n, sat, y);
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

int n2d2hip_elemwise_sum_f32_forward(int nb_inputs, const float* const* inputs, size_t n, const float* weights, const float* shifts, float* y,
                                     n2d2hip_stream_t stream)
{
    return elemwise_sum_forward("n2d2hip_elemwise_sum_f32_forward", nb_inputs, inputs, n, weights, shifts, y, SatStore{nullptr, 0.0f, nullptr}, stream);
}

int n2d2hip_elemwise_sum_f32_forward_sat(int nb_inputs, const float* const* inputs, size_t n, const float* weights, const float* shifts, float* y,
                                         float* full_precision, float range, const float* alpha, n2d2hip_stream_t stream)
{
    N2D2HIP_REQUIRE(alpha && full_precision != y, N2D2HIP_ERR_INVALID, "n2d2hip_elemwise_sum_f32_forward_sat: bad argument");
    return elemwise_sum_forward("n2d2hip_elemwise_sum_f32_forward_sat", nb_inputs, inputs, n, weights, shifts, y, SatStore{full_precision, range, alpha},
                                stream);
}

int n2d2hip_elemwise_sum_f32_backward(size_t n, float weight, const float* diff_y, float beta, float* diff_x, n2d2hip_stream_t stream)
{
    N2D2HIP_REQUIRE(n > 0 && diff_y && diff_x, N2D2HIP_ERR_INVALID, "n2d2hip_elemwise_sum_f32_backward: bad argument");
    if (n % 4 == 0 && ((uintptr_t)diff_y | (uintptr_t)diff_x) % 16 == 0)
        hipLaunchKernelGGL(elemwise_sum_f32_backward_kernel<4>, dim3(grid_for(n / 4)), dim3(TBLOCK), 0, (hipStream_t)stream, n, weight, diff_y, beta, diff_x);
    else
        hipLaunchKernelGGL(elemwise_sum_f32_backward_kernel<1>, dim3(grid_for(n)), dim3(TBLOCK), 0, (hipStream_t)stream, n, weight, diff_y, beta, diff_x);
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

size_t n2d2hip_loss_workspace_bytes(size_t n)
{
    return (size_t)grid_for(n) * sizeof(double);
}

int n2d2hip_loss_f32(const float* target, const float* output, float* diff, size_t n, int batch, double* loss,
                     void* workspace, size_t workspace_bytes, n2d2hip_stream_t stream)
{
    N2D2HIP_REQUIRE(target && output && diff && loss && n > 0 && batch > 0, N2D2HIP_ERR_INVALID, "n2d2hip_loss_f32: bad argument");
    const int nb = grid_for(n);
    N2D2HIP_REQUIRE(workspace && workspace_bytes >= (size_t)nb * sizeof(double), N2D2HIP_ERR_WORKSPACE,
                    "n2d2hip_loss_f32: workspace of %zu bytes, %zu needed", workspace_bytes, (size_t)nb * sizeof(double));
    const int blocks = n <= LOSS_ONE_BLOCK ? 1 : nb;
    hipLaunchKernelGGL(loss_f32_kernel, dim3(blocks), dim3(TBLOCK), 0, (hipStream_t)stream, target, output, diff, n, (double*)workspace, 1.0 / batch, loss);
    if (blocks > 1)
        hipLaunchKernelGGL(loss_finish_kernel, dim3(1), dim3(TBLOCK), 0, (hipStream_t)stream, (const double*)workspace, blocks, 1.0 / batch, loss);
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

int n2d2hip_softmax_loss_f32(const float* x, const float* target, float* y, float* diff, float* diff_x, int B, int C, int H, int W, double* loss, void* workspace,
                             size_t workspace_bytes, n2d2hip_stream_t stream)
{
    N2D2HIP_REQUIRE(B > 0 && C > 0 && H > 0 && W > 0 && x && target && y && diff && loss, N2D2HIP_ERR_INVALID, "n2d2hip_softmax_loss_f32: bad argument");
    const size_t n = (size_t)B * C * H * W;
    N2D2HIP_REQUIRE(workspace && workspace_bytes >= n2d2hip_loss_workspace_bytes(n), N2D2HIP_ERR_WORKSPACE,
                    "n2d2hip_softmax_loss_f32: workspace of %zu bytes, %zu needed", workspace_bytes, n2d2hip_loss_workspace_bytes(n));
    if (n <= LOSS_ONE_BLOCK && C <= 16) {
        N2D2HIP_LAUNCH_T(softmax_loss_f32_kernel, (16), dim3(1), dim3(TBLOCK), 0, (hipStream_t)stream, x, target, y, diff, diff_x, B * H * W, C, H * W, 1.0 / B, loss);
        N2D2HIP_HIP_CHECK(hipGetLastError());
        return N2D2HIP_OK;
    }
    int st = n2d2hip_softmax_f32_forward(x, y, B, C, H, W, stream);
    if (st == N2D2HIP_OK) st = n2d2hip_loss_f32(target, y, diff, n, B, loss, workspace, workspace_bytes, stream);
    if (st == N2D2HIP_OK && diff_x) st = n2d2hip_elemwise_sum_f32_backward(n, 1.0f, diff, 0.0f, diff_x, stream);
    return st;
}

static int sgd_check(const n2d2hip_sgd_item* items, int count)
{
    N2D2HIP_REQUIRE(items && count > 0, N2D2HIP_ERR_INVALID, "n2d2hip_sgd_update_f32: bad argument");
    for (int k = 0; k < count; ++k) {
        N2D2HIP_REQUIRE(items[k].data && items[k].diff && items[k].n > 0, N2D2HIP_ERR_INVALID, "n2d2hip_sgd_update_f32: bad argument");
        N2D2HIP_REQUIRE(items[k].momentum_data || (items[k].momentum == 0.0f && items[k].decay_times_rate == 0.0f), N2D2HIP_ERR_INVALID,
                        "n2d2hip_sgd_update_f32: momentum or decay without a momentum buffer");
    }
    return N2D2HIP_OK;
}
int n2d2hip_sgd_update_f32_batch(const n2d2hip_sgd_item* items, int count, n2d2hip_stream_t stream)
{
    const int rc = sgd_check(items, count);
    if (rc != N2D2HIP_OK) return rc;
    for (int k = 0; k < count; k += SGD_ITEMS) {
        const int nb = std::min(count - k, SGD_ITEMS);
        if (nb == 1) {
            const SgdBatch<1> b = sgd_batch<1>(items + k, nb);
            hipLaunchKernelGGL(sgd_f32_kernel<1>, dim3(b.first[nb]), dim3(TBLOCK), 0, (hipStream_t)stream, b);
        } else {
            const SgdBatch<SGD_ITEMS> b = sgd_batch<SGD_ITEMS>(items + k, nb);
            hipLaunchKernelGGL(sgd_f32_kernel<SGD_ITEMS>, dim3(b.first[nb]), dim3(TBLOCK), 0, (hipStream_t)stream, b);
        }
    }
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

int n2d2hip_sgd_update_f32_batch_sat(const n2d2hip_sgd_item* items, int count, const n2d2hip_sat_weight_grad_item* grads, int nb_grads, n2d2hip_stream_t stream)
{
    int rc = sgd_check(items, count);
    if (rc != N2D2HIP_OK) return rc;
    N2D2HIP_REQUIRE(nb_grads >= 0 && (grads || nb_grads == 0), N2D2HIP_ERR_INVALID, "n2d2hip_sgd_update_f32_batch_sat: bad argument");
    // whose gradient an item's is: at most one item's each; the others are computed first
    std::vector<int> grad_of(count, -1);
    std::vector<n2d2hip_sat_weight_grad_item> others;
    for (int g = 0; g < nb_grads; ++g) {
        rc = sat_weight_grad_check(grads[g]);
        if (rc != N2D2HIP_OK) return rc;
        int item = 0;
        while (item < count && !(items[item].diff == grads[g].diff_w && items[item].data == grads[g].w && items[item].n == grads[g].n && grad_of[item] < 0)) ++item;
        if (item < count) grad_of[item] = g;
        else others.push_back(grads[g]);
    }
    if (!others.empty()) {
        rc = n2d2hip_sat_weight_backward_batch(others.data(), (int)others.size(), stream);
        if (rc != N2D2HIP_OK) return rc;
    }
    if ((int)others.size() == nb_grads) return n2d2hip_sgd_update_f32_batch(items, count, stream);
    for (int k = 0; k < count;) {
        int nb = 0, nb_sat = 0;
        SgdSatBatch b = {};
        for (; nb < SGD_ITEMS && k + nb < count; ++nb) {
            const int g = grad_of[k + nb];
            if (g >= 0 && nb_sat == SGD_GRADS) break;
            b.grad_of[nb] = (signed char)(g < 0 ? -1 : nb_sat);
            if (g < 0) continue;
            b.grad[nb_sat] = grads[g];
            b.mode_factor[nb_sat++] = sat_weight_mode_factor(grads[g]);
        }
        b.sgd = sgd_batch<SGD_ITEMS>(items + k, nb);
        hipLaunchKernelGGL(sgd_sat_f32_kernel, dim3(b.sgd.first[nb]), dim3(TBLOCK), 0, (hipStream_t)stream, b);
        k += nb;
    }
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

int n2d2hip_sgd_update_f32(float* data, const float* diff, size_t n, float rate_diff, float momentum, float decay_times_rate,
                           float* momentum_data, int clamp, float clamp_min, float clamp_max, n2d2hip_stream_t stream)
{
    const n2d2hip_sgd_item item = {data, diff, n, momentum_data, rate_diff, momentum, decay_times_rate, clamp_min, clamp_max, clamp};
    return n2d2hip_sgd_update_f32_batch(&item, 1, stream);
}

} // extern "C"
