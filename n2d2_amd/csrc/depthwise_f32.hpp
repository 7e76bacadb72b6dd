// Float32 depthwise convolutions of 3x3 and 5x5 kernels at stride 1 or 2: forward, backward-data, backward-filter.
//
// A depthwise layer has 2 K^2 flops for 8 bytes: memory bounds it.  One thread per output took a load, its address and its
// validity test per product, and backward-filter read both tensors once per weight (9 times).  Here a thread takes a strip of
// four outputs of a row: its window of a source row comes in one or two 16-byte loads and serves all its products; a block
// works on one channel, so the weights are scalar.  Loads are of dwords at any 4-byte address, so widths need not be
// multiples of four: what a window reads beyond its row (the neighbouring row's values) is left out by a select per product,
// never multiplied by 0, so an infinity there does no harm.  Only a window that would leave the tensor is read value by value.
// Other kernels and strides stay with the kernels of one load per product.
#pragma once

#include "conv_f32_gemm.hpp"

namespace n2d2hip {

struct DepthwiseF32 {
    int C, H, W, oH, oW, pl, pt;
    int items;                                   // strips of four of one channel over batch and rows
    int strips;                                  // strips of a row
    int nx, ny;                                  // values of x (or dx) and y (or dy)
    DivF32 dstrips, drows;
    int narrow;                                  // backward-filter: strips are whole, and reach at most K / 2 columns past a row's ends
};

typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x2_any __attribute__((ext_vector_type(2), aligned(4)));

// dst[j] = p[base + j]; what lies outside the tensor of n values reads as 0
template <int N>
__device__ __forceinline__ void strip_load(float* dst, const float* __restrict__ p, int base, int n)
{
    if (base >= 0 && base <= n - N) {
        constexpr int V = N & ~3;
#pragma unroll
        for (int j = 0; j < V; j += 4) {
            const f32x4_any v = *(const f32x4_any*)(p + base + j);
            dst[j] = v.x; dst[j + 1] = v.y; dst[j + 2] = v.z; dst[j + 3] = v.w;
        }
        if (N & 2) {
            const f32x2_any v = *(const f32x2_any*)(p + base + V);
            dst[V] = v.x; dst[V + 1] = v.y;
        }
        if (N & 1) dst[N - 1] = p[base + N - 1];
    } else {
#pragma unroll
        for (int j = 0; j < N; ++j) dst[j] = base + j >= 0 && base + j < n ? p[base + j] : 0.0f;
    }
}

// out = sum + beta * out (+ bias) for the strip at out[base], of which `count` values exist
__device__ __forceinline__ void strip_store(float* __restrict__ out, int base, int count, float* r, float beta, const float* __restrict__ bias, int c)
{
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        r[u] = r[u] + (beta != 0.0f && u < count ? beta * out[base + u] : 0.0f);
        if (bias) r[u] = bias[c] + r[u];
    }
    if (count >= 4) {
        *(f32x4_any*)(out + base) = f32x4_any{r[0], r[1], r[2], r[3]};
    } else {
#pragma unroll
        for (int u = 0; u < 3; ++u)
            if (u < count) out[base + u] = r[u];
    }
}

// Forward.  The terms are added in the order of the one-output kernels: tap by tap over the clipped window, a full 3x3 window
// row by row, then the rows.
template <int K, int S>
__global__ __launch_bounds__(256) void depthwise_f32_forward_kernel(DepthwiseF32 q, const float* __restrict__ x, const float* __restrict__ w,
                                                                    const float* __restrict__ bias, float beta, float* __restrict__ y)
{
    constexpr int NX = 3 * S + K;
    const int i = blockIdx.x * 256 + threadIdx.x, c = blockIdx.y;
    if (i >= q.items) return;
    const int r = div_f32(i, q.dstrips), ox0 = (i - r * q.strips) * 4, b = div_f32(r, q.drows), oy = r - b * q.oH;
    const int iy0 = oy * S - q.pt, ix0 = ox0 * S - q.pl, img = b * q.C + c;
    const float* wc = w + c * (K * K);
    float xv[K][NX];
    bool row[K], col[NX];
#pragma unroll
    for (int j = 0; j < NX; ++j) col[j] = (unsigned)(ix0 + j) < (unsigned)q.W;
#pragma unroll
    for (int t = 0; t < K; ++t) {
        row[t] = (unsigned)(iy0 + t) < (unsigned)q.H;
        if (row[t]) {
            strip_load<NX>(xv[t], x, (img * q.H + iy0 + t) * q.W + ix0, q.nx);
        } else {
#pragma unroll
            for (int j = 0; j < NX; ++j) xv[t][j] = 0.0f;
        }
    }
    float sum[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        float s = 0.0f;
        float p[K][K];
#pragma unroll
        for (int t = 0; t < K; ++t)
#pragma unroll
            for (int j = 0; j < K; ++j) {
                p[t][j] = wc[t * K + j] * xv[t][u * S + j];
                s = row[t] && col[u * S + j] ? s + p[t][j] : s;
            }
        if (K == 3) {
            const float full = 0.0f + (p[0][0] + p[0][1] + p[0][2]) + (p[1][0] + p[1][1] + p[1][2]) + (p[2][0] + p[2][1] + p[2][2]);
            s = row[0] && row[1] && row[2] && col[u * S] && col[u * S + 1] && col[u * S + 2] ? full : s;
        }
        sum[u] = s;
    }
    strip_store(y, (img * q.oH + oy) * q.oW + ox0, q.oW - ox0, sum, beta, bias, c);
}

// Backward-data: dx[iy][ix] adds w[ty][tx] dy[(iy + pt - ty) / S][(ix + pl - tx) / S] over the taps that reach it, ascending.
// At stride 2 every other row and column of taps does: which columns is known at compile time from P, the parity of the left
// padding (a strip starts at a multiple of four); which rows, from the lane's own row.
// 128 channels, 3x3, 56 x 56, batch 32: one thread per value 167.5 us, strips 19.4 (5.3 TB/s).
template <int K, int S, int P>
__global__ __launch_bounds__(256) void depthwise_f32_data_kernel(DepthwiseF32 q, const float* __restrict__ w, const float* __restrict__ dy, float beta,
                                                                 float* __restrict__ dx)
{
    constexpr int NI = (K + S - 1) / S;                      // tap rows that reach a row
    constexpr int LO = S == 1 ? -(K - 1) : -((K - 1) / 2);   // the window: columns LO .. HI of dy, from the strip's own
    constexpr int HI = S == 1 ? 3 : (3 + P) / 2;
    constexpr int NX = HI - LO + 1;
    const int i = blockIdx.x * 256 + threadIdx.x, c = blockIdx.y;
    if (i >= q.items) return;
    const int r = div_f32(i, q.dstrips), ix0 = (i - r * q.strips) * 4, b = div_f32(r, q.drows), iy = r - b * q.H;
    const int img = b * q.C + c;
    const int iyPad = iy + q.pt, oy0 = iyPad / S, ty0 = iyPad - oy0 * S;
    const int oxb = (S == 1 ? ix0 + q.pl : ix0 / 2 + q.pl / 2) + LO;
    const float* wc = w + c * (K * K);
    float v[NI][NX];
    bool row[NI], col[NX];
#pragma unroll
    for (int j = 0; j < NX; ++j) col[j] = (unsigned)(oxb + j) < (unsigned)q.oW;
#pragma unroll
    for (int t = 0; t < NI; ++t) {
        row[t] = (unsigned)(oy0 - t) < (unsigned)q.oH && ty0 + t * S < K;
        if (row[t]) {
            strip_load<NX>(v[t], dy, (img * q.oH + oy0 - t) * q.oW + oxb, q.ny);
        } else {
#pragma unroll
            for (int j = 0; j < NX; ++j) v[t][j] = 0.0f;
        }
    }
    float sum[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        float s = 0.0f;
#pragma unroll
        for (int t = 0; t < NI; ++t)
#pragma unroll
            for (int tx = 0; tx < K; ++tx) {
                const int e = S == 1 ? u - tx : u + P - tx;
                if (S == 2 && (e & 1)) continue;
                const int j = (S == 1 ? e : e / 2) - LO;
                const float w0 = wc[t * S * K + tx];
                const float wt = S == 2 && t * S + 1 < K ? (ty0 ? wc[(t * S + 1) * K + tx] : w0) : w0;
                s = row[t] && col[j] ? s + wt * v[t][j] : s;
            }
        sum[u] = s;
    }
    strip_store(dx, (img * q.H + iy) * q.W + ix0, q.W - ix0, sum, beta, nullptr, c);
}

// Backward-filter: a block adds the products of all K^2 taps over one range of a channel's strips in double, so both tensors
// are read once (x's rows K times, out of the caches).  gridDim.y is the number of ranges; one: the sums are the gradient,
// more: they go to partial[range][channel][tap], which conv_f32_reduce_partials_kernel adds up.
// What bounds it is the vector ALU: four instructions a product (multiply, select, conversion, addition in double), three where the
// product's column is in the row for certain: rows of whole strips with at most K / 2 columns of padding on either side (q.narrow)
// select for the K / 2 outer columns of a strip alone.  us, all / these: 128 channels, 3x3, 56 x 56, batch 32 30.3 / 25.8; 64 channels,
// 112 x 112 46.7 / 38.5, at stride 2 28.4 / 27.0; 96 channels, 5x5, 56 x 56, batch 16 28.3 / 23.5.  (Multiply-adds in double, an
// instruction a product behind the conversions: 40.6 for the first.)
// 128 channels, 3x3, 56 x 56, batch 32: a block per channel and tap row, which loaded and converted dy's strip once per row
// and stood on 384 blocks, 48.6 us; now 31.1 with the launch that adds the ranges up.
// ROWS: tap rows of a block, all K, or one (blockIdx.z is which) where a channel's strips are few: depthwise_row_threads() in
// train_f32.hip says where and measures both.  THREADS: 256; of one row, where blocks are few, 512 or 1024, and so of all rows where
// a range is a whole channel because the caller gave no workspace.
template <int K, int S, int THREADS, int ROWS>
__global__ __launch_bounds__(THREADS) void depthwise_f32_filter_kernel(DepthwiseF32 q, int per_range, const float* __restrict__ x, const float* __restrict__ dy,
                                                                   float beta, float* __restrict__ dw, double* __restrict__ partial)
{
    constexpr int NX = 3 * S + K;
    const int c = blockIdx.x, end = min(q.items, ((int)blockIdx.y + 1) * per_range), ty0 = ROWS == K ? 0 : (int)blockIdx.z;
    double acc[ROWS][K] = {};
    const auto add = [&](auto narrow) {
        for (int i = (int)blockIdx.y * per_range + threadIdx.x; i < end; i += THREADS) {
            const int r = div_f32(i, q.dstrips), ox0 = (i - r * q.strips) * 4, b = div_f32(r, q.drows), oy = r - b * q.oH;
            const int iy0 = oy * S - q.pt + ty0, ix0 = ox0 * S - q.pl, img = b * q.C + c;
            float xv[ROWS][NX], dv[4];
            strip_load<4>(dv, dy, (img * q.oH + oy) * q.oW + ox0, q.ny);
#pragma unroll
            for (int ty = 0; ty < ROWS; ++ty)
                if ((unsigned)(iy0 + ty) < (unsigned)q.H)
                    strip_load<NX>(xv[ty], x, (img * q.H + iy0 + ty) * q.W + ix0, q.nx);
            bool inside[4][K];
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int t = 0; t < K; ++t)
                    inside[u][t] = (decltype(narrow)::value && u * S + t >= K / 2 && u * S + t < NX - K / 2)
                                   || (ox0 + u < q.oW && (unsigned)(ix0 + u * S + t) < (unsigned)q.W);
#pragma unroll
            for (int ty = 0; ty < ROWS; ++ty)
                if ((unsigned)(iy0 + ty) < (unsigned)q.H) {
#pragma unroll
                    for (int u = 0; u < 4; ++u)
#pragma unroll
                        for (int t = 0; t < K; ++t) {
                            const float p = xv[ty][u * S + t] * dv[u];
                            acc[ty][t] += (double)(inside[u][t] ? p : 0.0f);
                        }
                }
        }
    };
    if (q.narrow) add(std::true_type{});
    else add(std::false_type{});
    __shared__ double red[THREADS / 64][ROWS * K];
#pragma unroll
    for (int t = 0; t < ROWS * K; ++t) {
        double a = acc[t / K][t % K];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) a += __shfl_xor(a, off, 64);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][t] = a;
    }
    __syncthreads();
    if (threadIdx.x < ROWS * K) {
        double s = 0.0;
        for (int wv = 0; wv < THREADS / 64; ++wv) s += red[wv][threadIdx.x];
        const int idx = (c * K + ty0) * K + threadIdx.x;
        if (gridDim.y == 1) dw[idx] = (float)s + (beta != 0.0f ? beta * dw[idx] : 0.0f);
        else partial[(size_t)blockIdx.y * q.C * K * K + idx] = s;
    }
}

} // namespace n2d2hip
