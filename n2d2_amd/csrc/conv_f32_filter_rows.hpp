// Backward-filter of 3x3 float convolutions of stride 1 or 2 and one column of padding on the left, on the bf16 matrix cores with every
// float in three parts (conv_f32_patch.hpp): dw[q][c][tap] = sum over output pixels of dy[q][pixel] x[c][the tap's source pixel].
//
// K is the pixels, 8 consecutive ones of a row to an operand register, rows padded to whole octets.  A step brings a few rows of dy
// (64 channels) and the rows of x that they meet (32 channels) into LDS, apart in parts, and serves all nine taps: a tap's row is
// another LDS address, its column the octet shifted by one value in registers (stride 2: even and odd columns apart, one shift).
// Rows are counted over all images with room for the padding between them, so that a step's rows follow each other whatever image
// they are of; what lies outside is loaded as zero.
//
// us with the launch that adds the ranges, fp32 matrix cores (conv_f32_filter_kernel) / now, and error against 64 bits:
//   64 <- 64, 56 x 56, batch 64             168 / 115    5.3e-7 / 1.9e-7
//   64 <- 64, 32 x 32, batch 64              64 /  44    3.7e-7 / 1.1e-7
//   256 <- 256, 14 x 14, batch 32            86 /  61    3.7e-7 / 1.4e-7
//   512 <- 512, 14 x 14, batch 8             95 /  69    3.9e-7 / 1.4e-7
//   256 <- 128, stride 2, 27 x 27, batch 33  54 /  46    3.7e-7 / 1.0e-7
// 64 <- 64 on 32 x 32 is 14 us of matrix instructions at their rate.  Of the 74000 cycles of a block: 8000 until the first step is there; four
// times 14000, 7000 of them matrix instructions, 2300 that take the floats apart, 1100 for the next step's addresses, the rest loads that
// the L1 takes slowly (a lane's 16 bytes are of 64 different rows) and what one half waits for the other; 9000 for the results.
// (All loads of a step ahead of its products: 128 on 56 x 56; spread over both of a step's runs of four octets: registers spill, 160.)
#pragma once

#include "conv_f32_patch.hpp"

namespace n2d2hip {

struct FilterRows {
    int B, C, Q, H, W, oH, oW, pt;
    int D;                     // rows of dy from one image to the next, S D of x
    int pieces, chunks;        // steps of a row of octets; steps in all
    int per;                   // steps of one blockIdx.z
    int masked;                // a row ends inside an octet
    unsigned bytesX, bytesY;
    DivF32 dD, dSD, dpieces;
};
constexpr int ROWS_Q = 64, ROWS_C = 32, ROWS_TILE = ROWS_Q * ROWS_C * 9;

// Where a lane of a tile's wave has its results: value k (72 of them) of thread t (256)
__device__ __forceinline__ void rows_place(int k, int t, int* q, int* c, int* tap)
{
    const int lane = t & 63, wave = t >> 6, r = k & 3, m = (k >> 2) & 1;
    *tap = k >> 3;
    *q = (wave >> 1) * 32 + m * 16 + 4 * (lane >> 4) + r;
    *c = (wave & 1) * 16 + (lane & 15);
}

// A tile is 64 q x 32 c x 9 taps.  Four waves have 32 q x 16 c of it each; the block's two halves of four take every other step, and
// their sums are added before they are stored: half the partial results, with two waves to a SIMD.  NOL: log2 of the octets of a row
// in a step (of 8 octets; 4 at stride 2).
template <int S, int NOL>
__global__ __launch_bounds__(512, 2) void conv_f32_filter_rows_kernel(FilterRows g, const float* __restrict__ x, const float* __restrict__ dy,
                                                                      float* __restrict__ partial)
{
    constexpr int NO = 1 << NOL, NE = S == 1 ? 8 : 4, RW = NE >> NOL;
    static_assert(RW >= 1, "a row's octets fit a step");
    constexpr int RX = (RW - 1) * S + 3;         // rows of x
    constexpr int SL = S == 1 ? NO + 2 : 2 * NO + 1;         // 16-byte slots of a row and channel: octets -1 .. NO, or the odd columns of -1 .. NO - 1, then the even ones
    constexpr int XJ = S == 1 ? SL : NO + 1;     // loads of a row: 8 S columns each
    constexpr int YPART = NE * ROWS_Q * 16, XPART = RX * SL * ROWS_C * 16, HALF = 3 * (YPART + XPART);
    constexpr int NY = NE * ROWS_Q / 256, XU = RX * XJ * ROWS_C, NX = (XU + 255) / 256;
    __shared__ __attribute__((aligned(16))) char smem[2 * HALF];
    const int tid = threadIdx.x & 255, half = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8);
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, lo = lane >> 4, wq = wave >> 1, wc = wave & 1;
    const int c0 = blockIdx.x * ROWS_C, q0 = blockIdx.y * ROWS_Q;
    char* const ly = smem + half * HALF;
    char* const lx = ly + 3 * YPART;
    const __amdgpu_buffer_rsrc_t rsrcX = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(x), 0, g.bytesX, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrcY = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(dy), 0, g.bytesY, 0x00020000);

    float yv[NY][8], xv[NX][8 * S];
    unsigned yoff[NY], xoff[NX];
    // first column of a load
    auto ycol = [&](int piece, int u) { return 8 * (piece * NO + (u / ROWS_Q & (NO - 1))); };
    auto xcol = [&](int piece, int u) { return 8 * S * (piece * NO + u / ROWS_C % XJ - 1); };
    auto locate = [&](int chunk) {
        const int row = div_f32(chunk, g.dpieces), piece = chunk - row * g.pieces, v0 = row * RW;
#pragma unroll
        for (int i = 0; i < NY; ++i) {
            const int u = tid + 256 * i, q = q0 + (u & (ROWS_Q - 1)), e = u / ROWS_Q;
            const int v = v0 + (e >> NOL), img = div_f32(v, g.dD), oy = v - img * g.D;
            const int col = ycol(piece, u);
            yoff[i] = q < g.Q && img < g.B && oy < g.oH && col < g.oW ? 4u * (unsigned)(((img * g.Q + q) * g.oH + oy) * g.oW + col) : F32_OOB;
        }
#pragma unroll
        for (int i = 0; i < NX; ++i) {
            const int u = tid + 256 * i, c = c0 + (u & (ROWS_C - 1)), rx = u / (ROWS_C * XJ);
            const int v = S * v0 + rx - g.pt, img = div_f32(max(v, 0), g.dSD), y = v - img * S * g.D;
            const int col = xcol(piece, u);
            xoff[i] = u < XU && c < g.C && v >= 0 && img < g.B && y < g.H && col >= 0 && col < g.W
                          ? 4u * (unsigned)(((img * g.C + c) * g.H + y) * g.W + col) : F32_OOB;
        }
    };
    constexpr int LOADS = 2 * NY + 2 * S * NX;
    auto load = [&](int from, int to) {
#pragma unroll
        for (int l = from; l < to; ++l) {
            const bool of_y = l < 2 * NY;
            const int i = of_y ? l / 2 : (l - 2 * NY) / (2 * S), k = of_y ? l % 2 : (l - 2 * NY) % (2 * S);
            const v4u u = __builtin_bit_cast(v4u, of_y ? __builtin_amdgcn_raw_buffer_load_b128(rsrcY, yoff[i], 16 * k, 0)
                                                       : __builtin_amdgcn_raw_buffer_load_b128(rsrcX, xoff[i], 16 * k, 0));
            float* const v = of_y ? yv[i] : xv[i];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const unsigned w = u[j];
                v[4 * k + j] = __builtin_bit_cast(float, w);
            }
        }
    };
    auto put = [&](int chunk) {
        auto parts_of = [&](float (&v)[8], char* at, int stride) {
            v4u parts[3];
            bf16_parts(v, parts);
#pragma unroll
            for (int p = 0; p < 3; ++p) *(v4u*)(at + p * stride) = parts[p];
        };
        if (g.masked) {                          // (what is of the next row)
            const int piece = chunk - div_f32(chunk, g.dpieces) * g.pieces;
#pragma unroll
            for (int i = 0; i < NY; ++i) {
                const int left = g.oW - ycol(piece, tid + 256 * i);
#pragma unroll
                for (int j = 0; j < 8; ++j) yv[i][j] = j < left ? yv[i][j] : 0.0f;
            }
#pragma unroll
            for (int i = 0; i < NX; ++i) {
                const int left = g.W - xcol(piece, tid + 256 * i);
#pragma unroll
                for (int j = 0; j < 8 * S; ++j) xv[i][j] = j < left ? xv[i][j] : 0.0f;
            }
        }
#pragma unroll
        for (int i = 0; i < NY; ++i) parts_of(yv[i], ly + (tid + 256 * i) * 16, YPART);
#pragma unroll
        for (int i = 0; i < NX; ++i) {
            const int u = tid + 256 * i, c = u & (ROWS_C - 1), rest = u / ROWS_C, rx = rest / XJ, j = rest - rx * XJ;
            if (XU % 256 != 0 && u >= XU) continue;
            if constexpr (S == 1) {
                parts_of(xv[i], lx + u * 16, XPART);
            } else {
                float odd[8], even[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) { even[k] = xv[i][2 * k]; odd[k] = xv[i][2 * k + 1]; }
                char* const at = lx + ((rx * SL + j) * ROWS_C + c) * 16;
                parts_of(odd, at, XPART);
                if (j > 0) parts_of(even, at + NO * ROWS_C * 16, XPART);
            }
        }
    };
    v4f acc[9][2];
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int m = 0; m < 2; ++m) acc[t][m] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    // this lane's octet of the first four, and where the next four are from there
    const int r0 = S * (lo >> NOL), o0 = lo & (NO - 1);
    const unsigned ya = (lo * ROWS_Q + wq * 32 + l16) * 16, xa = ((r0 * SL + o0 + 1) * ROWS_C + wc * 16 + l16) * 16;
    constexpr int YNEXT = 4 * ROWS_Q * 16, XNEXT = (NOL == 3 ? 4 : ((4 >> NOL) * S * SL)) * ROWS_C * 16, ROW = SL * ROWS_C * 16, SLOT = ROWS_C * 16;
    // (a load of 16 bytes a lane, of 64 rows, takes the L1 some 50 cycles: spread over the matrix instructions)
    auto compute = [&](bool more) {
#pragma unroll 1
        for (int st = 0; st < NE / 4; ++st) {
            v4u a[2][3];
#pragma unroll
            for (int m = 0; m < 2; ++m)
#pragma unroll
                for (int p = 0; p < 3; ++p) a[m][p] = *(const v4u*)(ly + ya + st * YNEXT + p * YPART + m * 256);
#pragma unroll
            for (int ty = 0; ty < 3; ++ty) {
                if (more && st == 0) load(ty * LOADS / 3, (ty + 1) * LOADS / 3);
                __builtin_amdgcn_sched_barrier(0);
                const char* at = lx + xa + st * XNEXT + ty * ROW;
                v4u d[3], even[S == 1 ? 1 : 3];
                unsigned before[3], after[3];
#pragma unroll
                for (int p = 0; p < 3; ++p) {
                    d[p] = *(const v4u*)(at + p * XPART);
                    before[p] = *(const unsigned*)(at + p * XPART - SLOT + 12);
                    if (S == 1) after[p] = *(const unsigned*)(at + p * XPART + SLOT);
                    else even[S == 1 ? 0 : p] = *(const v4u*)(at + p * XPART + NO * SLOT);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    const int tx = i == 0 ? 1 : i == 1 ? 0 : 2;
                    v4u b[3];
#pragma unroll
                    for (int p = 0; p < 3; ++p) {
                        auto joined = [](unsigned hi, unsigned lo_) { return __builtin_amdgcn_alignbit(hi, lo_, 16); };
                        if (tx == 0) b[p] = v4u{joined(d[p][0], before[p]), joined(d[p][1], d[p][0]), joined(d[p][2], d[p][1]), joined(d[p][3], d[p][2])};
                        else if (S == 1) b[p] = tx == 1 ? d[p] : v4u{joined(d[p][1], d[p][0]), joined(d[p][2], d[p][1]), joined(d[p][3], d[p][2]), joined(after[p], d[p][3])};
                        else b[p] = tx == 1 ? even[S == 1 ? 0 : p] : d[p];
                    }
                    v4f small[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
                    for (int s = 0; s < 5; ++s) {
                        constexpr int pa[5] = {1, 0, 2, 0, 1}, pb[5] = {1, 2, 0, 1, 0};
#pragma unroll
                        for (int m = 0; m < 2; ++m)
                            small[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a[m][pa[s]]), __builtin_bit_cast(v8bf, b[pb[s]]), small[m], 0, 0, 0);
                    }
#pragma unroll
                    for (int m = 0; m < 2; ++m)
                        acc[3 * ty + tx][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a[m][0]), __builtin_bit_cast(v8bf, b[0]), acc[3 * ty + tx][m], 0, 0, 0);
#pragma unroll
                    for (int m = 0; m < 2; ++m)
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[3 * ty + tx][m][r] += small[m][r];
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
    };
    const int beg = blockIdx.z * g.per, end = min(beg + g.per, g.chunks);
    for (int chunk = beg + half - 2; chunk - half < end; chunk += 2) {           // (the first: only loads; both halves run as many)
        const bool more = chunk + 2 < end;
        if (more) locate(chunk + 2);
        if (chunk >= beg && chunk < end) compute(more);
        else if (more) load(0, LOADS);
        __syncthreads();
        if (more) put(chunk + 2);
        __syncthreads();
    }
    // each half of the block ends with the sums of 16 of a wave's 32 rows
    float* const red = (float*)smem;
#pragma unroll
    for (int t = 0; t < 9; ++t) *(v4f*)(red + ((half * 9 + t) * 256 + tid) * 4) = half ? acc[t][0] : acc[t][1];
    __syncthreads();
    float* const out = partial + ((size_t)blockIdx.z * gridDim.y * gridDim.x + blockIdx.y * gridDim.x + blockIdx.x) * ROWS_TILE;
    float finite = 0.0f;
    v4f sum[9];
#pragma unroll
    for (int t = 0; t < 9; ++t) {
        // (the sums of the first half first, in both)
        const v4f other = *(const v4f*)(red + (((1 - half) * 9 + t) * 256 + tid) * 4);
        sum[t] = (half ? other + acc[t][1] : acc[t][0] + other) * PARTS_UNSCALE;
#pragma unroll
        for (int r = 0; r < 4; ++r) finite = __builtin_fmaf(sum[t][r], 0.0f, finite);
    }
    if (__any(finite != finite)) {
        // Infinities, and what rounds to one in bf16, leave NaN where float products might not: a wave that holds such sums adds them
        // again, on the fp32 matrix cores straight from memory, in double from eight pixels to the next.  Where a tap lies outside x
        // both operands are 0.
        // us of 64 <- 64, 56 x 56, batch 64: finite 118; NaN throughout 960; a channel of x NaN 704 (a sum after the other by the lane that
        // held it: 15570, 9030).
        int here = lane;                         // (opaque: nothing of this is worked out ahead, and held, by waves that never come here)
        asm volatile("" : "+v"(here));
        const int l16 = here & 15, lo = here >> 4, q = q0 + wq * 32 + half * 16 + l16, ch = c0 + wc * 16 + l16;
        double folded[9][4] = {};
#pragma unroll 1
        for (int chunk = beg; chunk < end; ++chunk) {
            const int row = div_f32(chunk, g.dpieces), piece = chunk - row * g.pieces;
#pragma unroll 1
            for (int e = 0; e < NE; ++e) {
                const int v = row * RW + (e >> NOL), img = div_f32(v, g.dD), oy = v - img * g.D;
                if (img >= g.B || oy >= g.oH) continue;
                v4f part[9];
#pragma unroll
                for (int t = 0; t < 9; ++t) part[t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
                for (int h = 0; h < 8; h += 4) {
                    const int ox = 8 * (piece * NO + (e & (NO - 1))) + h + lo;
                    const float d = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                        rsrcY, q < g.Q && ox < g.oW ? 4u * (unsigned)(((img * g.Q + q) * g.oH + oy) * g.oW + ox) : F32_OOB, 0, 0));
#pragma unroll
                    for (int t = 0; t < 9; ++t) {
                        const int y = oy * S - g.pt + t / 3, col = ox * S - 1 + t % 3;
                        const bool there = ox < g.oW && (unsigned)y < (unsigned)g.H && (unsigned)col < (unsigned)g.W;
                        const float u = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                            rsrcX, there && ch < g.C ? 4u * (unsigned)(((img * g.C + ch) * g.H + y) * g.W + col) : F32_OOB, 0, 0));
                        part[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(there ? d : 0.0f, u, part[t], 0, 0, 0);
                    }
                }
#pragma unroll
                for (int t = 0; t < 9; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) folded[t][r] += (double)part[t][r];
            }
        }
#pragma unroll
        for (int t = 0; t < 9; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (!(__builtin_fabsf(sum[t][r]) < __builtin_inff())) sum[t][r] = (float)folded[t][r];
    }
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) out[((t * 2 + half) * 4 + r) * 256 + tid] = sum[t][r];
}

// dw[q][c][tap] = sum over the ranges + beta * dw: 64 values of a tile to a block, each of its four waves a quarter of the ranges, in
// double and in their order.
__global__ __launch_bounds__(256) void conv_f32_reduce_rows_kernel(const float* __restrict__ partial, int splits, int ctiles, size_t n, int Q, int C, float beta,
                                                                   float* __restrict__ dw)
{
    __shared__ double red[4][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int z0 = splits * w / 4, z1 = splits * (w + 1) / 4;
    const size_t i = (size_t)blockIdx.x * 64 + lane;         // (n is a multiple of 64)
    double s = 0.0;
    int z = z0;
    for (; z + 8 <= z1; z += 8) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = partial[(size_t)(z + j) * n + i];
#pragma unroll
        for (int j = 0; j < 8; ++j) s += (double)v[j];
    }
    for (; z < z1; ++z) s += (double)partial[(size_t)z * n + i];
    red[w][lane] = s;
    __syncthreads();
    if (w != 0) return;
    const int tile = (int)(i / ROWS_TILE), rest = (int)(i % ROWS_TILE);
    int q, c, tap;
    rows_place(rest >> 8, rest & 255, &q, &c, &tap);
    q += tile / ctiles * ROWS_Q;
    c += tile % ctiles * ROWS_C;
    if (q >= Q || c >= C) return;
    const size_t at = ((size_t)q * C + c) * 9 + tap;
    const double t = ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
    dw[at] = (float)t + (beta != 0.0f ? beta * dw[at] : 0.0f);
}

} // namespace n2d2hip
