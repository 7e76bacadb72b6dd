// Float32 convolution (forward, backward-data, backward-filter) as an implicit GEMM on the fp32 matrix cores
// (v_mfma_f32_32x32x2f32), for ungrouped convolutions without dilation on N2D2's NCHW / OCHW tensors.
//
// The product is out[q][p] = sum_k Qop[q][k] * Pop[k][p]:
//   forward          p = output pixel   q = output channel   k = (input channel, tap)    Pop = x gathered, Qop = w
//   backward data    p = input pixel    q = input channel    k = (output channel, tap)   Pop = dy gathered, Qop = w
//   backward filter  p = (channel, tap) q = output channel   k = output pixel            Pop = x gathered, Qop = dy
// Taps that fall outside the tensor contribute zero, which is what the reference's clipped window computes.
//
// Bound by the matrix cores: an fp32 matrix instruction is 4096 flops in 64 cycles, which is the rate of the vector ALU, and
// it runs on that ALU: every vector instruction beside it takes its 4 cycles from it (measured: loads and address
// arithmetic left out, the products alone take as much less time as those take alone).  So:
//  * operands go global -> LDS by direct loads (no registers on the way), into a ring of stages, and everything that does not
//    differ from lane to lane is scalar: a load adds a scalar offset to a per-lane one.  What does not exist (padding, edges
//    of tile and K range) is requested past the end of the buffer descriptor; the LDS receives 0.
//  * kernels of several taps, forward and at stride 1 backward, are mostly left to the bf16 matrix cores (conv_f32_patch.hpp); what that
//    kernel does not take (long rows, few channels), and forward where the caller asks for a rounding a term, stays here.
//  * 3x3 kernels, forward and at stride 1 backward, keep a lane's nine offsets in registers, so that a load costs no vector
//    instruction; 1x1 kernels and strided backward-data run K over chunks of 16 channels at one tap, so that the test whether
//    the tap lies inside the input is made once per step.  A small kernel lays the weights out for both first.  Any other
//    forward kernel, and short passes, test every load.  Kernels of more than 31 rows and columns, up to 64 taps (time series),
//    run on variants of the chunk, pixel and filter kernels that hold a bit per tap instead of one per row and column.
//  * backward-data of a strided convolution runs one residue class of input pixels at a time: the taps of a class form a
//    dense stride-1 convolution of dy, so no tap is tried that cannot hit (a 3x3 of stride 2: 9 taps for 4 classes, where
//    trying all of them is 36).
//  * rows of LDS that hold consecutive k hold the even ones in front of the odd ones, or (filter) give the two lane halves of
//    an instruction different groups of 4 k, so that a lane reads four instructions' operands in 16 bytes.
// A forward sum is added in one order by the 3x3, the chunk (1x1) and the pixel kernel: channel, tap, in pairs, in ranges that
// follow from the sizes.  Two forms have an order of their own: long kernels in chunks of 16 channels at one tap, and layers
// that span their input with up to 64 taps and have room for partial results, which are plain products on the filter kernel
// (its instructions pair k with k + 4).
// Within a block, float sums are added to sums in double after as many steps as keep them no longer than 128 x 128 tiles would.
// Backward-filter, whose K is the whole batch of pixels and whose output is small, splits K over blockIdx.z into partial
// results that a second kernel adds up in a fixed order; forward and backward-data do the same when their tiles alone would
// not fill the chip.
// Measured on these kernels (us, forward / data / filter, before: 128 x 128 tiles, operands through registers, one test per load; now):
//   64 -> 64, 3x3, 56 x 56, batch 64             236 / 284 / 263    149 / 157 / 180   (15 GFLOP: 99, 94, 82 TFLOP/s of 154)
//   128 -> 256, 3x3 stride 2, 27 x 27, batch 33   80 / 277 /  76     55 /  54 /  58
//   a layer spanning its input, 16384 -> 10, 64  2632 /  27 / 222    116 /   7 /   8
//   64 -> 64, 1 x 40, 1 x 512, batch 32            94 / 110 /  98     76 /  72 /  70
//   128 -> 128, 1 x 64, 1 x 256, batch 16         120 / 134 / 124    101 /  96 / 105
// A CU takes whole tiles, so the last round costs its share: 64 -> 64 on 56 x 56 at batch 64 is 12.25 tiles for each.
#pragma once

#include "common.h"
#include "mfma_util.hpp"
#include "sat_math.hpp"

namespace n2d2hip {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v2f __attribute__((ext_vector_type(2)));

struct DivF32 {
    unsigned mul, sh;
};

// The pixels of one launch: all output pixels (forward), or the input pixels of one residue class modulo the stride.
struct PixelClass {
    int tile0;                 // first tile of this class
    int P, gW, gHW;            // pixels over all images; row length and pixels per image of the class's grid
    int nx, nT;                // taps along x, taps
    int kchunk;                // a K range (a multiple of GK; chunked K: in steps of GK)
    int fold;                  // steps of a range after which its float sums are added to those in double; 0: all of it
    int ty0, tx0;              // first tap; the next one along an axis is osy / osx further in the kernel
    int y0, x0;                // source position of tap (0, 0) for grid pixel (0, 0)
    int stepy, stepx;          // element offset from one tap to the next in the source plane
    int soff0, bias;           // element offset of tap (0, 0) against the moved base `src - bias`; both make every offset >= 0
    int w0;                    // conv_f32_taps_kernel: steps of the classes before this one
    int ry, rx;                // output position of grid pixel (py, px): (py * osy + ry, px * osx + rx)
    DivF32 ghw, gw, nt, nxd;
};
constexpr int PIXEL_CLASSES = 4;

struct PixelGemm {
    int Q, Ch;                 // rows of q; channels that k runs over
    int nz;                    // K ranges of a block: blockIdx.z * nz ...
    int sy, sx, d;             // source step per grid pixel (the strides; 1 for backward-data); +1 / -1: per tap
    int Hs, Ws, planeS;        // source plane
    int qs, chs, kW;           // weight element (q, ch, ty, tx) at q * qs + ch * chs + ty * kW + tx
    int osy, osx;              // backward-data: the strides (1 forward)
    int planeO, Wo;            // output plane and its row length
    int ptiles, ptiles8, qtiles;
    int qpad, T;               // chunked K: rows of q in the laid-out weights, taps of the kernel
    unsigned bytesX, bytesW;   // sizes of the operand tensors (below 2 GiB)
    unsigned bytesO;           // of the result
    int npos;                  // source pixels over all images
    DivF32 dplane;             // by the source plane
    int nclass;
    PixelClass c[PIXEL_CLASSES];
};

struct FilterGemm {
    int P, Q, K;
    int kchunk;                // K range of one blockIdx.z (a multiple of FK)
    int fold;                  // steps of it after which the float sums are added to those in double; 0: all of it
    int C, H, W, kW, kH, s_y, s_x, pt, pl;
    int oW, plane;             // output row length and plane
    int imgX, imgY;
    int rowY;                  // from one row of q to the next in Y (the small kernel; others: plane)
    unsigned bytesX, bytesY;
    DivF32 dplane, dow;
};

constexpr int GK = 16;         // K step of the pixel kernels
constexpr int FK = 32;         // of the filter kernel
constexpr unsigned F32_OOB = 0x80000000u;      // byte offset past the end of every operand

__device__ __forceinline__ int div_f32(int n, DivF32 d) { return div_magic(n, d.mul, d.sh); }

template <int OFF>
__device__ __forceinline__ void lds_read128f(v4f& v, unsigned addr)
{
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF) : "memory");
}
template <int OFF>
__device__ __forceinline__ void lds_read64f(v2f& v, unsigned addr)
{
    asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF) : "memory");
}
// two dwords, OFF0 and OFF1 in units of 256 bytes
template <int OFF0, int OFF1>
__device__ __forceinline__ void lds_read2st64f(v2f& v, unsigned addr)
{
    static_assert(OFF0 < 256 && OFF1 < 256, "8-bit offsets");
    asm volatile("ds_read2st64_b32 %0, %1 offset0:%2 offset1:%3" : "=v"(v) : "v"(addr), "n"(OFF0), "n"(OFF1) : "memory");
}
__device__ __forceinline__ void tie(v4f& x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ void tie(v2f& x) { asm volatile("" : "+v"(x)); }

// Which tile a block of the forward / backward-data kernels takes.  Blocks 8 apart share an XCD and its L2: the q tiles of a
// pixel tile come one behind the other on one XCD, and an XCD takes consecutive pixel tiles (they share their halo).  With
// several classes, whose tiles differ in length, the tiles are dealt in turn instead.
__device__ __forceinline__ bool pixel_tile(const PixelGemm& g, int* tile, int* qtile, int* ci)
{
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, pt = slot / g.qtiles;
    *qtile = slot - pt * g.qtiles;
    *tile = g.nclass == 1 ? xcd * g.ptiles8 + pt : pt * 8 + xcd;
    *ci = 0;
#pragma unroll
    for (int i = 1; i < PIXEL_CLASSES; ++i)
        if (i < g.nclass && *tile >= g.c[i].tile0) *ci = i;
    return *tile < g.ptiles;
}

// Which taps lie inside the source.  Bit j: tap column j, bit nx + i: tap row i; bit 31 is never set.  LONG, for kernels of more
// rows and columns than that (1 x 40): a bit for each of up to 64 taps.
template <bool LONG>
struct TapMask {
    unsigned m, high;
    // `bit`: LONG: bit t of its word, or 0 past the range; else the tap's column and row, and bit 31 past the range
    __device__ __forceinline__ bool inside(int t, unsigned bit) const
    {
        // (chosen by bits: a choice between two members goes through their addresses, and the masks live in scratch memory)
        const unsigned upper = t & 32 ? ~0u : 0u;
        if (LONG) return (((high & upper) | (m & ~upper)) & bit) != 0;
        return (m & bit) == bit;
    }
};
// The first tap of each of a kernel's rows, and of the taps those in columns xl .. xh - 1 and rows yl .. yh - 1.
__device__ __forceinline__ unsigned long long long_rows(int ny, int nx)
{
    unsigned long long m = 0;
    for (int i = 0; i < ny; ++i) m |= 1ull << (i * nx);
    return m;
}
__device__ __forceinline__ unsigned long long long_taps(int xl, int xh, int yl, int yh, int nx, unsigned long long rows)
{
    auto below = [](int n) { return n >= 64 ? ~0ull : (1ull << n) - 1; };
    return ((below(xh) & ~below(xl)) * rows) & below(yh * nx) & ~below(yl * nx);
}
// (`left`: negative past the range)
template <bool LONG>
__device__ __forceinline__ unsigned tap_test(int t, int tap_bit, int left)
{
    if (LONG) return (1u << (t & 31)) & ~(unsigned)(left >> 31);
    return (unsigned)__builtin_amdgcn_readlane(tap_bit, t) | ((unsigned)left & 0x80000000u);
}

// A lane's pixel: byte offset of its tap (0, 0) (against the moved base), and its taps inside the source.
template <bool LONG>
__device__ __forceinline__ void pixel_source(const PixelGemm& g, const PixelClass& c, int p, unsigned* voff, TapMask<LONG>* mask)
{
    const int pp = p < c.P ? p : 0;
    const int b = div_f32(pp, c.ghw), rem = pp - b * c.gHW;
    const int py = div_f32(rem, c.gw), px = rem - py * c.gW;
    *voff = 4u * (unsigned)(b * g.Ch * g.planeS + py * g.sy * g.Ws + px * g.sx);
    const int ny = c.nT > 0 ? div_f32(c.nT, c.nxd) : 0;
    if (LONG) {
        const int x = px * g.sx + c.x0, y = py * g.sy + c.y0;
        auto first = [&](int v, int size, int n) { return min(max(g.d > 0 ? -v : v - size + 1, 0), n); };
        auto end = [&](int v, int size, int n) { return min(max(g.d > 0 ? size - v : v + 1, 0), n); };
        const unsigned long long m = long_taps(first(x, g.Ws, c.nx), end(x, g.Ws, c.nx), first(y, g.Hs, ny), end(y, g.Hs, ny), c.nx, long_rows(ny, c.nx));
        mask->m = p < c.P ? (unsigned)m : 0u;
        mask->high = p < c.P ? (unsigned)(m >> 32) : 0u;
        return;
    }
    unsigned m = 0;
    for (int j = 0; j < c.nx; ++j) {
        const int x = px * g.sx + c.x0 + j * g.d;
        m |= (unsigned)(x >= 0 && x < g.Ws) << j;
    }
    for (int i = 0; i < ny; ++i) {
        const int y = py * g.sy + c.y0 + i * g.d;
        m |= (unsigned)(y >= 0 && y < g.Hs) << (c.nx + i);
    }
    mask->m = p < c.P ? m : 0u;
    mask->high = 0;
}

// The products of a wave's 32 x 32 tile from one stage: [16 k][PT pixels] and behind it [QT][16 k], the even k of a row in
// front of the odd ones, in XOR-swizzled 16-byte slots.  A matrix instruction takes k = 2 j (lanes 0 .. 31) and 2 j + 1; group
// gi of the step is j = 4 gi .. 4 gi + 3.
template <int PT>
struct PixelTile {
    v16f acc;
    double folded[16];         // several ranges or folds in a block: their sums, as the partial results of several blocks are added
    v4f fa[2];
    v2f fb[2][2];
    unsigned xaddr, waddr0, waddr1;
    __device__ __forceinline__ void init(unsigned lds0, int wq, int wp, int lane)
    {
        const int l32 = lane & 31, lh = lane >> 5;
        xaddr = lds0 + 4u * (lh * PT + wp * 32 + l32);
        const unsigned wrow = lds0 + 4u * GK * PT + 64u * (wq * 32 + l32);
        waddr0 = wrow + 16u * ((2 * lh) ^ ((l32 >> 2) & 3));
        waddr1 = wrow + 16u * ((2 * lh + 1) ^ ((l32 >> 2) & 3));
#pragma unroll
        for (int r = 0; r < 16; ++r) { acc[r] = 0.0f; folded[r] = 0.0; }
    }
    __device__ __forceinline__ void fold()
    {
#pragma unroll
        for (int r = 0; r < 16; ++r) { folded[r] += (double)acc[r]; acc[r] = 0.0f; }
    }
    __device__ __forceinline__ void unfold()
    {
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = (float)folded[r];
    }
    template <bool LIVE, int gi>
    __device__ __forceinline__ void read_group(unsigned sb)
    {
        constexpr int U = PT / 64;
        if (!LIVE) return;
        const unsigned xa = xaddr + sb;
        lds_read128f<0>(fa[gi], (gi ? waddr1 : waddr0) + sb);
        lds_read2st64f<8 * gi * U, (8 * gi + 2) * U>(fb[gi][0], xa);
        lds_read2st64f<(8 * gi + 4) * U, (8 * gi + 6) * U>(fb[gi][1], xa);
    }
    template <bool LIVE>
    __device__ __forceinline__ void wait_group(int gi)
    {
        if (!LIVE) return;
        wait_lgkm<0>();
        tie(fa[gi]);
        tie(fb[gi][0]);
        tie(fb[gi][1]);
    }
    template <bool LIVE>
    __device__ __forceinline__ void mfma_half(int gi, int half)
    {
        if (!LIVE) return;
#pragma unroll
        for (int j = 2 * half; j < 2 * half + 2; ++j)
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[gi][j], fb[gi][j >> 1][j & 1], acc, 0, 0, 0);
    }
    // One step, with the loads of a coming stage (load_part(0..4)) spread between the matrix instructions, which run on for
    // 64 cycles each while the wave issues them.
    template <bool LIVE, class L>
    __device__ __forceinline__ void step(unsigned sb, L&& load_part)
    {
        read_group<LIVE, 0>(sb);
        load_part(0);
        wait_group<LIVE>(0);
        read_group<LIVE, 1>(sb);
        __builtin_amdgcn_sched_barrier(0);
        mfma_half<LIVE>(0, 0);
        load_part(1);
        __builtin_amdgcn_sched_barrier(0);
        mfma_half<LIVE>(0, 1);
        load_part(2);
        wait_group<LIVE>(1);
        __builtin_amdgcn_sched_barrier(0);
        mfma_half<LIVE>(1, 0);
        load_part(3);
        __builtin_amdgcn_sched_barrier(0);
        mfma_half<LIVE>(1, 1);
        load_part(4);
    }
    // Lane holds column p = .. + lane % 32 and rows q = .. + 8 * (r / 4) + 4 * (lane / 32) + r % 4.  `partial`: elements of
    // one K range's result, 0: one range.
    __device__ __forceinline__ void store(const PixelGemm& g, const PixelClass& c, int p0, int q0, int lane, const float* bias, float beta, float* out,
                                          size_t partial)
    {
        float* dst = out + (size_t)blockIdx.z * partial;
        const int p = p0 + (lane & 31);
        if (p >= c.P) return;
        const int img = div_f32(p, c.ghw), rem = p - img * c.gHW;
        const int py = div_f32(rem, c.gw), px = rem - py * c.gW;
        const size_t base = (size_t)img * g.Q * g.planeO + (py * g.osy + c.ry) * g.Wo + px * g.osx + c.rx;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int q = q0 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
            if (q >= g.Q) continue;
            const size_t idx = base + (size_t)q * g.planeO;
            float v = acc[r];
            if (partial == 0) {
                if (beta != 0.0f) v += beta * dst[idx];
                if (bias) v = bias[q] + v;
            }
            dst[idx] = v;
        }
    }
};

// Weights laid out for the chunked kernel: [chunk of 16 channels][tap][q, padded][16], a row's channels in the order they have
// in LDS; channels and rows that do not exist are zero.
__global__ __launch_bounds__(256) void conv_f32_lay_weights_kernel(const float* __restrict__ w, float* __restrict__ wt, int total, int Q, int qpad, int Ch,
                                                                   int T, int qs, int chs)
{
    for (int i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256) {
        const int q = (i >> 2) % qpad, rest = (i >> 2) / qpad, tap = rest % T, chunk = rest / T;
        const int slot = (i & 3) ^ ((q >> 2) & 3), ch = chunk * GK + 8 * (slot & 1) + (slot >> 1);
        v4f v;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            v[j] = (q < Q && ch + 2 * j < Ch) ? w[(size_t)q * qs + (size_t)(ch + 2 * j) * chs + tap] : 0.0f;
        ((v4f*)wt)[i] = v;
    }
}

// Forward and backward-data with K in chunks of 16 channels at one tap.
template <int WQ, int WP, int S, bool LONG>
__global__ __launch_bounds__(256) void conv_f32_chunk_kernel(PixelGemm g, const float* __restrict__ srcX, const float* __restrict__ wt,
                                                             const float* __restrict__ bias, float beta, float* __restrict__ out, size_t partial)
{
    static_assert(WQ * WP == 4, "four waves");
    constexpr int QT = 32 * WQ, PT = 32 * WP;
    constexpr int PH = PT / 64;                  // loads per k row
    constexpr int WJ = QT >= 64 ? QT / 64 : 1;   // weight loads of a wave per step (1 KB each)
    constexpr int LPI = 4 * PH + WJ;
    constexpr int STAGE = GK * PT + QT * GK;     // floats
    static_assert(LPI * (S - 1) < 60, "vmcnt is a 6-bit counter");
    __shared__ __attribute__((aligned(16))) float smem[S * STAGE];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wq = wave / WP, wp = wave % WP;
    int tile, qtile, ci;
    if (!pixel_tile(g, &tile, &qtile, &ci))
        return;
    const PixelClass& c = g.c[ci];
    const int p0 = (tile - c.tile0) * PT, q0 = qtile * QT;
    const int nT = c.nT, nchunks = (g.Ch + GK - 1) / GK;
    const __amdgpu_buffer_rsrc_t rsrcX = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(srcX) - c.bias, 0, g.bytesX + 4u * c.bias, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrcW = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(wt), 0, nchunks * g.T * g.qpad * GK * 4, 0x00020000);
    unsigned voff[PH], mv[PH];
    TapMask<LONG> mask[PH];
#pragma unroll
    for (int h = 0; h < PH; ++h)
        pixel_source(g, c, p0 + h * 64 + lane, &voff[h], &mask[h]);
    // Tap t of this class lives in lane t, looked up with v_readlane: its offset in the source, its validity bits, its place
    // in the weights.
    const int tl = min(lane, max(nT - 1, 0)), ti = div_f32(tl, c.nxd), tj = tl - ti * c.nx;
    const int tap_off = 4 * (c.soff0 + ti * c.stepy + tj * c.stepx);
    const int tap_bit = LONG ? 0 : (1 << tj) | (1 << (c.nx + ti));
    const int tap_w = ((c.ty0 + ti * g.osy) * g.kW + c.tx0 + tj * g.osx) * g.qpad * (GK * 4);
    const int plane4 = g.planeS * 4;
    PixelTile<PT> tl_acc;
    tl_acc.init((unsigned)(unsigned long)(__attribute__((address_space(3))) float*)smem, wq, wp, lane);
    for (int z = blockIdx.z * g.nz; z < (int)(blockIdx.z + 1) * g.nz; ++z) {
        const int sbeg = z * c.kchunk, nsteps = max(0, min(c.kchunk, nchunks * nT - sbeg));
        int chunk = nT > 0 ? div_f32(sbeg, c.nt) : 0, t = sbeg - chunk * nT;
        int ch_off = (chunk * GK + wave * 4) * plane4, ch_left = g.Ch - chunk * GK - wave * 4;
        int w_off = chunk * g.T * g.qpad * (GK * 4) + q0 * (GK * 4) + (QT >= 64 ? wave : wave & 1) * 1024;
        const int w_chunk = g.T * g.qpad * (GK * 4);
        unsigned xdst = 0;                           // LDS bytes of the stage to load next
        int soff = 0, left = nsteps;
        auto load_part = [&](int part) {
            if (part == 0) {
                const unsigned bit = tap_test<LONG>(t, tap_bit, left - 1);
                soff = ch_off + __builtin_amdgcn_readlane(tap_off, t);
#pragma unroll
                for (int h = 0; h < PH; ++h) mv[h] = mask[h].inside(t, bit) ? voff[h] : F32_OOB;
            }
            if (part < 4) {
#pragma unroll
                for (int h = 0; h < PH; ++h) {
                    const lds_ptr_t dst = (lds_ptr_t)((char*)smem + xdst + ((wave * 4 + part) * PT + h * 64) * 4);
                    if (ch_left >= 4) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrcX, dst, 4, mv[h], soff + part * plane4, 0, 0);
                    else __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrcX, dst, 4, part < ch_left ? mv[h] : F32_OOB, soff + part * plane4, 0, 0);
                }
            } else {
                const int wo = w_off + __builtin_amdgcn_readlane(tap_w, t);
#pragma unroll
                for (int j = 0; j < WJ; ++j)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrcW, (lds_ptr_t)((char*)smem + xdst + GK * PT * 4 + ((QT >= 64 ? wave : wave & 1) + 4 * j) * 1024), 16,
                                                             lane * 16, wo + j * 4096, 0, 0);
                xdst = xdst == 4u * STAGE * (S - 1) ? 0u : xdst + 4u * STAGE;
                --left;
                if (++t >= nT) {
                    t = 0;
                    ch_off += GK * plane4;
                    ch_left -= GK;
                    w_off += w_chunk;
                }
            }
        };

        if (nsteps > 0) {
#pragma unroll
            for (int st = 0; st < S - 1; ++st)       // (steps past the range load zeros: the number in flight stays the same)
#pragma unroll
                for (int part = 0; part < 5; ++part) load_part(part);
            auto k_loop = [&](auto live) {
                unsigned sb = 0;
                for (int st = 0; st < nsteps;) {
                    const int end = c.fold ? min(st + c.fold, nsteps) : nsteps;
                    for (; st < end; ++st) {
                        wait_loads_and_barrier<LPI*(S - 2)>();
                        tl_acc.template step<decltype(live)::value>(sb, load_part);
                        sb = sb == 4u * STAGE * (S - 1) ? 0u : sb + 4u * STAGE;
                    }
                    if (decltype(live)::value && c.fold) tl_acc.fold();      // (not in both loops: that doubles the registers)
                }
            };
            if (q0 + wq * 32 < g.Q) k_loop(std::true_type{});
            else k_loop(std::false_type{});          // (rows past the last: only the loads)
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        if (g.nz > 1 || c.fold) {
            tl_acc.fold();
            __syncthreads();                     // (the next range's loads go where slower waves may still read)
        }
    }
    if (g.nz > 1 || c.fold) tl_acc.unfold();
    tl_acc.store(g, c, p0 + wp * 32, q0 + wq * 32, lane, bias, beta, out, partial);
}

// Weights laid out for the 3x3 kernel: [chunk of 4 channels][q, padded][40], the 36 (channel, tap) products of a row of q with
// the even ones at 0 .. 17 and the odd ones at 20 .. 37.
constexpr int K33 = 36, W33 = 40;
__global__ __launch_bounds__(256) void conv_f32_lay_weights3x3_kernel(const float* __restrict__ w, float* __restrict__ wt, int total, int Q, int qpad, int Ch,
                                                                      int qs, int chs)
{
    for (int i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256) {
        const int e = i % W33, rest = i / W33, q = rest % qpad, chunk = rest / qpad;
        const int half = e >= 20, k = 2 * (e - 20 * half) + half, ch = chunk * 4 + k / 9;
        wt[i] = (e - 20 * half < 18 && q < Q && ch < Ch) ? w[(size_t)q * qs + (size_t)ch * chs + k % 9] : 0.0f;
    }
}

// Forward of a 3x3 kernel, and backward-data at stride 1, with K in the tensors' own order, 4 channels (36 products) a step.
// A lane's nine source offsets, or the one past the end where the tap lies outside, are worked out once for the tile; a load
// then adds only its channel's scalar offset, and between the matrix instructions there is no vector arithmetic left.  A
// wave loads one channel.  Two stages of 19 KB and 4 blocks to a CU: the other blocks cover a step's loads.  (K ranges need
// not start or end with a step: what lies outside is loaded as zero.)
template <int WQ, int WP>
__global__ __launch_bounds__(256) void conv_f32_3x3_kernel(PixelGemm g, const float* __restrict__ srcX, const float* __restrict__ wt,
                                                           const float* __restrict__ bias, float beta, float* __restrict__ out, size_t partial)
{
    static_assert(WQ * WP == 4, "four waves");
    constexpr int QT = 32 * WQ, PT = 32 * WP, PH = PT / 64, U = PT / 64;
    constexpr int STAGE = K33 * PT + QT * W33;   // floats
    constexpr int WL = QT * W33 * 4 / 1024;      // weight loads of a block per step
    __shared__ __attribute__((aligned(16))) float smem[2 * STAGE];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, lh = lane >> 5, wq = wave / WP, wp = wave % WP;
    int tile, qtile, ci;
    if (!pixel_tile(g, &tile, &qtile, &ci))
        return;
    const PixelClass& c = g.c[0];                // (one class)
    const int p0 = tile * PT, q0 = qtile * QT;
    const __amdgpu_buffer_rsrc_t rsrcX = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(srcX) - c.bias, 0, g.bytesX + 4u * c.bias, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrcW = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(wt), 0, (g.Ch + 3) / 4 * g.qpad * W33 * 4, 0x00020000);
    unsigned tap[PH][9];
#pragma unroll
    for (int h = 0; h < PH; ++h) {
        unsigned voff;
        TapMask<false> mask;
        pixel_source(g, c, p0 + h * 64 + lane, &voff, &mask);
#pragma unroll
        for (int t = 0; t < 9; ++t) {
            const unsigned bit = (1u << t % 3) | (8u << t / 3);
            tap[h][t] = mask.inside(t, bit) ? voff + 4 * (c.soff0 + t / 3 * c.stepy + t % 3 * c.stepx) : F32_OOB;
        }
    }
    const int plane4 = g.planeS * 4, wstep = g.qpad * W33 * 4;
    PixelTile<PT> acc;
    acc.init(0, wq, wp, lane);
    const unsigned lds0 = (unsigned)(unsigned long)(__attribute__((address_space(3))) float*)smem;
    const unsigned xaddr = lds0 + 4u * (lh * PT + wp * 32 + l32), waddr = lds0 + 4u * (K33 * PT + (wq * 32 + l32) * W33 + 20 * lh);
    for (int z = blockIdx.z * g.nz; z < (int)(blockIdx.z + 1) * g.nz; ++z) {
        const int kbeg = z * c.kchunk, kend = min(kbeg + c.kchunk, g.Ch * 9);
        const int step0 = kbeg / K33, nsteps = kend > kbeg ? (kend + K33 - 1) / K33 - step0 : 0;
        int ch_off = (step0 * 4 + wave) * plane4, k_row = step0 * K33 + wave * 9 - kbeg, w_off = step0 * wstep + q0 * W33 * 4;
        const unsigned krange = kend - kbeg;
        unsigned xdst = 0;                           // LDS bytes of the stage to load next
        auto load_part = [&](int part) {             // 0 .. 4
#pragma unroll
            for (int t = 2 * part; t < 2 * part + 2 && t < 9; ++t) {
                // (a product outside the range: past the end of the tensor, which is shorter than 2 GiB)
                const int soff = (unsigned)(k_row + t) < krange ? ch_off : 0x7ffffffc;
#pragma unroll
                for (int h = 0; h < PH; ++h)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrcX, (lds_ptr_t)((char*)smem + xdst + ((wave * 9 + t) * PT + h * 64) * 4), 4, tap[h][t], soff, 0, 0);
            }
            if (part < (WL + 3) / 4 && wave + 4 * part < WL)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrcW, (lds_ptr_t)((char*)smem + xdst + K33 * PT * 4 + (wave + 4 * part) * 1024), 16, lane * 16,
                                                         w_off + (wave + 4 * part) * 1024, 0, 0);
            if (part == 4) {
                ch_off += 4 * plane4;
                k_row += K33;
                w_off += wstep;
                xdst = xdst ? 0u : 4u * STAGE;
            }
        };

        auto k_loop = [&](auto livec) {
            constexpr bool LIVE = decltype(livec)::value;
            v4f fa[2];
            v2f fb[2][2], ta, tb;
            auto read_group = [&](auto gic, unsigned sb) {       // products 8 gi .. 8 gi + 7 (the last: 32 .. 35)
                constexpr int gi = decltype(gic)::value;
                if (!LIVE) return;
                if (gi < 4) {
                    lds_read128f<16 * gi>(fa[gi & 1], waddr + sb);
                    lds_read2st64f<8 * gi * U, (8 * gi + 2) * U>(fb[gi & 1][0], xaddr + sb);
                    lds_read2st64f<(8 * gi + 4) * U, (8 * gi + 6) * U>(fb[gi & 1][1], xaddr + sb);
                } else {
                    lds_read64f<64>(ta, waddr + sb);
                    lds_read2st64f<32 * U, 34 * U>(tb, xaddr + sb);
                }
            };
            auto wait_group = [&](int gi) {
                if (!LIVE) return;
                wait_lgkm<0>();
                if (gi < 4) {
                    tie(fa[gi & 1]);
                    tie(fb[gi & 1][0]);
                    tie(fb[gi & 1][1]);
                } else {
                    tie(ta);
                    tie(tb);
                }
                __builtin_amdgcn_sched_barrier(0);
            };
            unsigned sb = 0;
            int until = c.fold;
            for (int st = 0; st < nsteps; ++st) {
                const bool more = st + 1 < nsteps;
                wait_loads_and_barrier<0>();
                read_group(std::integral_constant<int, 0>{}, sb);
                auto group = [&](auto gic) {
                    constexpr int gi = decltype(gic)::value;
                    wait_group(gi);
                    read_group(std::integral_constant<int, gi + 1>{}, sb);
                    if (LIVE) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) acc.acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[gi & 1][j], fb[gi & 1][j >> 1][j & 1], acc.acc, 0, 0, 0);
                    }
                    if (more) load_part(gi);
                };
                group(std::integral_constant<int, 0>{});
                group(std::integral_constant<int, 1>{});
                group(std::integral_constant<int, 2>{});
                group(std::integral_constant<int, 3>{});
                wait_group(4);
                if (LIVE) {
#pragma unroll
                    for (int j = 0; j < 2; ++j) acc.acc = __builtin_amdgcn_mfma_f32_32x32x2f32(ta[j], tb[j], acc.acc, 0, 0, 0);
                }
                if (more) load_part(4);
                sb = sb ? 0u : 4u * STAGE;
                if (LIVE && --until == 0) {
                    acc.fold();
                    until = c.fold;
                }
            }
        };
        if (nsteps > 0) {
#pragma unroll
            for (int part = 0; part < 5; ++part) load_part(part);
            if (q0 + wq * 32 < g.Q) k_loop(std::true_type{});
            else k_loop(std::false_type{});          // (rows past the last: only the loads)
        }
        if (g.nz > 1 || c.fold) {
            acc.fold();
            __syncthreads();                     // (the next range's loads go where slower waves may still read)
        }
    }
    if (g.nz > 1 || c.fold) acc.unfold();
    acc.store(g, c, p0 + wp * 32, q0 + wq * 32, lane, bias, beta, out, partial);
}

// A layer that spans its input, forward, in the reference's order of terms: y[b][o] = sum over k of x[b][k] w[o][k], one
// after the other in float.  The chain of additions is what takes the time: a wave alone on its SIMD issues one in 6 to 8 cycles, and
// every other instruction between two of them costs about as much.  Which kernel is the fastest depends on how many sums there are:
//  * Up to two waves a SIMD (32 sums a compute unit), conv_f32_chain_kernel<4>: a wave holds four sums, one to a row of 16 lanes.  The lanes
//    of a row multiply 64 terms, four each, straight from memory, and an addition takes its product out of the lane that has it by a broadcast
//    within the row: 64 additions for 4 multiplications and 2 loads, 2.5 ns a term.  With LDS between (the next kernel) 16 reads of
//    about 15 cycles each stood between 64 additions.
//  * Up to one block of 8 images x 8 outputs a compute unit, conv_f32_chain_kernel<64>: a lane holds a sum, and everything but the additions
//    is kept off the wave that does them.  Two waves load the operands, two stages of 256 terms ahead, multiply them, 64 terms of 128 each, and
//    leave the products in LDS; the third reads those a step later and only adds, 5.5 ns a term.  (Steps of 64 terms: 95 us where
//    this takes 90.)
//  * More, conv_f32_chain_wave_kernel: one wave multiplies and adds 64 sums, 7.1 ns a term, but its 49 KB let three blocks share a unit
//    where the other kernel's 115 KB let one.
// us, conv_f32_chain_kernel<4> / <64> (images x outputs, terms): 64 x 10, 16384 41.7 / 88.9; 64 x 10, 1024 4.5 / 7.5; 32 x 120, 400 4.0 / 5.5;
// 32 x 84, 120 4.0 / 4.0; 40 x 100, 25088 63.5 / 139; 64 x 64, 4096 13.0 / 23.7; 64 x 100 21.0 / 24.0; 64 x 128 21.0 / 23.8; 96 x 120
// 29.0 / 24.0; 40 x 400, 25088 196 / 140.
// us, conv_f32_chain_kernel<64> / conv_f32_chain_wave_kernel (images x outputs, blocks, terms): 40 x 400,
// 250, 25088 140.5 / 178.1; 128 x 120, 240, 400 5.8 / 5.4; 144 x 120, 270, 400 9.7 / 5.8; 192 x 96, 288, 1024 13.7 / 10.4; 48 x 400, 300,
// 25088 272.5 / 198.7; 256 x 120, 480, 400 9.9 / 5.9; 64 x 1000, 1000, 25088 552.5 / 381.1; 1024 x 120, 1920, 400 35.0 / 14.5.
constexpr int CHAIN_K = 256, CHAIN_ROW = CHAIN_K + 4, CHAIN_STAGES = 3;      // (rows 16 bytes apart in the banks)
constexpr int CHAIN_T = 128, CHAIN_PROD = CHAIN_T + 4;                        // terms between two barriers; a lane's row of products

// 32 terms of an image's row and of an output's, from OFF bytes on
template <int OFF>
__device__ __forceinline__ void chain_read(v4f (&xv)[8], v4f (&wv)[8], unsigned xa, unsigned wa)
{
    lds_read128f<OFF>(xv[0], xa); lds_read128f<OFF>(wv[0], wa);
    lds_read128f<OFF + 16>(xv[1], xa); lds_read128f<OFF + 16>(wv[1], wa);
    lds_read128f<OFF + 32>(xv[2], xa); lds_read128f<OFF + 32>(wv[2], wa);
    lds_read128f<OFF + 48>(xv[3], xa); lds_read128f<OFF + 48>(wv[3], wa);
    lds_read128f<OFF + 64>(xv[4], xa); lds_read128f<OFF + 64>(wv[4], wa);
    lds_read128f<OFF + 80>(xv[5], xa); lds_read128f<OFF + 80>(wv[5], wa);
    lds_read128f<OFF + 96>(xv[6], xa); lds_read128f<OFF + 96>(wv[6], wa);
    lds_read128f<OFF + 112>(xv[7], xa); lds_read128f<OFF + 112>(wv[7], wa);
}
// (The SAT quantizer that follows on the way out, a: its |alpha|.  32 x 84 and 32 x 10 sums: 2.9 + 2.6 and 2.6 + 1.9 us in two kernels each, 3.7 and
// 3.1 in one.)
__device__ __forceinline__ void chain_store(int B, int O, int b, int o, float sum, const float* __restrict__ bias, float beta, const SatStore& sat, float a,
                                            float* __restrict__ y)
{
    if (b >= B || o >= O) return;
    const size_t idx = (size_t)b * O + o;
    float r = sum + (beta != 0.0f ? beta * y[idx] : 0.0f);
    if (bias) r = bias[o] + r;
    if (sat.alpha) {
        if (sat.fp) sat.fp[idx] = r;
        r = sat_quantize(r, sat.range, a);
    }
    y[idx] = r;
}

// The products of a row's 16 lanes, four each, one after the other: each addition takes a lane's for the whole row.  (In assembly:
// the compiler puts a wait before each, as if the lanes' operand had just been written.)
#define N2D2HIP_CHAIN_LANE(I)                                                                                                   \
    "v_add_f32_dpp %0, %1, %0 row_newbcast:" #I " row_mask:0xf bank_mask:0xf\n\tv_add_f32_dpp %0, %2, %0 row_newbcast:" #I     \
    " row_mask:0xf bank_mask:0xf\n\tv_add_f32_dpp %0, %3, %0 row_newbcast:" #I " row_mask:0xf bank_mask:0xf\n\t"              \
    "v_add_f32_dpp %0, %4, %0 row_newbcast:" #I " row_mask:0xf bank_mask:0xf\n\t"
__device__ __forceinline__ void chain_add_row(float& sum, const v4f& p)
{
    const float p0 = p[0], p1 = p[1], p2 = p[2], p3 = p[3];
    asm volatile("s_nop 1\n\t" N2D2HIP_CHAIN_LANE(0) N2D2HIP_CHAIN_LANE(1) N2D2HIP_CHAIN_LANE(2) N2D2HIP_CHAIN_LANE(3) N2D2HIP_CHAIN_LANE(4)
                 N2D2HIP_CHAIN_LANE(5) N2D2HIP_CHAIN_LANE(6) N2D2HIP_CHAIN_LANE(7) N2D2HIP_CHAIN_LANE(8) N2D2HIP_CHAIN_LANE(9)
                 N2D2HIP_CHAIN_LANE(10) N2D2HIP_CHAIN_LANE(11) N2D2HIP_CHAIN_LANE(12) N2D2HIP_CHAIN_LANE(13) N2D2HIP_CHAIN_LANE(14)
                 N2D2HIP_CHAIN_LANE(15)
                 : "+&v"(sum) : "v"(p0), "v"(p1), "v"(p2), "v"(p3));
}
// The first `lanes` lanes' products
__device__ __forceinline__ void chain_add_lanes(float& sum, const v4f& p, int lanes)
{
    const float p0 = p[0], p1 = p[1], p2 = p[2], p3 = p[3];
#define N2D2HIP_CHAIN_ONE(I) if (lanes > I) asm volatile("s_nop 1\n\t" N2D2HIP_CHAIN_LANE(I) : "+&v"(sum) : "v"(p0), "v"(p1), "v"(p2), "v"(p3))
    N2D2HIP_CHAIN_ONE(0); N2D2HIP_CHAIN_ONE(1); N2D2HIP_CHAIN_ONE(2); N2D2HIP_CHAIN_ONE(3); N2D2HIP_CHAIN_ONE(4);
    N2D2HIP_CHAIN_ONE(5); N2D2HIP_CHAIN_ONE(6); N2D2HIP_CHAIN_ONE(7); N2D2HIP_CHAIN_ONE(8); N2D2HIP_CHAIN_ONE(9);
    N2D2HIP_CHAIN_ONE(10); N2D2HIP_CHAIN_ONE(11); N2D2HIP_CHAIN_ONE(12); N2D2HIP_CHAIN_ONE(13); N2D2HIP_CHAIN_ONE(14);
#undef N2D2HIP_CHAIN_ONE
}
#undef N2D2HIP_CHAIN_LANE
// (SUMS: of a work-group; the two have nothing but the name in common)
template <int SUMS>
__global__ void conv_f32_chain_kernel(int B, int O, int K, const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias, float beta,
                                      SatStore sat, float* __restrict__ y);
template <>
__global__ __launch_bounds__(64) void conv_f32_chain_kernel<4>(int B, int O, int K, const float* __restrict__ x, const float* __restrict__ w,
                                                               const float* __restrict__ bias, float beta, SatStore sat, float* __restrict__ y)
{
    const float a = sat.alpha ? fabsf(sat.alpha[0]) : 0.0f;
    constexpr int D = 8;                         // groups of 64 terms requested ahead
    const int lane = threadIdx.x, li = lane & 15, bi = lane >> 5, oi = lane >> 4 & 1, b0 = blockIdx.x * 2, o0 = blockIdx.y * 2;
    const __amdgpu_buffer_rsrc_t rsrcX = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(x + (size_t)b0 * K), 0, min(2, B - b0) * K * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrcW = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(w + (size_t)o0 * K), 0, min(2, O - o0) * K * 4, 0x00020000);
    const int xoff = (bi * K + li * 4) * 4, woff = (oi * K + li * 4) * 4;
    v4f xv[D], wv[D];
    float sum = 0.0f;
    // (terms past a row: of the next row, or zeros; rows past the last: zeros; not used)
    const auto load = [&](v4f& xr, v4f& wr, int group) {
        xr = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rsrcX, xoff, group * 256, 0));
        wr = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rsrcW, woff, group * 256, 0));
    };
    const int full = K / 64, rest = K % 64 / 4;
#pragma unroll
    for (int u = 0; u < D; ++u) load(xv[u], wv[u], u);
    int g = 0;
    for (; g + D <= full; g += D) {
#pragma unroll
        for (int u = 0; u < D; ++u) {
            tie(xv[u]); tie(wv[u]);
            const v4f p = wv[u] * xv[u];
            load(xv[u], wv[u], g + D + u);
            __builtin_amdgcn_sched_barrier(0);
            chain_add_row(sum, p);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int u = 0; u < D; ++u) {
        if (g + u < full) chain_add_row(sum, wv[u] * xv[u]);
        else if (g + u == full) chain_add_lanes(sum, wv[u] * xv[u], rest);
    }
    if (li == 0) chain_store(B, O, b0 + bi, o0 + oi, sum, bias, beta, sat, a, y);
}

template <>
__global__ __launch_bounds__(192) void conv_f32_chain_kernel<64>(int B, int O, int K, const float* __restrict__ x, const float* __restrict__ w,
                                                                 const float* __restrict__ bias, float beta, SatStore sat, float* __restrict__ y)
{
    const float a = sat.alpha ? fabsf(sat.alpha[0]) : 0.0f;
    __shared__ __attribute__((aligned(16))) float smem[CHAIN_STAGES * 16 * CHAIN_ROW + 2 * 64 * CHAIN_PROD];
    float* const products = smem + CHAIN_STAGES * 16 * CHAIN_ROW;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int bi = lane >> 3, oi = lane & 7, b0 = blockIdx.x * 8, o0 = blockIdx.y * 8;
    const int steps = (K + CHAIN_T - 1) / CHAIN_T;
    constexpr int PER_STAGE = CHAIN_K / CHAIN_T;
    // both sides pass barrier 0, ..., steps: step t multiplies between barriers t and t + 1 and is added between t + 1 and the next
    if (wave < 2) {
        // wave 0 loads the images' rows and wave 1 the outputs' (terms past a row: zeros, or of the next row; rows past the last: zeros)
        const float* const rows = wave ? w + (size_t)o0 * K : x + (size_t)b0 * K;
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(rows), 0, min(8, wave ? O - o0 : B - b0) * K * 4, 0x00020000);
        int soff = 0;
        unsigned dst = wave * 8u * CHAIN_ROW * 4u;
        auto load = [&]() {
#pragma unroll
            for (int r = 0; r < 8; ++r)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr_t)((char*)smem + dst + r * CHAIN_ROW * 4), 16, lane * 16, soff + r * K * 4, 0, 0);
            soff += CHAIN_K * 4;
            dst = dst >= (CHAIN_STAGES - 1) * 16u * CHAIN_ROW * 4u ? wave * 8u * CHAIN_ROW * 4u : dst + 16u * CHAIN_ROW * 4u;
        };
        const unsigned lds0 = (unsigned)(unsigned long)(__attribute__((address_space(3))) float*)smem;
        const unsigned first = lds0 + 2u * CHAIN_T * wave;       // this wave's terms of a step
        unsigned src = first;
        float* const out = products + lane * CHAIN_PROD + CHAIN_T / 2 * wave;
        load();
        load();
        wait_loads_and_barrier<8>();             // (barrier 0: the first stage is there)
        for (int t = 0; t < steps; ++t) {
            if (t % PER_STAGE == 0) load();      // where the stage before this one was, which both waves have read
            float* const to = out + (t & 1) * 64 * CHAIN_PROD;
            v4f xv[2][8], wv[2][8];
            const unsigned xa = src + 4u * bi * CHAIN_ROW, wa = src + 4u * (8 + oi) * CHAIN_ROW;
            chain_read<0>(xv[0], wv[0], xa, wa);
            wait_lgkm<0>();
#pragma unroll
            for (int i = 0; i < 8; ++i) { tie(xv[0][i]); tie(wv[0][i]); }
            chain_read<128>(xv[1], wv[1], xa, wa);
#pragma unroll
            for (int i = 0; i < 8; ++i) *(v4f*)(to + 4 * i) = wv[0][i] * xv[0][i];
            wait_lgkm<0>();
#pragma unroll
            for (int i = 0; i < 8; ++i) { tie(xv[1][i]); tie(wv[1][i]); *(v4f*)(to + 32 + 4 * i) = wv[1][i] * xv[1][i]; }
            src += 4u * CHAIN_T;
            if ((t + 1) % PER_STAGE == 0)
                src = t + 1 == PER_STAGE * CHAIN_STAGES * ((t + 1) / (PER_STAGE * CHAIN_STAGES)) ? first : src + 4u * (16 * CHAIN_ROW - CHAIN_K);
            if ((t + 1) % PER_STAGE == 0) asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");       // (the next stage is there)
            else asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        return;
    }
    float sum = 0.0f;
    const unsigned in = (unsigned)(unsigned long)(__attribute__((address_space(3))) float*)(products + lane * CHAIN_PROD);
    asm volatile("s_barrier" ::: "memory");
    for (int t = 0; t < steps; ++t) {
        asm volatile("s_barrier" ::: "memory");
        const unsigned from = in + (t & 1) * 4u * 64u * CHAIN_PROD;
        const int rest = K - t * CHAIN_T;
        // quarters of 32 products, each requested a quarter ahead; the first adds as its reads arrive
        v4f p[2][8];
        const auto read = [&](auto quarter) {
            constexpr int h = decltype(quarter)::value & 1, o = 128 * decltype(quarter)::value;
            lds_read128f<o>(p[h][0], from); lds_read128f<o + 16>(p[h][1], from);
            lds_read128f<o + 32>(p[h][2], from); lds_read128f<o + 48>(p[h][3], from);
            lds_read128f<o + 64>(p[h][4], from); lds_read128f<o + 80>(p[h][5], from);
            lds_read128f<o + 96>(p[h][6], from); lds_read128f<o + 112>(p[h][7], from);
        };
        const auto add = [&](auto quarter) {
            constexpr int h = decltype(quarter)::value & 1, k0 = 32 * decltype(quarter)::value;
#pragma unroll
            for (int i = 0; i < 8; ++i) tie(p[h][i]);
            if (rest >= k0 + 32) {
#pragma unroll
                for (int i = 0; i < 32; ++i) sum = sum + p[h][i >> 2][i & 3];
            } else {
#pragma unroll
                for (int i = 0; i < 31; ++i) sum = k0 + i < rest ? sum + p[h][i >> 2][i & 3] : sum;
            }
        };
        read(std::integral_constant<int, 0>{});
        read(std::integral_constant<int, 1>{});
        wait_lgkm<8>();
        add(std::integral_constant<int, 0>{});
        __builtin_amdgcn_sched_barrier(0);
        read(std::integral_constant<int, 2>{});
        wait_lgkm<8>();
        add(std::integral_constant<int, 1>{});
        __builtin_amdgcn_sched_barrier(0);
        read(std::integral_constant<int, 3>{});
        wait_lgkm<8>();
        add(std::integral_constant<int, 2>{});
        __builtin_amdgcn_sched_barrier(0);
        wait_lgkm<0>();
        add(std::integral_constant<int, 3>{});
        __builtin_amdgcn_sched_barrier(0);
    }
    chain_store(B, O, b0 + bi, o0 + oi, sum, bias, beta, sat, a, y);
}

__global__ __launch_bounds__(64) void conv_f32_chain_wave_kernel(int B, int O, int K, const float* __restrict__ x, const float* __restrict__ w,
                                                                 const float* __restrict__ bias, float beta, SatStore sat, float* __restrict__ y)
{
    const float a = sat.alpha ? fabsf(sat.alpha[0]) : 0.0f;
    __shared__ __attribute__((aligned(16))) float smem[CHAIN_STAGES * 16 * CHAIN_ROW];
    const int lane = threadIdx.x, bi = lane >> 3, oi = lane & 7, b0 = blockIdx.x * 8, o0 = blockIdx.y * 8;
    const __amdgpu_buffer_rsrc_t rsrcX = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(x + (size_t)b0 * K), 0, min(8, B - b0) * K * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrcW = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(w + (size_t)o0 * K), 0, min(8, O - o0) * K * 4, 0x00020000);
    int soff = 0;
    unsigned dst = 0;
    auto load = [&]() {                          // (terms past a row: zeros, or of the next row; rows past the last: zeros; not used)
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrcX, (lds_ptr_t)((char*)smem + dst + r * CHAIN_ROW * 4), 16, lane * 16, soff + r * K * 4, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrcW, (lds_ptr_t)((char*)smem + dst + (r + 8) * CHAIN_ROW * 4), 16, lane * 16, soff + r * K * 4, 0, 0);
        }
        soff += CHAIN_K * 4;
        dst = dst == (CHAIN_STAGES - 1) * 16u * CHAIN_ROW * 4u ? 0u : dst + 16u * CHAIN_ROW * 4u;
    };
    const unsigned lds0 = (unsigned)(unsigned long)(__attribute__((address_space(3))) float*)smem;
    const unsigned xrow = lds0 + 4u * bi * CHAIN_ROW, wrow = lds0 + 4u * (8 + oi) * CHAIN_ROW;
    const int full = K / 32, rest = K % 32, groups = full + (rest > 0);
    v4f xv[2][8], wv[2][8];                      // 32 terms each: those that are added, the next ones
    unsigned src = 0;
    float sum = 0.0f;
    auto group = [&](auto bufc, int h) {
        constexpr int buf = decltype(bufc)::value;
        wait_lgkm<0>();
#pragma unroll
        for (int i = 0; i < 8; ++i) { tie(xv[buf][i]); tie(wv[buf][i]); }
        if ((h & 7) == 7) {                      // the stage has been read: its place is free, and the next one is there
            wait_loads_and_barrier<16 * (CHAIN_STAGES - 2)>();
            load();
            src = src == (CHAIN_STAGES - 1) * 16u * CHAIN_ROW * 4u ? 0u : src + 16u * CHAIN_ROW * 4u;
        }
        const unsigned off = src + 128u * ((h + 1) & 7);
        if (h + 1 < groups) chain_read<0>(xv[1 - buf], wv[1 - buf], xrow + off, wrow + off);
        __builtin_amdgcn_sched_barrier(0);
        if (h < full) {
            float p[32];
#pragma unroll
            for (int i = 0; i < 32; ++i) p[i] = wv[buf][i >> 2][i & 3] * xv[buf][i >> 2][i & 3];
#pragma unroll
            for (int i = 0; i < 32; ++i) sum = sum + p[i];
        } else {
#pragma unroll
            for (int i = 0; i < 31; ++i) {
                const float t = sum + wv[buf][i >> 2][i & 3] * xv[buf][i >> 2][i & 3];
                sum = i < rest ? t : sum;
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int st = 0; st < CHAIN_STAGES; ++st) load();
    wait_loads_and_barrier<16 * (CHAIN_STAGES - 1)>();
    chain_read<0>(xv[0], wv[0], xrow, wrow);
    for (int h = 0; h < groups; h += 2) {
        group(std::integral_constant<int, 0>{}, h);
        if (h + 1 < groups) group(std::integral_constant<int, 1>{}, h + 1);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    chain_store(B, O, b0 + bi, o0 + oi, sum, bias, beta, sat, a, y);
}

// Forward (BWD = false) and backward-data with K in the tensors' own order, (channel, tap).
template <bool BWD, int WQ, int WP, int S, bool LONG>
__global__ __launch_bounds__(256) void conv_f32_pixel_kernel(PixelGemm g, const float* __restrict__ srcX, const float* __restrict__ srcW,
                                                             const float* __restrict__ bias, float beta, float* __restrict__ out, size_t partial)
{
    static_assert(WQ * WP == 4, "four waves");
    constexpr int QT = 32 * WQ, PT = 32 * WP;
    constexpr int PH = PT / 64;                  // loads per k row
    constexpr int WJ = QT / 16;                  // weight loads of a wave per step
    constexpr int LPI = 4 * PH + WJ;             // loads of a wave per step
    constexpr int STAGE = GK * PT + QT * GK;     // floats
    static_assert(LPI * (S - 1) < 60, "vmcnt is a 6-bit counter");
    __shared__ __attribute__((aligned(16))) float smem[S * STAGE];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wq = wave / WP, wp = wave % WP;
    int tile, qtile, ci;
    if (!pixel_tile(g, &tile, &qtile, &ci))
        return;
    const PixelClass& c = g.c[ci];
    const int p0 = (tile - c.tile0) * PT, q0 = qtile * QT;
    const int nT = c.nT, K = g.Ch * nT;
    const __amdgpu_buffer_rsrc_t rsrcX = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(srcX) - c.bias, 0, g.bytesX + 4u * c.bias, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrcW = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(srcW), 0, g.bytesW, 0x00020000);
    unsigned voff[PH], wbase[WJ];
    TapMask<LONG> mask[PH];
    const int fold = BWD ? c.fold : 0;           // (forward: ranges)
#pragma unroll
    for (int h = 0; h < PH; ++h)
        pixel_source(g, c, p0 + h * 64 + lane, &voff[h], &mask[h]);
    const int slot = ((lane & 15) >> 2) ^ wave, kk = 8 * (slot & 1) + 2 * (lane & 3) + (slot >> 1);    // this lane's k of a step in the weights
#pragma unroll
    for (int j = 0; j < WJ; ++j) {
        const int q = q0 + 4 * (wave + 4 * j) + (lane >> 4);
        wbase[j] = q < g.Q ? 4u * (unsigned)(q * g.qs) : F32_OOB;
    }
    // Tap t of this class lives in lane t; the running (channel, tap) of each of the wave's rows is scalar.
    const int tl = min(lane, max(nT - 1, 0)), ti = div_f32(tl, c.nxd), tj = tl - ti * c.nx;
    const int tap_off = 4 * (c.soff0 + ti * c.stepy + tj * c.stepx);
    const int tap_bit = LONG ? 0 : (1 << tj) | (1 << (c.nx + ti));
    PixelTile<PT> tl_acc;
    tl_acc.init((unsigned)(unsigned long)(__attribute__((address_space(3))) float*)smem, wq, wp, lane);
    for (int z = blockIdx.z * g.nz; z < (int)(blockIdx.z + 1) * g.nz; ++z) {
        const int kbeg = z * c.kchunk, kend = min(kbeg + c.kchunk, K);
        const int nsteps = kend > kbeg ? (kend - kbeg + GK - 1) / GK : 0;
        int row_t[4], row_ch[4];                     // row_ch: byte offset of the row's channel
        const int plane4 = g.planeS * 4, adv = nT > 0 ? div_f32(GK, c.nt) : 0, adv_t = nT > 0 ? GK - adv * nT : 0, adv_ch = adv * plane4;
        {
            int ch = nT > 0 ? div_f32(kbeg + wave * 4, c.nt) : 0, t = nT > 0 ? kbeg + wave * 4 - ch * nT : 0;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                row_t[r] = t; row_ch[r] = ch * plane4;
                if (++t >= nT) { t = 0; ++ch; }
            }
        }
        int row_left = kend - kbeg - wave * 4, wk = kbeg + kk;
        unsigned xdst = 0;                           // LDS bytes of the stage to load next
        auto load_part = [&](int part) {
            if (part < 4) {
                const int t = row_t[part];
                const int soff = row_ch[part] + __builtin_amdgcn_readlane(tap_off, t);
                const unsigned bit = tap_test<LONG>(t, tap_bit, row_left - 1 - part);
#pragma unroll
                for (int h = 0; h < PH; ++h)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrcX, (lds_ptr_t)((char*)smem + xdst + ((wave * 4 + part) * PT + h * 64) * 4), 4,
                                                             mask[h].inside(t, bit) ? voff[h] : F32_OOB, soff, 0, 0);
                const int tn = t + adv_t;
                const bool carry = tn >= nT;
                row_t[part] = carry ? tn - nT : tn;
                row_ch[part] += adv_ch + (carry ? plane4 : 0);
            } else {
                unsigned off = 4u * wk;
                if (BWD) {
                    const int ch = div_f32(wk, c.nt), t = wk - ch * nT;
                    const int i = div_f32(t, c.nxd), j = t - i * c.nx;
                    off = 4u * (ch * g.chs + (c.ty0 + i * g.osy) * g.kW + c.tx0 + j * g.osx);
                }
                const bool v = wk < kend;
#pragma unroll
                for (int j = 0; j < WJ; ++j)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrcW, (lds_ptr_t)((char*)smem + xdst + (GK * PT + (wave + 4 * j) * 64) * 4), 4,
                                                             v ? wbase[j] + off : F32_OOB, 0, 0, 0);
                wk += GK;
                row_left -= GK;
                xdst = xdst == 4u * STAGE * (S - 1) ? 0u : xdst + 4u * STAGE;
            }
        };

        if (nsteps > 0) {
#pragma unroll
            for (int st = 0; st < S - 1; ++st)       // (steps past the range load zeros: the number in flight stays the same)
#pragma unroll
                for (int part = 0; part < 5; ++part) load_part(part);
            auto k_loop = [&](auto live) {
                unsigned sb = 0;
                for (int st = 0; st < nsteps;) {
                    const int end = fold ? min(st + fold, nsteps) : nsteps;
                    for (; st < end; ++st) {
                        wait_loads_and_barrier<LPI*(S - 2)>();
                        tl_acc.template step<decltype(live)::value>(sb, load_part);
                        sb = sb == 4u * STAGE * (S - 1) ? 0u : sb + 4u * STAGE;
                    }
                    if (decltype(live)::value && fold) tl_acc.fold();      // (not in both loops: that doubles the registers)
                }
            };
            if (q0 + wq * 32 < g.Q) k_loop(std::true_type{});
            else k_loop(std::false_type{});          // (rows past the last: only the loads)
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        if (g.nz > 1 || fold) {
            tl_acc.fold();
            __syncthreads();                     // (the next range's loads go where slower waves may still read)
        }
    }
    if (g.nz > 1 || fold) tl_acc.unfold();
    tl_acc.store(g, c, p0 + wp * 32, q0 + wq * 32, lane, BWD ? nullptr : bias, beta, out, partial);
}

// Backward-filter: both operands hold consecutive k (pixels), rows of 32 of them in LDS, two rows to a load.  Row pairs are
// 272 bytes apart, so that 8 rows' 16-byte reads fall into different banks.
template <int WQ, int WP, int S, bool LONG, bool FOLD>
__global__ __launch_bounds__(256) void conv_f32_filter_kernel(FilterGemm g, const float* __restrict__ srcX, const float* __restrict__ srcY,
                                                              float* __restrict__ out)
{
    static_assert(WQ * WP == 4, "four waves");
    constexpr int QT = 32 * WQ, PT = 32 * WP;
    constexpr int PJ = PT / 8, QJ = QT / 8;      // loads of a wave per step (two rows each)
    constexpr int PAIR = 68;                     // floats from one row pair to the next
    constexpr int STAGE = (PT + QT) / 2 * PAIR;
    static_assert((PJ + QJ) * (S - 1) < 60, "vmcnt is a 6-bit counter");
    __shared__ __attribute__((aligned(16))) float smem[S * STAGE];
    const unsigned lds0 = (unsigned)(unsigned long)(__attribute__((address_space(3))) float*)smem;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, lh = lane >> 5;
    const int wq = wave / WP, wp = wave % WP;
    const int p0 = blockIdx.x * PT, q0 = blockIdx.y * QT;
    const int kbeg = blockIdx.z * g.kchunk, kend = min(kbeg + g.kchunk, g.K);
    const int nsteps = kend > kbeg ? (kend - kbeg + FK - 1) / FK : 0;
    const int xbias = g.pt * g.W + g.pl;
    const __amdgpu_buffer_rsrc_t rsrcX = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(srcX) - xbias, 0, g.bytesX + 4u * xbias, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrcY = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(srcY), 0, g.bytesY, 0x00020000);

    // ---- loader state: this lane's half of the row pairs its wave loads
    typedef std::conditional_t<LONG, unsigned long long, unsigned> Mask;
    unsigned poff[PJ], qoff[QJ];
    Mask pbit[PJ];
    const int kHW = g.kH * g.kW;
    const unsigned long long rows = LONG ? long_rows(g.kH, g.kW) : 0;
#pragma unroll
    for (int j = 0; j < PJ; ++j) {
        const int p = p0 + 2 * (wave + 4 * j) + lh, pp = min(p, g.P - 1);
        const int ch = pp / kHW, t = pp - ch * kHW, ty = t / g.kW, tx = t - ty * g.kW;
        poff[j] = 4u * (unsigned)(ch * g.H * g.W + ty * g.W + tx);
        if (LONG) pbit[j] = p < g.P ? (Mask)1 << t : 0;
        else pbit[j] = p < g.P ? (1u << tx) | (1u << (g.kW + ty)) : 0x80000000u;
    }
#pragma unroll
    for (int j = 0; j < QJ; ++j) {
        const int q = q0 + 2 * (wave + 4 * j) + lh;
        qoff[j] = q < g.Q ? 4u * (unsigned)(q * g.plane) : F32_OOB;
    }
    unsigned xo = 0, yo = 0, dst_bytes = 0;
    Mask pmask = 0;
    bool kv = false;
    int k_next = kbeg + l32;
    auto locate = [&]() {                        // this lane's pixel of the step to load next
        kv = k_next < kend;
        const int k = kv ? k_next : 0;
        const int img = div_f32(k, g.dplane), rem = k - img * g.plane;
        const int oy = div_f32(rem, g.dow), ox = rem - oy * g.oW;
        const int iy0 = oy * g.s_y - g.pt, ix0 = ox * g.s_x - g.pl;
        xo = 4u * (unsigned)(img * g.imgX + oy * g.s_y * g.W + ox * g.s_x);
        yo = 4u * (unsigned)(img * g.imgY + rem);
        // bits lo .. hi - 1 of the columns, then of the rows, that lie inside the input
        const int xl = min(max(-ix0, 0), g.kW), xh = min(max(g.W - ix0, 0), g.kW), yl = min(max(-iy0, 0), g.kH), yh = min(max(g.H - iy0, 0), g.kH);
        if (LONG) {
            pmask = kv ? (Mask)long_taps(xl, xh, yl, yh, g.kW, rows) : 0;
        } else {
            const unsigned mx = ((1u << xh) - 1u) & ~((1u << xl) - 1u), my = ((1u << yh) - 1u) & ~((1u << yl) - 1u);
            pmask = kv ? (Mask)(mx | (my << g.kW)) : 0;
        }
        k_next += FK;
    };
    auto issue_part = [&](int part) {            // a quarter of a stage's loads
#pragma unroll
        for (int j = part * PJ / 4; j < (part + 1) * PJ / 4; ++j)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrcX, (lds_ptr_t)((char*)smem + dst_bytes + (wave + 4 * j) * PAIR * 4), 4,
                                                     (LONG ? (pmask & pbit[j]) != 0 : (pmask & pbit[j]) == pbit[j]) ? xo + poff[j] : F32_OOB, 0, 0, 0);
#pragma unroll
        for (int j = part * QJ / 4; j < (part + 1) * QJ / 4; ++j)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrcY, (lds_ptr_t)((char*)smem + dst_bytes + (PT / 2 + wave + 4 * j) * PAIR * 4), 4,
                                                     kv ? yo + qoff[j] : F32_OOB, 0, 0, 0);
        if (part == 3)
            dst_bytes = dst_bytes == 4u * STAGE * (S - 1) ? 0u : dst_bytes + 4u * STAGE;
    };

    v16f acc;
    double folded[16];                           // (FOLD)
#pragma unroll
    for (int r = 0; r < 16; ++r) { acc[r] = 0.0f; folded[r] = 0.0; }
    auto fold = [&]() {
#pragma unroll
        for (int r = 0; r < 16; ++r) { folded[r] += (double)acc[r]; acc[r] = 0.0f; }
    };

    // ---- fragments: group gi of a step: k = 4 (2 gi + lh) + 0..3
    const unsigned lrow = 4u * ((l32 >> 1) * PAIR + (l32 & 1) * 32) + 16u * lh;
    const unsigned paddr = lds0 + 4u * (wp * 16 * PAIR) + lrow, qaddr = lds0 + 4u * (PT / 2 * PAIR + wq * 16 * PAIR) + lrow;
    auto k_loop = [&](auto livec) {
        constexpr bool LIVE = decltype(livec)::value;
        v4f fa[2], fb[2];
        auto read_group = [&](auto gic, unsigned sb) {
            constexpr int gi = decltype(gic)::value;
            if (!LIVE) return;
            lds_read128f<32 * gi>(fa[gi & 1], qaddr + sb);
            lds_read128f<32 * gi>(fb[gi & 1], paddr + sb);
        };
        auto wait_group = [&](int gi) {
            if (!LIVE) return;
            wait_lgkm<0>();
            tie(fa[gi & 1]);
            tie(fb[gi & 1]);
            __builtin_amdgcn_sched_barrier(0);
        };
        auto mfma_group = [&](int gi) {
            if (!LIVE) return;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[gi & 1][j], fb[gi & 1][j], acc, 0, 0, 0);
        };
        unsigned sb = 0;
        for (int st = 0; st < nsteps;) {
            const int end = FOLD ? min(st + g.fold, nsteps) : nsteps;
            for (; st < end; ++st) {
                wait_loads_and_barrier<(PJ + QJ) * (S - 2)>();
                read_group(std::integral_constant<int, 0>{}, sb);
                locate();
                issue_part(0);
                wait_group(0);
                read_group(std::integral_constant<int, 1>{}, sb);
                mfma_group(0);
                issue_part(1);
                wait_group(1);
                read_group(std::integral_constant<int, 2>{}, sb);
                mfma_group(1);
                issue_part(2);
                wait_group(2);
                read_group(std::integral_constant<int, 3>{}, sb);
                mfma_group(2);
                issue_part(3);
                wait_group(3);
                mfma_group(3);
                sb = sb == 4u * STAGE * (S - 1) ? 0u : sb + 4u * STAGE;
            }
            if (FOLD && LIVE) fold();
        }
    };
    if (nsteps > 0) {
#pragma unroll
        for (int st = 0; st < S - 1; ++st) {
            locate();
#pragma unroll
            for (int part = 0; part < 4; ++part) issue_part(part);
        }
        if (p0 + wp * 32 < g.P && q0 + wq * 32 < g.Q) k_loop(std::true_type{});
        else k_loop(std::false_type{});          // (past the last column or row: only the loads)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }

    float* dst = out + (size_t)blockIdx.z * g.Q * g.P;
    const int p = p0 + wp * 32 + l32;
    if (p >= g.P) return;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int q = q0 + wq * 32 + 8 * (r >> 2) + 4 * lh + (r & 3);
        if (q < g.Q) dst[(size_t)q * g.P + p] = FOLD ? (float)(folded[r] + (double)acc[r]) : acc[r];
    }
}

// Backward-filter of small problems, and of spanning kernels of more than 64 taps (backward-data of spanning kernels of up to
// 64 as well, which is such a sum over the outputs), in double on the fp64 matrix cores (16 x 16 x 4): a block is a 16 x 16
// tile of dw and a range of pixels, dealt to its four waves 16 at a time; a lane takes four consecutive pixels of its row of q and of its
// column of p, one per matrix instruction.  Nothing here is near a rate: the time is that of the loads' latency and of two
// launches, so the range is as short as fills the chip, and the next 16 pixels are on their way while these are multiplied.
// Against one block per weight summing all pixels (32 images, 1 x 32 x 32 -> 6, 5x5): 46 -> 12 us; 16 -> 32 channels, 3x3 on
// 16 x 16: 50 -> 12 us.  Spanning layers, whose K is the batch: 16384 -> 10, 64 images: 211 -> 8.2 us; 20736 -> 64, 64 images:
// 1690 -> 22 (fp32 matrix instructions take 10, with four times the error of a sum in double: 1.4e-7 against 2.5e-8).
typedef double v4d __attribute__((ext_vector_type(4)));
// (WAVES: of the block, the first four take part)
template <int WAVES>
__device__ __forceinline__ void filter_small_tile(const FilterGemm& g, int tp, int tq, int range, const float* __restrict__ srcX, const float* __restrict__ srcY,
                                                  double* __restrict__ partial, float beta, float* __restrict__ out)
{
    __shared__ double red[4][256];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, row = lane & 15, kg = lane >> 4;
    const int p = tp * 16 + row, q = tq * 16 + row;
    const bool takes = WAVES == 4 || wave < 4;
    const int kbeg = range * g.kchunk, kend = takes ? min(kbeg + g.kchunk, g.K) : kbeg;
    const int kHW = g.kH * g.kW, pp = min(p, g.P - 1);
    const int ch = pp / kHW, t = pp - ch * kHW, ty = t / g.kW, tx = t - ty * g.kW;
    const float* xb = srcX + (size_t)ch * g.H * g.W;
    const float* yb = srcY + (size_t)min(q, g.Q - 1) * g.rowY;
    float a[2][4], b[2][4];
    auto load = [&](int k0, float (&av)[4], float (&bv)[4]) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = k0 + j;
            const bool kv = k < kend;
            const int kk = kv ? k : 0;
            const int img = div_f32(kk, g.dplane), rem = kk - img * g.plane;
            const int oy = div_f32(rem, g.dow), ox = rem - oy * g.oW;
            const int iy = oy * g.s_y - g.pt + ty, ix = ox * g.s_x - g.pl + tx;
            const bool v = kv && iy >= 0 && iy < g.H && ix >= 0 && ix < g.W;
            av[j] = kv ? yb[(size_t)img * g.imgY + rem] : 0.0f;
            bv[j] = v ? xb[(size_t)img * g.imgX + iy * g.W + ix] : 0.0f;
        }
    };
    v4d acc = {0.0, 0.0, 0.0, 0.0};
    int k0 = kbeg + wave * 16 + kg * 4;
    load(k0, a[0], b[0]);
    for (int s = kbeg + wave * 16; s < kend; s += 128) {
        load(k0 + 64, a[1], b[1]);
#pragma unroll
        for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a[0][j], (double)b[0][j], acc, 0, 0, 0);
        k0 += 128;
        load(k0, a[0], b[0]);
#pragma unroll
        for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a[1][j], (double)b[1][j], acc, 0, 0, 0);
    }
    // lane holds column p = lane % 16 and rows q = 4 r + lane / 16
#pragma unroll
    for (int r = 0; r < 4; ++r)
        if (takes) red[wave][(4 * r + kg) * 16 + row] = acc[r];
    __syncthreads();
    if (!takes) return;
    const int oq = tq * 16 + threadIdx.x / 16, op = tp * 16 + threadIdx.x % 16;
    if (oq >= g.Q || op >= g.P) return;
    const double v = ((red[0][threadIdx.x] + red[1][threadIdx.x]) + red[2][threadIdx.x]) + red[3][threadIdx.x];
    const size_t idx = (size_t)oq * g.P + op;
    if (partial) partial[(size_t)range * g.Q * g.P + idx] = v;
    else out[idx] = (float)v + (beta != 0.0f ? beta * out[idx] : 0.0f);
}
__global__ __launch_bounds__(256) void conv_f32_filter_small_kernel(FilterGemm g, const float* __restrict__ srcX, const float* __restrict__ srcY,
                                                                    double* __restrict__ partial, float beta, float* __restrict__ out)
{
    filter_small_tile<4>(g, blockIdx.x, blockIdx.y, blockIdx.z, srcX, srcY, partial, beta, out);
}
// Both gradients of a small spanning layer in one launch: two such products, of which neither reads what the other writes, and a launch
// each was what they took.  us, two launches / one: 84 <- 120, 32 images 8.4 / 4.5; 120 <- 16 x 5 x 5 8.3 / 4.6; 64 <- 512, 255 images
// 10.2 / 6.1.
struct SmallProduct {
    FilterGemm g;
    int ptiles;                                  // of 16 columns of p
    const float *srcX, *srcY;
    float beta;
    float* out;
};
struct SmallPair {
    SmallProduct of[2];
    unsigned first;                              // first block of the second
};
__global__ __launch_bounds__(256) void conv_f32_small_pair_kernel(const SmallPair a)
{
    const int k = blockIdx.x >= a.first;
    const SmallProduct& s = a.of[k];
    const int block = blockIdx.x - (k ? a.first : 0), tq = block / s.ptiles;
    filter_small_tile<4>(s.g, block - tq * s.ptiles, tq, 0, s.srcX, s.srcY, nullptr, s.beta, s.out);
}

// Backward-data of small problems, the same way: dx[c][pixel] adds w[o][c][tap] dy[o][the pixel that the tap reaches] over (o, tap)
// in double.  A block is 16 channels x 16 input pixels; its waves take 16 terms in turn.  Bound by the latency of its loads, a
// microsecond for each wave's two rounds of them: 8 waves where K is more than four waves take in two, 16 from 1025 terms; and where
// the tiles are more than the chip holds blocks, a tile to each wave.  Which pixel a tap reaches is worked out once for the tile
// (for every term: half as long again).  Beyond the range of the rule: 8 <- 512, 3x3, 7 x 7, K 4608 15.5 us on the pixel kernel and 29.1 on this; 8 <- 8,
// 3x3, 32 x 32, batch 64, 2.9e5 11.5 / 13.7.
// us, the pixel kernel with its ranges / this (error against 64 bits 1.4e-7, 2.5e-8):
//   6 <- 16, 5x5, 14 x 14, batch 32, K 400   14.1 /  6.8             16 <- 16, 3x3, 28 x 28, batch 8, K 144    12.0 /  4.6
//   8 <- 16, 3x3, 32 x 32, batch 16, K 144   12.0 /  5.8             64 <- 64, 3x3, 28 x 28, K 576             11.4 /  6.0
//   64 <- 64, 3x3 stride 2, 14 x 14, batch 4 10.3 /  6.0             256 <- 256, 3x3, 7 x 7, K 2304            20.1 / 14.9
//   477 <- 11, 1x1 stride 2, 17 x 78, batch 7, 17430 tiles 12.1 / 12.0 (four waves to a tile 28.0)
//   121 <- 13, 1x1, 26 x 36, batch 31, 14512 tiles 10.3 / 10.1 (23.3)
struct DataSmall {
    int P, C, O, T, K;                           // input pixels over all images; taps; O * T
    int kW, HW, W, oH, oW, sy, sx, pt, pl;
    unsigned bytesW, bytesY;
    DivF32 dHW, dW, dT, dkW, dsy, dsx;
};
// (TILES: a block's, 1, or one to each of its waves, which then takes all of K; `tp` is the first)
template <int WAVES, int TILES>
__device__ __forceinline__ void data_small_tile(const DataSmall& g, int tp, int tc, const float* __restrict__ w, const float* __restrict__ dy, float beta,
                                                float* __restrict__ dx)
{
    static_assert(TILES == 1 || TILES == WAVES, "a tile of the block or of a wave");
    constexpr int SHARE = WAVES / TILES;         // waves of a tile
    __shared__ double red[TILES == 1 ? WAVES : 1][256];
    __shared__ int reach_of[TILES][64 * 16];     // where in a channel's image a pixel's tap is; -1: outside
    const int lane = threadIdx.x & 63, wave = TILES == 1 ? threadIdx.x >> 6 : 0, row = lane & 15, kg = lane >> 4;
    int* const reach = reach_of[TILES == 1 ? 0 : threadIdx.x >> 6];
    if (TILES > 1) tp += threadIdx.x >> 6;
    const __amdgpu_buffer_rsrc_t rsrcW = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(w), 0, g.bytesW, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrcY = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(dy), 0, g.bytesY, 0x00020000);
    const int c = tc * 16 + row, plane = g.oH * g.oW, p = min(tp * 16 + row, g.P - 1), img = div_f32(p, g.dHW);
    {
        const int rem = p - img * g.HW, iy = div_f32(rem, g.dW), ix = rem - iy * g.W;
        for (int t = TILES == 1 ? threadIdx.x >> 4 : kg; t < g.T; t += 4 * SHARE) {
            const int ty = div_f32(t, g.dkW), y = iy + g.pt - ty, x = ix + g.pl - (t - ty * g.kW);
            const int oy = div_f32(max(y, 0), g.dsy), ox = div_f32(max(x, 0), g.dsx);
            reach[t * 16 + row] = y >= 0 && x >= 0 && oy * g.sy == y && ox * g.sx == x && oy < g.oH && ox < g.oW ? oy * g.oW + ox : -1;
        }
    }
    __syncthreads();
    float a[2][4], b[2][4];
    const int adv_o = div_f32(16 * SHARE, g.dT), adv_t = 16 * SHARE - adv_o * g.T;
    int ko = div_f32(wave * 16 + kg * 4, g.dT), kt = wave * 16 + kg * 4 - ko * g.T;     // this lane's next term
    auto load = [&](float (&av)[4], float (&bv)[4]) {
        int o = ko, t = kt;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int at = o < g.O ? reach[t * 16 + row] : -1;
            av[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrcW, o < g.O && c < g.C ? 4u * (unsigned)((o * g.C + c) * g.T + t) : F32_OOB, 0, 0));
            bv[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrcY, at >= 0 ? 4u * (unsigned)((img * g.O + o) * plane + at) : F32_OOB, 0, 0));
            if (++t == g.T) { t = 0; ++o; }
        }
        ko += adv_o;
        kt += adv_t;
        if (kt >= g.T) { kt -= g.T; ++ko; }
    };
    v4d acc = {0.0, 0.0, 0.0, 0.0};
    auto multiply = [&](const float (&av)[4], const float (&bv)[4]) {
#pragma unroll
        for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f64_16x16x4f64((double)av[j], (double)bv[j], acc, 0, 0, 0);
    };
    load(a[0], b[0]);
    for (int s = wave * 16; s < g.K; s += 32 * SHARE) {
        const bool second = s + 16 * SHARE < g.K;
        if (second) load(a[1], b[1]);
        multiply(a[0], b[0]);
        if (!second) break;
        load(a[0], b[0]);
        multiply(a[1], b[1]);
    }
    const auto store = [&](int oc, int op, double v) {
        if (oc >= g.C || op >= g.P) return;
        const int oi = div_f32(op, g.dHW);
        const size_t idx = ((size_t)oi * g.C + oc) * g.HW + (op - oi * g.HW);
        dx[idx] = (float)v + (beta != 0.0f ? beta * dx[idx] : 0.0f);
    };
    // lane holds column p = lane % 16 and rows c = 4 r + lane / 16
    if constexpr (TILES > 1) {
#pragma unroll
        for (int r = 0; r < 4; ++r) store(tc * 16 + 4 * r + kg, tp * 16 + row, acc[r]);
        return;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wave][(4 * r + kg) * 16 + row] = acc[r];
    __syncthreads();
    if (threadIdx.x >= 256) return;
    double v = red[0][threadIdx.x];
#pragma unroll
    for (int i = 1; i < (TILES == 1 ? WAVES : 1); ++i) v += red[i][threadIdx.x];
    store(tc * 16 + threadIdx.x / 16, tp * 16 + threadIdx.x % 16, v);
}
// (across: blocks along the pixels.  Those of both directions are in the grid's first: channels alone can be more than 16 x 65535)
template <int WAVES, int TILES>
__global__ __launch_bounds__(64 * WAVES) void conv_f32_data_small_kernel(DataSmall g, int across, const float* __restrict__ w, const float* __restrict__ dy,
                                                                         float beta, float* __restrict__ dx)
{
    const int tc = blockIdx.x / across;
    data_small_tile<WAVES, TILES>(g, (blockIdx.x - tc * across) * TILES, tc, w, dy, beta, dx);
}
// Both gradients of a small layer in one launch, the blocks of the data first, which take longer, then those of the weights, whose ranges
// are added by the launch that follows.  us, two launches / one, with the one that adds: 6 <- 16, 5x5, 14 x 14, batch 32 15.5 / 12.4; 64 <- 64,
// 3x3 stride 2, 14 x 14, batch 4 12.1 / 8.5; 8 <- 8, 3x3, 16 x 16, batch 2 11.3 / 7.4.
struct SmallBoth {
    DataSmall data;
    int across;                                  // the data's blocks along the pixels
    unsigned first;                              // first block of the weights'
    SmallProduct filter;
    int ftiles;                                  // tiles of a range
    const float *w, *dy;
    float beta;
    float* dx;
    double* partial;
};
template <int WAVES, int TILES>
__global__ __launch_bounds__(64 * WAVES) void conv_f32_small_both_kernel(const SmallBoth a)
{
    if (blockIdx.x < a.first) {
        const int tc = blockIdx.x / a.across;
        data_small_tile<WAVES, TILES>(a.data, (blockIdx.x - tc * a.across) * TILES, tc, a.w, a.dy, a.beta, a.dx);
    } else {
        const int block = blockIdx.x - a.first, range = block / a.ftiles, tile = block - range * a.ftiles, tq = tile / a.filter.ptiles;
        filter_small_tile<WAVES>(a.filter.g, tile - tq * a.filter.ptiles, tq, range, a.filter.srcX, a.filter.srcY, a.partial, a.filter.beta, a.filter.out);
    }
}

// out[i] = sum over the K ranges + beta * out[i] (+ bias of element i's channel, NCHW with `plane` pixels per channel and O
// channels).  A block adds 64 elements: each of its four waves a quarter of the ranges in double, in their order, then the
// four in order, so the result does not depend on timing.
template <class T>
__global__ __launch_bounds__(256) void conv_f32_reduce_partials_kernel(const T* __restrict__ partial, int splits, size_t n, float beta,
                                                                       float* __restrict__ out, const float* __restrict__ bias, int plane, int O)
{
    __shared__ double red[4][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int z0 = splits * w / 4, z1 = splits * (w + 1) / 4;
    for (size_t i0 = (size_t)blockIdx.x * 64; i0 < n; i0 += (size_t)gridDim.x * 64) {
        const size_t i = i0 + lane;
        double s = 0.0;
        if (i < n) {
            int z = z0;
            for (; z + 8 <= z1; z += 8) {
                T v[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) v[j] = partial[(size_t)(z + j) * n + i];
#pragma unroll
                for (int j = 0; j < 8; ++j) s += (double)v[j];
            }
            for (; z < z1; ++z) s += (double)partial[(size_t)z * n + i];
        }
        __syncthreads();
        red[w][lane] = s;
        __syncthreads();
        if (w == 0 && i < n) {
            const double t = ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
            float v = (float)t + (beta != 0.0f ? beta * out[i] : 0.0f);
            if (bias) v = bias[(i / plane) % O] + v;
            out[i] = v;
        }
    }
}

} // namespace n2d2hip
