// The first cells of a small network in one launch: convolutions with a handful of channels, the max poolings behind them
// and the fully-connected cells at the end (LeNet whole: conv, pool, conv, pool, three fully-connected cells).
//
// What bounds such a network is not arithmetic (0.42 million multiply-adds an image) but the chain of launches: five
// dependent ones of 3.5 - 9 us each on a few work-groups, 34 us for one image.  Every tensor between the cells is a few KB, so
// a work-group of 8 waves takes one image through all the cells with its tensors in LDS; what a cell hands to the next
// costs a barrier instead of a launch.  Each cell's output is also stored to its tensor, as the cells run in turn do (the
// stores wait for nobody), so a caller finds the same values everywhere.  LeNet, conversion of the bytes included: one image
// 33.9 -> 7.1 us, 256 images launched one by one 45.7 -> 11.2 us (the host's two calls).  Of a launch's 16000 cycles 4200 go by until the image
// and the weights are there, 2900 in the first convolution (6600 before its pixels went in pairs), and the other cells take 750 to 2200 each: a
// descriptor, a few dependent LDS reads and a barrier.  16 waves took as long (each pays for its cells' descriptors and set-up); so did
// the fully-connected weights requested four loads at a time behind the first cells (the compiler waits for them there), and the next
// cell's descriptor loaded a cell ahead (its registers are spilled).  With many images
// the cells' own launches fill the chip and overtake it: cells and run, us, 1024 images 56.4 and 35.3, 2048 82.2 and 66.2, 4096 130.1
// and 127.6, 6144 179.0 and 188.5, 8192 230.7 and 249.8, 16384 458 and 495 (n2d2hip_cell_run_pays).
//
//  * Convolutions run on the matrix cores, 16 channels x 16 pixels a tile (v_mfma_i32_16x16x64_i8): a lane's 16 bytes of K
//    are one tap of a 16-channel pixel, or four taps of a 4-channel pixel, read from LDS where they lie; the 16 x 16 tile
//    leaves less padding than 32 x 32 for 6 or 16 outputs, and the accumulators hold four consecutive channels of a pixel,
//    one dword of the output.
//  * Weight fragments and rescale tables of all cells lie in one image in memory, which goes to LDS by direct loads at the
//    start; the fully-connected weights (the bulk: 58 KB of LeNet's 61) go into registers then, and arrive while the
//    convolutions run: memory latency is met once, not once per cell.
//  * In a fully-connected cell a wave owns 16 outputs and its lanes a quarter of K each; the partial sums meet by lane
//    exchanges, so a cell costs one barrier.  All sums are 32-bit integers: the results are those of the separate launches.
#include <algorithm>
#include <cstring>
#include <type_traits>
#include <vector>

#include "common.h"
#include "conv_handle.hpp"
#include "conv_small.hpp"
#include "epilogue.hpp"
#include "fc_chain.hpp"
#include "mfma_util.hpp"

namespace n2d2hip {

enum { RUN_CELLS = 8, RUN_THREADS = 512, RUN_WAVES = RUN_THREADS / 64, RUN_LDS = 65536, RUN_TAB = 6 /* bias, a, b, c, d, e */ };

enum { RUN_CONV16, RUN_CONV16_PADDED, RUN_CONV4, RUN_CONV4_PADDED, RUN_POOL, RUN_POOL_PADDED, RUN_CONV4_PAIRS, RUN_CONV4_PAIRS_FAST };

// (What a wave needs before its first pixel is computed by the host as far as it goes: the scalar unit, too, issues one
// instruction a clock for all waves.)
struct RunCell {
    int op;                              // RUN_*; padded: some window reaches outside the input
    int H, W, OW, npix, out_cs;          // input size, output columns and pixels (RUN_CONV4_PAIRS: pairs of them), channel stride of the output
    int out_bytes;                       // of an image's output
    int in_off, out_off;                 // LDS offsets of the two tensors
    int sx, sy, px, py;                  // stride, padding
    unsigned ow_mul, ow_sh;              // p / OW == p * ow_mul >> ow_sh for every output pixel p, the product below 2^32
    int tap_off;                         // LDS offset of the taps: bytes from the window's origin, or (padded) row << 16 | column.  Convolution:
                                         // [K step][lane / 16], one (16 channels), four (4 channels) or two (pairs: of two columns) each; pooling: a multiple of 4
    int nk;                              // convolution: K steps of 64 bytes (16 channels: a multiple of 4); pooling: groups of 4 taps
    int hop_x;                           // columns between a pixel of a wave's tile and that of its next tile, less than OW
    int hop, wrap, last;                 // the same in bytes of the window's origin, what a step into the next row adds, the last pixel's origin
    int hop_y;                           // (padded) rows of the input; the column's step is hop_x * sx
    int w_off, tab_off;                  // LDS offsets of the weight fragments and of the tables ([6][32])
    int O, mblocks;                      // outputs, blocks of 16 of them
    int kind, lo, hi, relu;              // rescale
    unsigned fill, out_xor;
};

struct RunFc {
    int O, tab_off, store;
    int kind, lo, hi, relu;
};

// What does not change from call to call: the first bytes of the image in device memory.
struct RunPlan {
    RunCell cell[RUN_CELLS];
    RunFc fc[FC_CHAIN_MAX];
};

struct CellRunArgs {
    const signed char* in;               // B images, NHWC, channel stride in_cs
    const unsigned char* edge;           // or null: the network's byte planes, NCHW, from which `in` is written
    signed char* in_w;
    unsigned edge_xor;                   // what turns a byte of the planes into a stored byte
    int in_cs, C, H, W;
    int ncells;
    const signed char* blob;             // plan, weight fragments and tables, blob_bytes (a multiple of 1024) to LDS offset 0
    int blob_bytes;
    int in_off;                          // LDS offset of the image
    // fully-connected cells behind the others (0: none)
    int nfc, fc_off;                     // LDS offset of the first one's input
    int kper;                            // dwords of K of the first one that a lane multiplies
    int fc_w[FC_CHAIN_MAX];              // weights, from the blob's start: [wave][4 dwords of a lane's K][lane][4 dwords]
    int x_off;                           // LDS: vectors between the cells, [2][128] bytes
    void* out;
    int out_cs, out_dtype;
    signed char* outs[RUN_CELLS];
};

namespace {

__device__ __forceinline__ void barrier_lds()
{
    // (not __syncthreads(): the fully-connected weights on their way to registers and the outputs' stores need not wait)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// t: a channel's bias, a, b, c, d, e
__device__ __forceinline__ int run_rescale(const int* t, int kind, int lo, int hi, int relu, int v)
{
    v += t[0];
    if (kind == EPI_RAW)
        return epi_apply<EPI_RAW>(v, 0, 0, 0, 0, 0, lo, hi, relu);
    if (kind == EPI_I24)
        return epi_apply<EPI_I24>(v, t[1], t[2], t[3], t[4], t[5], lo, hi, 0);
    if (kind == EPI_I64)
        return epi_apply<EPI_I64>(v, t[1], t[2], t[3], 0, t[5], lo, hi, 0);
    return epi_apply<EPI_F32>(v, t[1], t[2], t[3], 0, 0, lo, hi, 0);
}

// a struct of words in memory that does not change while kernels run, read by scalar loads
template <class T>
__device__ __forceinline__ T scalar_load(const T __attribute__((address_space(4)))* p)
{
    static_assert(sizeof(T) % 4 == 0, "words");
    struct Words { int w[sizeof(T) / 4]; } v;
#pragma unroll
    for (unsigned i = 0; i < sizeof(T) / 4; ++i)
        v.w[i] = ((const int __attribute__((address_space(4)))*)p)[i];
    return __builtin_bit_cast(T, v);
}

// One output pixel of a tile: its number, its window's place and its column.
template <bool PADDED>
struct RunPixel {
    int pix, ox, iy0, ix0, origin;
    // to the pixel RUN_WAVES tiles on
    __device__ __forceinline__ void hop(const RunCell& c)
    {
        pix += RUN_WAVES * 16;
        ox += c.hop_x;
        const bool over = ox >= c.OW;
        ox -= over ? c.OW : 0;
        if (PADDED) {
            iy0 += c.hop_y + (over ? c.sy : 0);
            ix0 = __mul24(ox, c.sx) - c.px;
        } else {
            origin += c.hop + (over ? c.wrap : 0);
        }
    }
};

// Instructions, not memory, are what a convolution costs here (a compute unit issues one vector and one scalar instruction a
// clock for all its waves): the taps come from a table, a wave steps from pixel to pixel without dividing, the rescale of a
// lane's four channels stays in registers, and a wave takes two tiles at a time so that 8 waves hide the LDS's latency.
template <int CS, bool PADDED>
__device__ __forceinline__ void run_conv(const RunCell& c, signed char* out, unsigned char* smem, int wave, int lane)
{
    const int l16 = lane & 15, kg = lane >> 4;
    const int ntiles = (c.npix + 15) >> 4;
    const unsigned char* x = smem + c.in_off;
    const unsigned char* taps = smem + c.tap_off + kg * (CS == 4 ? 16 : 4);
    RunPixel<PADDED> first;
    first.pix = wave * 16 + l16;
    {
        const int pc = min(first.pix, c.npix - 1), oy = (int)(__umul24((unsigned)pc, c.ow_mul) >> c.ow_sh);
        first.ox = pc - __mul24(oy, c.OW);
        first.iy0 = __mul24(oy, c.sy) - c.py;
        first.ix0 = __mul24(first.ox, c.sx) - c.px;
        first.origin = (__mul24(first.iy0, c.W) + first.ix0) * CS;
    }
#pragma unroll 1
    for (int mb = 0; mb < c.mblocks; ++mb) {
        const unsigned char* wf = smem + c.w_off + mb * c.nk * 1024 + lane * 16;
        // the lane's four channels; past the last one the tables are zero
        const int ch = 16 * mb + 4 * kg;
        const int* tab = (const int*)(smem + c.tab_off) + ch;
        v4i tq[6];
#pragma unroll
        for (int r = 0; r < RUN_TAB; ++r)
            tq[r] = *(const v4i*)(tab + r * 32);
        // (the channels past the last output hold the stored 0)
        const int live = c.O - ch;
        const unsigned keep = live >= 4 ? 0xffffffffu : live <= 0 ? 0u : (1u << (8 * live)) - 1u;
        // N tiles: RUN_WAVES apart, their pixels in px
        auto tiles = [&](auto n, const RunPixel<PADDED>* px) {
            constexpr int N = decltype(n)::value;
            v4i acc[N];
            // a tap of pixel u's window; `in`: it lies inside the input
            auto address = [&](int u, int tap, bool& in) -> const unsigned char* {
                if (!PADDED) {
                    in = true;
                    return x + (min(px[u].origin, c.last) + tap);
                }
                const int iy = px[u].iy0 + (tap >> 16), ix = px[u].ix0 + (tap & 0xffff);
                in = (unsigned)iy < (unsigned)c.H && (unsigned)ix < (unsigned)c.W;
                return x + (in ? (__mul24(iy, c.W) + ix) * CS : 0);
            };
#pragma unroll
            for (int u = 0; u < N; ++u)
                acc[u] = tq[0];             // the bias
            if (CS == 16) {
                // four steps' reads in flight together (the steps past the last tap have zero weights)
#pragma unroll 1
                for (int s = 0; s < c.nk; s += 4) {
                    v4i p[N][4], w[4];
                    int tap[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        tap[i] = *(const int*)(taps + (s + i) * 16);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        w[i] = *(const v4i*)(wf + (s + i) * 1024);
#pragma unroll
                        for (int u = 0; u < N; ++u) {
                            bool in;
                            p[u][i] = *(const v4i*)address(u, tap[i], in);
                            if (PADDED && !in)
                                p[u][i] = v4i{(int)c.fill, (int)c.fill, (int)c.fill, (int)c.fill};
                        }
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int u = 0; u < N; ++u)
                            acc[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[i], p[u][i], acc[u], 0, 0, 0);
                }
            } else {
                // (a 5 x 5 window has two steps; both are read before the first multiplies)
                auto read = [&](int s, v4i* p) {
                    const v4i tap = *(const v4i*)(taps + s * 64);
#pragma unroll
                    for (int u = 0; u < N; ++u)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            bool in;
                            const int v = *(const int*)address(u, tap[i], in);
                            p[u][i] = in ? v : (int)c.fill;
                        }
                };
#pragma unroll 1
                for (int s = 0; s < c.nk; s += 2) {
                    const int s1 = min(s + 1, c.nk - 1);
                    v4i p0[N], p1[N];
                    const v4i w0 = *(const v4i*)(wf + s * 1024), w1 = *(const v4i*)(wf + s1 * 1024);
                    read(s, p0);
                    read(s1, p1);
#pragma unroll
                    for (int u = 0; u < N; ++u)
                        acc[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w0, p0[u], acc[u], 0, 0, 0);
                    if (s + 1 < c.nk) {
#pragma unroll
                        for (int u = 0; u < N; ++u)
                            acc[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w1, p1[u], acc[u], 0, 0, 0);
                    }
                }
            }
            // channels ch .. ch + 3 of the lane's pixels: one dword of the output each
#pragma unroll
            for (int u = 0; u < N; ++u) {
                int r[4];
                // (clamp_i32 on the accumulators: what assembly reads of a matrix instruction's result the compiler does not wait for)
                if (c.kind == EPI_I24) {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        r[i] = med3_i32((__mul24(clamp_i32(acc[u][i], tq[1][i], tq[2][i]), tq[3][i]) + tq[4][i]) >> tq[5][i], c.lo, c.hi);
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int tr[RUN_TAB] = {0, tq[1][i], tq[2][i], tq[3][i], tq[4][i], tq[5][i]};
                        r[i] = run_rescale(tr, c.kind, c.lo, c.hi, c.relu, acc[u][i]);
                    }
                }
                if (px[u].pix < c.npix && ch < c.out_cs) {
                    const unsigned v = (pack_bytes(r[0], r[1], r[2], r[3]) & keep) ^ c.out_xor;
                    const unsigned at = __umul24((unsigned)px[u].pix, (unsigned)c.out_cs) + (unsigned)ch;
                    *(unsigned*)(smem + c.out_off + at) = v;
                    *(unsigned*)(out + at) = v;
                }
            }
        };
        RunPixel<PADDED> px[2] = {first, first};
        int t = wave;
#pragma unroll 1
        for (; t + RUN_WAVES < ntiles; t += 2 * RUN_WAVES) {
            px[1] = px[0];
            px[1].hop(c);
            tiles(std::integral_constant<int, 2>(), px);
            px[0] = px[1];
            px[0].hop(c);
        }
        if (t < ntiles)
            tiles(std::integral_constant<int, 1>(), px);
    }
}

// A convolution of 4 channels to at most 8, whose windows lie inside the input: a tile's 16 rows are 8 outputs of a pixel and 8 of the one to its
// right.  Both windows together are one column (at stride 1) wider than one, which costs no K step where the taps did not fill theirs (5 x 5:
// 30 of 32), and half as many tiles are read, multiplied and rescaled, with no row of them for outputs that do not exist.  Pairs begin 8 bytes
// apart, so that a lane's 16 bytes of K are two reads of two columns each, and the weights of the first two steps stay in registers.
// Bound by the latencies of a tile's chain and by instruction issue: a wave has up to four tiles under way together, and what differs from
// network to network (the rescale's kind) is decided outside the tiles.  LeNet, one image, us: a pixel a column 8.39, pairs, two tiles
// at a time 7.71, four and FAST 7.25 (with the poolings' pixels a thread each, and the arguments asked for together, 7.1).
// FAST: two K steps, rescale EPI_I24
template <bool FAST>
__device__ __forceinline__ void run_conv_pairs(const RunCell& c, signed char* out, unsigned char* smem, int wave, int lane)
{
    const int l16 = lane & 15, kg = lane >> 4, half = kg >> 1, ch = 4 * (kg & 1);
    const int ntiles = (c.npix + 15) >> 4;
    const unsigned char* x = smem + c.in_off;
    const unsigned char* taps = smem + c.tap_off + kg * 8;
    const unsigned char* wf = smem + c.w_off + lane * 16;
    const int* tab = (const int*)(smem + c.tab_off) + ch;
    // (the host has them be an even number)
    const v4i w0 = *(const v4i*)wf, w1 = *(const v4i*)(wf + 1024);
    const v2i t0 = *(const v2i*)taps, t1 = *(const v2i*)(taps + 32);
    v4i tq[6];
#pragma unroll
    for (int r = 0; r < RUN_TAB; ++r)
        tq[r] = *(const v4i*)(tab + r * 32);
    const int live = c.O - ch;
    const unsigned keep = live >= 4 ? 0xffffffffu : live <= 0 ? 0u : (1u << (8 * live)) - 1u;
    RunPixel<false> px;
    px.pix = wave * 16 + l16;
    {
        const int pc = min(px.pix, c.npix - 1), oy = (int)(__umul24((unsigned)pc, c.ow_mul) >> c.ow_sh);
        px.ox = pc - __mul24(oy, c.OW);
        px.iy0 = px.ix0 = 0;
        px.origin = (__mul24(oy, __mul24(c.sy, c.W)) + __mul24(px.ox, c.sx)) * 4;
    }
    // N tiles, RUN_WAVES apart
    auto tiles = [&](auto n) {
        constexpr int N = decltype(n)::value;
        v4i acc[N], p0[N], p1[N];
        const unsigned char* at[N];
        int pix[N];
        auto read = [&](const unsigned char* from, v2i t) {
            const v2i a = *(const v2i*)(from + t[0]), b = *(const v2i*)(from + t[1]);
            return v4i{a[0], a[1], b[0], b[1]};
        };
#pragma unroll
        for (int u = 0; u < N; ++u) {
            at[u] = x + min(px.origin, c.last);
            pix[u] = px.pix;
            p0[u] = read(at[u], t0);
            p1[u] = read(at[u], t1);
            px.hop(c);
        }
#pragma unroll
        for (int u = 0; u < N; ++u)
            acc[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w0, p0[u], tq[0], 0, 0, 0);
#pragma unroll
        for (int u = 0; u < N; ++u)
            acc[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w1, p1[u], acc[u], 0, 0, 0);
        if (!FAST) {
#pragma unroll 1
            for (int s = 2; s < c.nk; ++s) {
                const v4i w = *(const v4i*)(wf + s * 1024);
                const v2i t = *(const v2i*)(taps + s * 32);
#pragma unroll
                for (int u = 0; u < N; ++u)
                    acc[u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w, read(at[u], t), acc[u], 0, 0, 0);
            }
        }
#pragma unroll
        for (int u = 0; u < N; ++u) {
            int r[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (FAST) {
                    r[i] = med3_i32((__mul24(clamp_i32(acc[u][i], tq[1][i], tq[2][i]), tq[3][i]) + tq[4][i]) >> tq[5][i], c.lo, c.hi);
                } else {
                    const int tr[RUN_TAB] = {0, tq[1][i], tq[2][i], tq[3][i], tq[4][i], tq[5][i]};
                    r[i] = run_rescale(tr, c.kind, c.lo, c.hi, c.relu, acc[u][i]);
                }
            }
            const unsigned v = (pack_bytes(r[0], r[1], r[2], r[3]) & keep) ^ c.out_xor;
            const unsigned to = __umul24((unsigned)(2 * pix[u] + half), (unsigned)c.out_cs);
            if (c.out_cs == 16) {
                // channels 0 .. 7 of a pixel in the lanes that have its first four, and 8 .. 15, which hold the stored 0, in the others
                const auto both = __builtin_amdgcn_permlane16_swap(v, v, false, false);
                const v2i w2 = ch ? v2i{(int)c.out_xor, (int)c.out_xor} : v2i{(int)both[0], (int)both[1]};
                if (pix[u] < c.npix) {
                    *(v2i*)(smem + c.out_off + to + 2 * ch) = w2;
                    *(v2i*)(out + to + 2 * ch) = w2;
                }
            } else if (pix[u] < c.npix && ch == 0) {
                *(unsigned*)(smem + c.out_off + to) = v;
                *(unsigned*)(out + to) = v;
            }
        }
    };
    for (int t = wave; t < ntiles; t += 4 * RUN_WAVES) {
        const int left = ntiles - t;
        if (left > 3 * RUN_WAVES) tiles(std::integral_constant<int, 4>());
        else if (left > 2 * RUN_WAVES) tiles(std::integral_constant<int, 3>());
        else if (left > RUN_WAVES) tiles(std::integral_constant<int, 2>());
        else tiles(std::integral_constant<int, 1>());
    }
}

// Max pooling, four channels a thread, four taps in flight.  A tap outside the input is replaced by the nearest one inside,
// which cannot change a maximum; the host knows that every window has one.
template <bool PADDED>
__device__ __forceinline__ void run_pool(const RunCell& c, signed char* out, unsigned char* smem, int tid)
{
    if (!PADDED && c.out_cs == 16 && c.nk == 1) {
        // (2 x 2 and the like, 16 channels: a pixel a thread, whose reads are four of 16 bytes in place of sixteen of four)
        const v4i tap = *(const v4i*)(smem + c.tap_off);
#pragma unroll 1
        for (int pix = tid; pix < c.npix; pix += RUN_THREADS) {
            const int oy = (int)(__umul24((unsigned)pix, c.ow_mul) >> c.ow_sh), ox = pix - __mul24(oy, c.OW);
            const unsigned char* origin = smem + c.in_off + ((__mul24(__mul24(oy, c.sy), c.W) + __mul24(ox, c.sx)) << 4);
            v4i w[4], v;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                w[j] = *(const v4i*)(origin + tap[j]);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                v2s me = as_v2s((int)((unsigned)w[0][k] << 8)), mo = as_v2s(w[0][k]);
#pragma unroll
                for (int j = 1; j < 4; ++j) {
                    me = __builtin_elementwise_max(me, as_v2s((int)((unsigned)w[j][k] << 8)));
                    mo = __builtin_elementwise_max(mo, as_v2s(w[j][k]));
                }
                v[k] = (int)((((unsigned)__builtin_bit_cast(int, me) >> 8) & 0x00FF00FFu) | ((unsigned)__builtin_bit_cast(int, mo) & 0xFF00FF00u));
            }
            *(v4i*)(smem + c.out_off + 16 * pix) = v;
            *(v4i*)(out + 16 * pix) = v;
        }
        return;
    }
    const int q = c.out_cs >> 2;                        // 1, 4 or 8
    const int qs = q == 1 ? 0 : q == 4 ? 2 : 3;
    const unsigned char* taps = smem + c.tap_off;
    const v4i tap0 = *(const v4i*)taps;
#pragma unroll 1
    for (int i = tid; i < c.npix * q; i += RUN_THREADS) {
        const int pix = i >> qs, ch = (i & (q - 1)) * 4;
        const int oy = (int)(__umul24((unsigned)pix, c.ow_mul) >> c.ow_sh), ox = pix - __mul24(oy, c.OW);
        const int x0 = __mul24(ox, c.sx) - c.px, y0 = __mul24(oy, c.sy) - c.py;
        const unsigned char* src = smem + c.in_off + ch;
        const unsigned char* origin = src + ((__mul24(y0, c.W) + x0) << (qs + 2));
        v2s me = splat_v2s(-32768), mo = splat_v2s(-32768);
        v4i tap = tap0;
#pragma unroll 1
        for (int k = 0;;) {
            unsigned w[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (PADDED) {
                    const int y = min(max(y0 + (tap[j] >> 16), 0), c.H - 1), x = min(max(x0 + (tap[j] & 0xffff), 0), c.W - 1);
                    w[j] = *(const unsigned*)(src + ((__mul24(y, c.W) + x) << (qs + 2)));
                } else {
                    w[j] = *(const unsigned*)(origin + tap[j]);
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                // a signed byte in the high half of each 16 bits: the 16-bit maximum orders them as bytes, whatever the low halves hold
                me = __builtin_elementwise_max(me, as_v2s((int)(w[j] << 8)));
                mo = __builtin_elementwise_max(mo, as_v2s((int)w[j]));
            }
            if (++k >= c.nk)
                break;
            tap = *(const v4i*)(taps + 16 * k);
        }
        const unsigned v = (((unsigned)__builtin_bit_cast(int, me) >> 8) & 0x00FF00FFu) | ((unsigned)__builtin_bit_cast(int, mo) & 0xFF00FF00u);
        *(unsigned*)(smem + c.out_off + 4 * i) = v;
        *(unsigned*)(out + 4 * i) = v;
    }
}

// The sum over the four lanes whose number agrees in the last four bits, in each of them.
__device__ __forceinline__ int sum_of_quarters(int v)
{
    const auto r16 = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
    v = (int)(r16[0] + r16[1]);
    const auto r32 = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
    return (int)(r32[0] + r32[1]);
}

// HELD: the first fully-connected cell has at most 512 inputs, and its weights wait in registers (more would push the
// convolutions' values out of theirs).
template <bool HELD>
__global__ __launch_bounds__(RUN_THREADS) void cell_run_kernel(const CellRunArgs q)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int b = blockIdx.x;
    // (what the first loads need of the arguments, asked for together: one after the other, each waits for the last)
    asm volatile("" ::"s"(q.in), "s"(q.edge), "s"(q.in_w), "s"(q.edge_xor), "s"(q.in_cs), "s"(q.C), "s"(q.H), "s"(q.W), "s"(q.blob), "s"(q.blob_bytes),
                 "s"(q.in_off), "s"(q.nfc), "s"(q.kper), "s"(q.fc_w[0]), "s"(q.fc_w[1]), "s"(q.fc_w[FC_CHAIN_MAX - 1]));
    // (the plan does not change while kernels run: scalar loads)
    const auto* plan = (const RunPlan __attribute__((address_space(4)))*)(unsigned long long)q.blob;
    // ---- the image, the convolutions' weights and all tables
    for (int c = wave; c < q.blob_bytes / 1024; c += RUN_WAVES)
        __builtin_amdgcn_global_load_lds((gbl_ptr_t)(q.blob + c * 1024 + lane * 16), (lds_ptr_t)(smem + c * 1024), 16, 0, 0);
    // The image: the loads of its first 2048 dwords are all under way before the first is stored, and those of the
    // fully-connected weights behind them.
    const int hw = q.H * q.W, words = q.edge ? hw : hw * (q.in_cs >> 2);
    unsigned* x0 = (unsigned*)(smem + q.in_off);
    const unsigned char* planes = q.edge + (q.edge ? (size_t)b * q.C * hw : 0);
    const unsigned* src = (const unsigned*)q.in + (size_t)b * words;
    unsigned* in_w = (unsigned*)q.in_w + (size_t)b * words;
    auto load_word = [&](int i) -> unsigned {
        if (!q.edge)
            return src[i];
        // the graph edge's conversion (at most 4 channels: one dword a pixel)
        unsigned v = planes[i];
        for (int ch = 1; ch < q.C; ++ch)
            v |= (unsigned)planes[ch * hw + i] << (8 * ch);
        return v;
    };
    auto keep_word = [&](int i, unsigned v) {
        v ^= q.edge_xor;
        x0[i] = v;
        if (q.edge)
            in_w[i] = v;            // its tensor
    };
    constexpr int AHEAD = 4;
    unsigned xw[AHEAD];
#pragma unroll
    for (int j = 0; j < AHEAD; ++j)
        xw[j] = load_word(min(tid + j * RUN_THREADS, words - 1));

    // The fully-connected weights of the wave's 16 outputs (a lane whose K is shorter than Q4 groups reads its last group again,
    // and skips it when its turn comes): 12 loads, which nothing waits for until then.
    constexpr int Q4 = HELD ? 8 : 16;
    v4i w0[Q4] = {}, wn[FC_CHAIN_MAX - 1][2] = {};
    auto load_first = [&]() {
        const v4i* w = (const v4i*)(q.blob + q.fc_w[0]) + (size_t)wave * (q.kper / 4) * 64 + lane;
#pragma unroll
        for (int j = 0; j < Q4; ++j)
            w0[j] = w[min(j, q.kper / 4 - 1) * 64];
    };
    if (q.nfc > 0) {
        if (HELD)
            load_first();
#pragma unroll
        for (int l = 1; l < FC_CHAIN_MAX; ++l)          // (a cell that is not there has the first one's weights)
#pragma unroll
            for (int j = 0; j < 2; ++j)
                wn[l - 1][j] = *((const v4i*)(q.blob + q.fc_w[l]) + (wave * 2 + j) * 64 + lane);
    }
    // What is read by scalar loads later on is touched here, a word of every 64 bytes, while the image is on its way (behind its loads:
    // ahead of them it held them up by a microsecond): the arguments lie in host memory, the plan in the device's, and each miss would
    // hold all waves up (2000 and 500 cycles).
    {
        constexpr int LINES = (sizeof(RunPlan) + 63) / 64;
        int touched = 0;
#pragma unroll
        for (int i = 0; i < LINES; i += RUN_WAVES)          // (each wave an eighth of the plan)
            touched |= ((const int __attribute__((address_space(4)))*)plan)[min(i + wave, LINES - 1) * 16];
        asm volatile("" ::"s"(touched), "s"(q.outs[0]), "s"(q.outs[RUN_CELLS - 1]), "s"(q.out), "s"(q.x_off), "s"(q.kper));
    }
#pragma unroll
    for (int j = 0; j < AHEAD; ++j)
        if (tid + j * RUN_THREADS < words)
            keep_word(tid + j * RUN_THREADS, xw[j]);
    for (int i = tid + AHEAD * RUN_THREADS; i < words; i += RUN_THREADS)
        keep_word(i, load_word(i));
    // Loads answer in order: with no more under way than the weights' number, the blob, requested before them, is in LDS
    // (whatever the stores do, which count too).
    if (q.nfc > 0)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(HELD ? Q4 + 4 : 4) : "memory");
    else
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    barrier_lds();

    for (int i = 0; i < q.ncells; ++i) {
        const RunCell c = scalar_load(&plan->cell[i]);
        signed char* out = q.outs[i] + (size_t)b * (unsigned)c.out_bytes;
        switch (c.op) {
        case RUN_CONV16: run_conv<16, false>(c, out, smem, wave, lane); break;
        case RUN_CONV16_PADDED: run_conv<16, true>(c, out, smem, wave, lane); break;
        case RUN_CONV4: run_conv<4, false>(c, out, smem, wave, lane); break;
        case RUN_CONV4_PADDED: run_conv<4, true>(c, out, smem, wave, lane); break;
        case RUN_CONV4_PAIRS: run_conv_pairs<false>(c, out, smem, wave, lane); break;
        case RUN_CONV4_PAIRS_FAST: run_conv_pairs<true>(c, out, smem, wave, lane); break;
        case RUN_POOL: run_pool<false>(c, out, smem, tid); break;
        default: run_pool<true>(c, out, smem, tid); break;
        }
        barrier_lds();
    }

    if (q.nfc == 0)
        return;
    const int o = wave * 16 + (lane & 15), grp = lane >> 4;
    RunFc fc[FC_CHAIN_MAX];
    int ft[FC_CHAIN_MAX][RUN_TAB];
#pragma unroll
    for (int l = 0; l < FC_CHAIN_MAX; ++l) {
        fc[l] = scalar_load(&plan->fc[l]);              // (the tables' offset is the first one's where there is no cell)
#pragma unroll
        for (int k = 0; k < RUN_TAB; ++k)
            ft[l][k] = ((const int*)(smem + fc[l].tab_off))[k * FC_CHAIN_O + o];
    }
    const unsigned char* x = smem + q.fc_off;
#pragma unroll
    for (int l = 0; l < FC_CHAIN_MAX; ++l) {
        if (l >= q.nfc)
            return;
        int acc = 0;
        if (l == 0) {
            if (!HELD)
                load_first();
            const v4i* xv = (const v4i*)(x + grp * q.kper * 4);        // (what lies past K meets zero weights)
#pragma unroll
            for (int j = 0; j < Q4; ++j)
                if (4 * j < q.kper) {
                    const v4i xj = xv[j];
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        acc = __builtin_amdgcn_sdot4(xj[i], w0[j][i], acc, false);
                }
        } else {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const v4i xj = *(const v4i*)(x + grp * 32 + j * 16);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    acc = __builtin_amdgcn_sdot4(xj[i], wn[l > 0 ? l - 1 : 0][j][i], acc, false);
            }
        }
        acc = sum_of_quarters(acc);
        unsigned char* nx = smem + q.x_off + (l & 1) * FC_CHAIN_O;
        if (grp == 0) {
            const bool live = o < fc[l].O;
            int v = 0;
            if (live)
                v = run_rescale(ft[l], fc[l].kind, fc[l].lo, fc[l].hi, fc[l].relu, acc);
            if (l + 1 == q.nfc) {
                if (live)
                    store_value(q.out, (size_t)b * q.out_cs + o, q.out_dtype, v);
            } else {
                nx[o] = live ? (unsigned char)(fc[l].store == N2D2HIP_U8B ? v - 128 : v) : (unsigned char)0;
            }
        }
        barrier_lds();
        x = nx;
    }
}

} // namespace
} // namespace n2d2hip

using namespace n2d2hip;

struct n2d2hip_cell_run_s {
    CellRunArgs a;                       // all but the tensors' pointers and the batch
    signed char* d_blob;
    int lds;
    bool long_fc;
    int ncells;                          // tensors the run writes: convolutions and poolings, then the fully-connected cells' output
    int in_dtype;
    struct { int C, H, W, cs, dtype; } out[RUN_CELLS + 1];
    int fc_kind;                         // rescale kind of the last fully-connected cell
    int fc_min, fc_max;
};

static unsigned stored_zero(int dtype) { return dtype == N2D2HIP_U8B ? 0x80808080u : 0u; }

extern "C" {

int n2d2hip_cell_run_destroy(n2d2hip_cell_run_t h)
{
    if (!h) return N2D2HIP_OK;
    if (h->d_blob) (void)hipFree(h->d_blob);
    delete h;
    return N2D2HIP_OK;
}

int n2d2hip_cell_run_create(int nb_cells, const n2d2hip_run_cell* cells, int H, int W, n2d2hip_cell_run_t* out)
{
    N2D2HIP_REQUIRE(cells && out && nb_cells > 0, N2D2HIP_ERR_INVALID, "cell_run_create: null argument");
    const bool has_fc = cells[nb_cells - 1].fcs != nullptr;
    const int n = nb_cells - (has_fc ? 1 : 0);
#define N2D2HIP_RUN_NEEDS(cond, what) N2D2HIP_REQUIRE(cond, N2D2HIP_ERR_UNSUPPORTED, "cell_run_create: %s", what)
    N2D2HIP_RUN_NEEDS(n >= 1 && n <= RUN_CELLS && cells[0].conv, "a run begins with a convolution and holds at most 8 convolutions and poolings");
    CellRunArgs a;
    RunPlan plan;
    memset(&a, 0, sizeof(a));
    memset(&plan, 0, sizeof(plan));
    std::vector<signed char> blob(round_up((int)sizeof(RunPlan), 16), 0);
    std::vector<unsigned> fcw[FC_CHAIN_MAX];
    n2d2hip_cell_run_s proto;
    memset(&proto, 0, sizeof(proto));
    auto put_table = [&](const n2d2hip_conv_s* c, int stride) -> int {
        std::vector<int> t((size_t)RUN_TAB * stride, 0);
        const n2d2hip_act_s* act = c->act;
        for (int o = 0; o < c->desc.O; ++o) {
            t[o] = c->hbias[o];
            if (act->args.kind != EPI_RAW)
                for (int r = 0; r < 5; ++r)
                    t[(size_t)(r + 1) * stride + o] = act->htab[(size_t)r * act->cpad + o];
        }
        const size_t off = blob.size();
        blob.resize(off + t.size() * sizeof(int));
        memcpy(blob.data() + off, t.data(), t.size() * sizeof(int));
        return (int)off;
    };
    int h = H, w = W, dtype = -1, cs = 0, ch = 0, lds = 0;
    int tensor_off[RUN_CELLS + 1];           // offsets among the tensors; the weights and tables come before them
    for (int i = 0; i < n; ++i) {
        RunCell& c = plan.cell[i];
        const n2d2hip_conv_s* cv = cells[i].conv;
        N2D2HIP_RUN_NEEDS((cv != nullptr) != (cells[i].pool != nullptr) && !cells[i].fcs, "each cell but the last is one convolution or one pooling");
        if (i == 0) {
            dtype = cv->in_dtype; ch = cv->desc.C; cs = cv->in_cs;
            N2D2HIP_REQUIRE(H > 0 && W > 0, N2D2HIP_ERR_INVALID, "cell_run_create: input of %d x %d", H, W);
            N2D2HIP_RUN_NEEDS((long long)H * W * cs <= RUN_LDS, "the input does not fit");
            a.in_cs = cs; a.C = ch; a.H = H; a.W = W;
            proto.in_dtype = dtype;
            tensor_off[0] = 0;
            lds = round_up(H * W * cs, 16);
        }
        c.H = h; c.W = w;
        int OH, OW, taps, kW, dy = 1, dx = 1, listed;
        bool padded, pairs = false;
        const int in_cs = cs;
        if (cv) {
            const n2d2hip_conv_desc& d = cv->desc;
            N2D2HIP_RUN_NEEDS(cv->d_wsmall && !cv->is_fc && !cv->sub_inner && !cv->sum && !cv->depthwise && d.groups <= 1 && cv->d_bias && cv->act,
                              "a convolution has more than 16 inputs, 32 outputs or 64 taps, 4-bit weights, groups or a folded sum");
            N2D2HIP_RUN_NEEDS(cv->in_dtype == dtype && (dtype == N2D2HIP_U8B || dtype == N2D2HIP_I8) && d.C == ch && cv->in_cs == cs && (cs == 4 || cs == 16),
                              "a convolution does not read what the cell before it writes");
            const int to = cells[i].out_dtype;
            N2D2HIP_RUN_NEEDS(cv->act->args.kind != EPI_RAW && (to == N2D2HIP_U8B || to == N2D2HIP_I8) && cv->act->min_out >= (to == N2D2HIP_I8 ? -128 : 0)
                                  && cv->act->max_out <= (to == N2D2HIP_I8 ? 127 : 255), "a convolution's output is no byte of its type");
            const int rc = n2d2hip_conv_out_dims(&d, h, w, &OH, &OW);
            if (rc != N2D2HIP_OK)
                return rc;
            c.sx = d.strideX; c.sy = d.strideY; c.px = d.padL; c.py = d.padT;
            taps = d.kW * d.kH; kW = d.kW; dy = d.dilY; dx = d.dilX;
            c.nk = cs == 16 ? round_up((taps + 3) / 4, 4) : (taps + 15) / 16;
            listed = c.nk * (cs == 4 ? 16 : 4);
            c.O = d.O; c.mblocks = (d.O + 15) / 16;
            padded = d.padL > 0 || d.padT > 0 || (OH - 1) * d.strideY - d.padT + (d.kH - 1) * d.dilY >= h || (OW - 1) * d.strideX - d.padL + (d.kW - 1) * d.dilX >= w;
            // two columns of a window to a read; the K steps of a pair are no more than those of two pixels
            const int columns = (d.kW + d.strideX + 1) / 2, pair_steps = round_up((d.kH * columns + 7) / 8, 2);
            pairs = cs == 4 && d.O <= 8 && !padded && OW % 2 == 0 && w % 2 == 0 && dy == 1 && dx == 1 && pair_steps <= 2 * c.nk;
            if (pairs) {
                c.nk = pair_steps;
                listed = c.nk * 8;
            }
            c.kind = cv->act->args.kind; c.lo = cv->act->args.lo; c.hi = cv->act->args.hi; c.relu = cv->act->args.relu;
            c.fill = stored_zero(dtype);
            // weights as matrix-core fragments: [block of 16 outputs][K step][lane][16 bytes], lane l output l % 16, bytes 16 * (l / 16) of the step
            const int rows = conv_small_rows(d.C, d.O, taps);
            const std::vector<signed char>& img = cv->hsmall;
            c.w_off = (int)blob.size();
            blob.resize(blob.size() + (size_t)c.mblocks * c.nk * 1024, 0);
            for (int mb = 0; mb < c.mblocks; ++mb)
                for (int s = 0; s < c.nk; ++s)
                    for (int l = 0; l < 64; ++l)
                        for (int k = 0; k < 16; ++k) {
                            int o = 16 * mb + (l & 15), kb = 64 * s + 16 * (l >> 4) + k, tap = kb / cs;
                            if (pairs) {        // (column 2 (tap / 2 % columns) + tap % 2 of the first pixel's window)
                                const int x = 2 * (tap / 2 % columns) + tap % 2 - (o >= 8 ? d.strideX : 0), y = tap / 2 / columns;
                                tap = y < d.kH && x >= 0 && x < d.kW ? y * d.kW + x : taps;
                                o &= 7;
                            }
                            if (o < d.O && tap < taps)
                                blob[(size_t)c.w_off + ((size_t)(mb * c.nk + s) * 64 + l) * 16 + k] = img[((size_t)tap * rows + o) * cs + kb % cs];
                        }
            c.tab_off = put_table(cv, 32);
            dtype = to;
            ch = d.O;
            cs = n2d2hip_nhwc_cs(d.O);
            c.out_xor = stored_zero(dtype);
        } else {
            const n2d2hip_pool_desc& p = *cells[i].pool;
            const int rc = n2d2hip_pool_out_dims(&p, h, w, &OH, &OW);
            if (rc != N2D2HIP_OK)
                return rc;
            N2D2HIP_RUN_NEEDS(p.pooling == N2D2HIP_POOL_MAX && p.padX < p.poolW && p.padY < p.poolH && (OW - 1) * p.strideX - p.padX < w
                                  && (OH - 1) * p.strideY - p.padY < h, "a pooling is not a maximum or has an empty window");
            N2D2HIP_RUN_NEEDS(cells[i].out_dtype == dtype, "a pooling keeps its input's type");
            c.sx = p.strideX; c.sy = p.strideY; c.px = p.padX; c.py = p.padY;
            taps = p.poolW * p.poolH; kW = p.poolW;
            c.nk = (taps + 3) / 4;
            listed = 4 * c.nk;
            padded = p.padX > 0 || p.padY > 0 || (OH - 1) * p.strideY + p.poolH > h || (OW - 1) * p.strideX + p.poolW > w;
        }
        N2D2HIP_RUN_NEEDS(cs == 4 || cs == 16 || cs == 32, "a tensor has more than 32 channels");
        N2D2HIP_RUN_NEEDS((long long)OH * OW * cs <= RUN_LDS, "a tensor does not fit");
        c.out_bytes = OH * OW * cs; c.out_cs = cs;
        const int columns_out = pairs ? OW / 2 : OW;
        if (pairs) c.sx *= 2;
        c.OW = columns_out; c.npix = OH * columns_out;
        c.op = pairs ? (c.nk == 2 && c.kind == EPI_I24 ? RUN_CONV4_PAIRS_FAST : RUN_CONV4_PAIRS) : (cv ? (in_cs == 16 ? RUN_CONV16 : RUN_CONV4) : RUN_POOL) + (padded ? 1 : 0);
        const int hop_y = RUN_WAVES * 16 / columns_out;
        c.hop_x = RUN_WAVES * 16 % columns_out;
        c.hop = (hop_y * c.sy * w + c.hop_x * c.sx) * in_cs;
        c.wrap = (c.sy * w - columns_out * c.sx) * in_cs;
        c.last = ((OH - 1) * c.sy * w + (columns_out - 1) * c.sx) * in_cs;
        c.hop_y = hop_y * c.sy;
        // K position (step, lane / 16, i) is tap 4 * step + lane / 16, or with 4 channels tap 16 * step + 4 * (lane / 16) + i; behind the
        // last tap it is listed again (a convolution has zero weights there, a maximum does not change)
        std::vector<int> tap(listed);
        for (int t = 0; t < listed; ++t) {
            int k = std::min(t, taps - 1), ty = k / kW * dy, tx = k % kW * dx;
            if (pairs) {            // (pairs of columns; behind the last one: of the last)
                const int columns = (kW + c.sx / 2 + 1) / 2;
                k = std::min(t, columns * (taps / kW) - 1); ty = k / columns; tx = 2 * (k % columns);
            }
            tap[t] = padded ? ty << 16 | tx : (ty * w + tx) * in_cs;
        }
        c.tap_off = (int)blob.size();
        blob.resize(blob.size() + round_up(listed * (int)sizeof(int), 16));
        memcpy(blob.data() + c.tap_off, tap.data(), tap.size() * sizeof(int));
        // (at most 16384 pixels: tried on every one of them)
        bool divides = false;
        for (c.ow_sh = 8; c.ow_sh <= 22 && !divides; ++c.ow_sh) {
            c.ow_mul = (1u << c.ow_sh) / (unsigned)c.OW + 1u;
            divides = (unsigned long long)c.ow_mul * (unsigned)c.npix < (1ull << 32);
            for (unsigned p = 0; p < (unsigned)c.npix && divides; ++p)
                divides = (p * c.ow_mul) >> c.ow_sh == p / (unsigned)c.OW;
        }
        --c.ow_sh;
        N2D2HIP_RUN_NEEDS(divides, "a tensor's rows do not divide");
        tensor_off[i + 1] = lds;
        lds += round_up(OH * OW * cs, 16);
        N2D2HIP_RUN_NEEDS(lds <= RUN_LDS, "the tensors do not fit");
        h = OH; w = OW;
        proto.out[i] = {ch, OH, OW, cs, dtype};
    }
    a.ncells = n;
    proto.ncells = n;
    if (has_fc) {
        n2d2hip_fc_chain_t f = cells[n].fcs;
        const n2d2hip_conv_s* first = f->fc[0];
        N2D2HIP_RUN_NEEDS(first->in_dtype == dtype && first->desc.C == ch && first->in_cs == cs && first->fcH == h && first->fcW == w && h * w * cs <= first->ktot,
                          "the fully-connected cells do not read what the cell before them writes");
        a.nfc = f->n;
        for (int l = 0; l < f->n; ++l) {
            const n2d2hip_conv_s* fc = f->fc[l];
            N2D2HIP_RUN_NEEDS(f->k4[l] <= (l == 0 ? FC_CHAIN_K4 : FC_CHAIN_O / 4), "a fully-connected cell behind the first has more than 128 inputs");
            const std::vector<unsigned>& wt = f->hwt[l];
            const int kper = l == 0 ? (f->k4[0] + 15) / 16 * 4 : 8;
            if (l == 0)
                a.kper = kper;
            std::vector<unsigned>& img = fcw[l];
            img.assign((size_t)FC_CHAIN_O * 4 * kper, 0u);
            for (int o = 0; o < FC_CHAIN_O; ++o)
                for (int k = 0; k < f->k4[l]; ++k) {
                    const int g = k / kper, j = k % kper;
                    img[(((size_t)(o / 16) * (kper / 4) + j / 4) * 64 + g * 16 + o % 16) * 4 + j % 4] = wt[(size_t)k * FC_CHAIN_O + o];
                }
            plan.fc[l] = {fc->desc.O, put_table(fc, FC_CHAIN_O), l + 1 < f->n ? f->fc[l + 1]->in_dtype : N2D2HIP_I32,
                          fc->act->args.kind, fc->act->args.lo, fc->act->args.hi, fc->act->args.relu};
        }
        const n2d2hip_conv_s* last = f->fc[f->n - 1];
        proto.out[n] = {last->desc.O, 1, 1, 0, -1};
        proto.ncells = n + 1;
        proto.fc_kind = last->act->args.kind; proto.fc_min = last->act->min_out; proto.fc_max = last->act->max_out;
    }
    blob.resize((blob.size() + 1023) / 1024 * 1024, 0);
    const int base = (int)blob.size();
    for (int i = 0; i < n; ++i) {
        plan.cell[i].in_off = base + tensor_off[i];
        plan.cell[i].out_off = base + tensor_off[i + 1];
    }
    a.in_off = base;
    a.blob_bytes = base;         // (the fully-connected weights behind it do not go to LDS)
    for (int l = 0; l < a.nfc; ++l) {
        a.fc_w[l] = (int)blob.size();
        blob.resize(blob.size() + fcw[l].size() * sizeof(unsigned));
        memcpy(blob.data() + a.fc_w[l], fcw[l].data(), fcw[l].size() * sizeof(unsigned));
    }
    for (int l = a.nfc; l < FC_CHAIN_MAX; ++l)
        { a.fc_w[l] = a.fc_w[0]; plan.fc[l] = plan.fc[0]; }
    memcpy(blob.data(), &plan, sizeof(plan));
    a.fc_off = base + tensor_off[n];
    if (has_fc) {
        // the first cell's lanes read whole runs of K: past the last tensor's own bytes
        lds = round_up(std::max(lds, tensor_off[n] + 4 * a.kper * 4), 16);
        a.x_off = base + lds;
        lds += 2 * FC_CHAIN_O;
    }
    lds += base;
    N2D2HIP_RUN_NEEDS(lds <= RUN_LDS, "tensors, weights and tables do not fit");
#undef N2D2HIP_RUN_NEEDS
    n2d2hip_cell_run_s* r = new n2d2hip_cell_run_s(proto);
    r->d_blob = nullptr;
    hipError_t e = hipMalloc((void**)&r->d_blob, blob.size());
    if (e == hipSuccess) e = hipMemcpy(r->d_blob, blob.data(), blob.size(), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        n2d2hip_cell_run_destroy(r);
        return fail(N2D2HIP_ERR_HIP, "cell_run_create: device upload failed: %s", hipGetErrorString(e));
    }
    a.blob = r->d_blob;
    r->a = a; r->lds = lds;
    r->long_fc = a.kper > 32;
    *out = r;
    return N2D2HIP_OK;
}

int n2d2hip_cell_run_pays(int images)
{
    return images > 0 && images <= 16 * num_cus() ? 1 : 0;       // (16 images one after the other on a compute unit: measured above)
}

int n2d2hip_cell_run_forward(n2d2hip_cell_run_t r, const n2d2hip_tensor* edge, const n2d2hip_tensor* in, const n2d2hip_tensor* outs, n2d2hip_stream_t stream)
{
    int rc;
    N2D2HIP_REQUIRE(r && outs, N2D2HIP_ERR_INVALID, "cell_run_forward: null argument");
    if ((rc = check_tensor(in, "cell_run input")))
        return rc;
    CellRunArgs a = r->a;
    N2D2HIP_REQUIRE(in->layout == N2D2HIP_NHWC && in->C == a.C && in->H == a.H && in->W == a.W && in->cs == a.in_cs && in->dtype == r->in_dtype,
                    N2D2HIP_ERR_INVALID, "cell_run_forward: input is %dx%dx%d (stride %d) of type %d, the run was built for %dx%dx%d (stride %d) of type %d",
                    in->C, in->H, in->W, in->cs, in->dtype, a.C, a.H, a.W, a.in_cs, r->in_dtype);
    a.in = (const signed char*)in->data;
    if (edge) {
        if ((rc = check_tensor(edge, "cell_run edge")))
            return rc;
        N2D2HIP_REQUIRE(edge->layout == N2D2HIP_NCHW && edge->B == in->B && edge->C == a.C && edge->H == a.H && edge->W == a.W && a.in_cs == 4
                            && edge->dtype == (in->dtype == N2D2HIP_U8B ? N2D2HIP_U8 : N2D2HIP_I8),
                        N2D2HIP_ERR_UNSUPPORTED, "cell_run_forward: the edge must be byte planes (NCHW) of the input's shape and signedness, at most 4 channels");
        a.edge = (const unsigned char*)edge->data;
        a.in_w = (signed char*)in->data;
        a.edge_xor = stored_zero(in->dtype);
    }
    for (int i = 0; i < r->ncells; ++i) {
        const n2d2hip_tensor* o = outs + i;
        if ((rc = check_tensor(o, "cell_run output")))
            return rc;
        const auto& want = r->out[i];
        N2D2HIP_REQUIRE(o->layout == N2D2HIP_NHWC && o->B == in->B && o->C == want.C && o->H == want.H && o->W == want.W, N2D2HIP_ERR_INVALID,
                        "cell_run_forward: output %d must be NHWC, %dx%dx%dx%d", i, in->B, want.C, want.H, want.W);
        if (i < a.ncells) {
            N2D2HIP_REQUIRE(o->cs == want.cs && o->dtype == want.dtype, N2D2HIP_ERR_INVALID,
                            "cell_run_forward: output %d must have type %d and channel stride %d", i, want.dtype, want.cs);
            a.outs[i] = (signed char*)o->data;
        } else {
            N2D2HIP_REQUIRE(o->dtype == N2D2HIP_I32 || (is_byte_type(o->dtype) && r->fc_kind != EPI_RAW && r->fc_min >= (o->dtype == N2D2HIP_I8 ? -128 : 0)
                                                        && r->fc_max <= (o->dtype == N2D2HIP_I8 ? 127 : 255)),
                            N2D2HIP_ERR_INVALID, "cell_run_forward: the last cell's range does not fit output type %d", o->dtype);
            a.out = o->data; a.out_cs = o->cs; a.out_dtype = o->dtype;
        }
    }
    const dim3 grid((unsigned)in->B);
    if (r->long_fc)
        N2D2HIP_LAUNCH_T(cell_run_kernel, (false), grid, dim3(RUN_THREADS), (unsigned)r->lds, (hipStream_t)stream, a);
    else
        N2D2HIP_LAUNCH_T(cell_run_kernel, (true), grid, dim3(RUN_THREADS), (unsigned)r->lds, (hipStream_t)stream, a);
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

} // extern "C"
