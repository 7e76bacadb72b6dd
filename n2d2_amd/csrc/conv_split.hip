// Implicit-GEMM convolution for layers with few output tiles and a long K: the deep stages of a network on one or a few
// images (7 x 7 and 14 x 14 pixels, 256 to 2048 channels).
//
// With 64 x 64 tiles such a layer is a few dozen work-groups, and each walks its K steps one behind the other: a step of the
// pipelined kernel takes about 640 cycles there, most of them the LDS's latency and a barrier between four waves that have
// their SIMDs to themselves (3 x 3, 512 -> 512, 7 x 7: 36 steps, 13 us on 32 of 256 compute units).  Here a work-group owns
// 32 pixels x 32 channels, so four times as many of them share the layer, and its waves share K: wave w takes
// every fourth step of 128 bytes through a ring of its own (direct loads to LDS, no barrier: a wave waits for its own
// loads only), so that four steps are under way at once.  At the end the partial sums, 32-bit integers, meet in LDS, and
// every thread finishes four channels of a pixel.  The same layer: 6.2 us.  Whole nets, us: ResNet-50 1 image 331 -> 239,
// 5 of 193 x 193 341 -> 280, 16 403 -> 391; ResNet-18 W4A4 1 image 188 -> 114, 16 214 -> 180; MobileNet 1 image 114 -> 106.
//
// Work-groups are dealt to the XCDs so that an XCD has a run of channel tiles: the weights, the larger operand here, pass
// through one XCD's L2 only.
#include "conv_split.hpp"

#include <algorithm>

namespace n2d2hip {

namespace {

// Four waves of two stages: eight of two, four of four (128 KB) and tiles of 64 pixels were nowhere ahead by more than 3 %.
constexpr int NW = 4, S = 2;               // waves, ring stages of a wave

// VALID, W4: as conv_pipe_kernel; RAW: no rescale
template <int VALID, bool W4, bool RAW>
__global__ __launch_bounds__(NW * 64) void conv_split_kernel(ConvPipeArgs q)
{
    const ConvArgs& p = q.c;
    constexpr int BK = 128, KH = BK / 32;
    constexpr int A_CH = 4, B_CH = W4 ? 2 : 4;             // 1 KB loads per stage: 8 rows of pixels or weights, or half a weight chunk
    constexpr int LPI = A_CH + B_CH;
    constexpr int STAGE = LPI * 1024;
    constexpr int RP = 36;                                 // ints per pixel of the partial sums: 32 and a pad that spreads the banks
    constexpr int ITEMS = 32 * 8 / (NW * 64);              // dwords of output per thread
    static_assert(NW * 32 * RP * 4 <= NW * S * STAGE, "the partial sums fit the rings");
    static_assert(LPI * (S - 1) < 60, "vmcnt is a 6-bit counter");
    __shared__ __attribute__((aligned(16))) unsigned char smem[NW * S * STAGE];
    const unsigned lds0 = (unsigned)(unsigned long)(__attribute__((address_space(3))) unsigned char*)smem;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, lh = lane >> 5;
    // blocks 8 apart run on the same XCD
    const int idx = (int)(blockIdx.x & 7) * q.mlanes + (int)(blockIdx.x >> 3);
    if (idx >= q.mtiles * p.ntiles_n)
        return;
    const int tile_n = div_magic(idx, q.xcd_mul, q.xcd_sh);
    const int m0 = (idx - tile_n * q.mtiles) * 32, n0 = tile_n * 32;

    // ---- loads: lane l of a 1 KB load fills 16-byte slot l, row l / 8; swz_k() places logical slots
    const int lrow = lane >> 3;
    int rowoff[A_CH];
    unsigned rowmask[VALID == 0 ? A_CH : 1];
#pragma unroll
    for (int j = 0; j < A_CH; ++j) {
        const int m = m0 + j * 8 + lrow;
        const int mm = m < p.M ? m : 0;                    // (rows past the end read like pixel 0 and are not stored)
        const int b = div_magic(mm, q.ohw_mul, q.ohw_sh);
        const int rem = mm - b * (p.OH * p.OW);
        const int oy = div_magic(rem, q.ow_mul, q.ow_sh);
        const int ox = rem - oy * p.OW;
        const int by = oy * p.strideY - p.padT, bx = ox * p.strideX - p.padL;
        rowoff[j] = ((b * p.H + by) * p.W + bx) * p.in_cs + (((lane & 7) ^ (((j & 1) << 2) | (lane >> 4))) << 4);
        if (VALID == 0) {
            unsigned xmask = 0u, mk = 0u;
            for (int kx = 0; kx < q.kW; ++kx)
                xmask |= (unsigned)((kx >= -bx) & (kx < p.W - bx)) << kx;
            for (int ky = 0; ky < q.kH; ++ky)
                mk |= ((ky >= -by) & (ky < p.H - by)) ? (xmask << (ky * q.kW)) : 0u;
            rowmask[VALID == 0 ? j : 0] = mk;
        }
    }
    unsigned woff[B_CH];
#pragma unroll
    for (int j = 0; j < B_CH; ++j)
        woff[j] = W4 ? (unsigned)(tile_n * p.niter * 2048 + j * 1024 + lane * 16)
                     : (unsigned)((n0 + j * 8 + lrow) * p.ktot + (((lane & 7) ^ (((j & 1) << 2) | (lane >> 4))) << 4));
    unsigned char* ring = smem + wave * (S * STAGE);
    auto issue = [&](int it, int slot) {
        unsigned char* base = ring + slot * STAGE;
        int toff = it * BK;
        unsigned tapbit = 1u;
        if (VALID != 1) {
            const int tap = div_magic(it, q.cper_mul, q.cper_sh);
            const int ky = (tap * q.kw_mul) >> 16, kx = tap - ky * q.kW;
            toff = (ky * p.W + kx) * p.in_cs + (it - tap * q.cper) * BK;
            tapbit = 1u << tap;
        }
#pragma unroll
        for (int j = 0; j < A_CH; ++j) {
            const signed char* src = p.in + toff + (long long)rowoff[j];
            if (VALID == 0)
                src = (rowmask[VALID == 0 ? j : 0] & tapbit) ? src : q.fill16;
            __builtin_amdgcn_global_load_lds((gbl_ptr_t)src, (lds_ptr_t)(base + j * 1024), 16, 0, 0);
        }
        const signed char* wbase = p.w + (W4 ? it * 2048 : it * BK);
#pragma unroll
        for (int j = 0; j < B_CH; ++j)
            __builtin_amdgcn_global_load_lds((gbl_ptr_t)(wbase + woff[j]), (lds_ptr_t)(base + (A_CH + j) * 1024), 16, 0, 0);
    };

    // ---- this wave's steps: wave, wave + NW, ...
    const int n = p.niter > wave ? (p.niter - wave + NW - 1) / NW : 0;
#pragma unroll
    for (int s = 0; s < S; ++s)
        if (s < n)
            issue(wave + s * NW, s);

    // ---- what the last part needs: its channels' tables and the other input's bytes, on their way behind the first steps
    const int ch = n0 + (tid & 7) * 4;
    int4 ta = {}, tb = {}, tc = {}, td = {}, te = {}, sa = {}, sb = {}, sc = {}, sd = {}, se = {}, xa = {}, xb = {}, xc = {}, xd = {}, xe = {};
    unsigned other[ITEMS];
    int pixel[ITEMS];                                      // place in the output buffer, -1: past the end
#pragma unroll
    for (int u = 0; u < ITEMS; ++u) {
        const int m = m0 + (tid >> 3) + u * (NW * 8);
        const int mm = m < p.M ? m : 0;
        const int b = div_magic(mm, q.ohw_mul, q.ohw_sh);
        const int rem = mm - b * (p.OH * p.OW);
        const int oy = div_magic(rem, q.ow_mul, q.ow_sh);
        const int ox = rem - oy * p.OW;
        auto place = [&](int halo) { return (b * (p.OH + 2 * halo) + oy + halo) * (p.OW + 2 * halo) + ox + halo; };
        pixel[u] = m < p.M && ch < p.out_cs ? place(q.out_halo) : -1;
        other[u] = 0u;
        if (!RAW && q.res && pixel[u] >= 0)
            other[u] = *(const unsigned*)(q.res + (long long)place(q.res_halo) * q.res_cs + ch);
    }
    if (RAW) {
        ta = *(const int4*)(p.bias + ch);
    } else {
        ta = *(const int4*)(p.epi.a + ch); tb = *(const int4*)(p.epi.b + ch); tc = *(const int4*)(p.epi.c + ch);
        td = *(const int4*)(p.epi.d + ch); te = *(const int4*)(p.epi.e + ch);
        if (q.res) {
            sa = *(const int4*)(q.sum.a + ch); sb = *(const int4*)(q.sum.b + ch); sc = *(const int4*)(q.sum.c + ch);
            sd = *(const int4*)(q.sum.d + ch); se = *(const int4*)(q.sum.e + ch);
            if (q.has_pre) {
                xa = *(const int4*)(q.pre.a + ch); xb = *(const int4*)(q.pre.b + ch); xc = *(const int4*)(q.pre.c + ch);
                xd = *(const int4*)(q.pre.d + ch); xe = *(const int4*)(q.pre.e + ch);
            }
        }
    }

    // ---- the steps: a stage's fragments are read together, the stage is refilled, then they are multiplied
    unsigned pa[KH], wa[KH];
#pragma unroll
    for (int kk = 0; kk < KH; ++kk) {
        pa[kk] = lds0 + wave * (S * STAGE) + swz_k<BK>(l32, 2 * kk + lh);
        wa[kk] = lds0 + wave * (S * STAGE) + A_CH * 1024
               + (W4 ? (kk / 2) * 1024 + l32 * 32 + (((2 * (kk % 2) + lh) ^ ((l32 >> 3) & 3)) << 3) : swz_k<BK>(l32, 2 * kk + lh));
    }
    v16i acc = v16i{};
    int slot = 0;
    for (int i = 0; i < n; ++i) {
        // loads answer in order; the tables' and the residual's were issued behind the first S steps: at the latest after the first
        // wait of the tail everything has landed
        if (i + S <= n) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LPI * (S - 1)) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        v4i fp[KH], fw[KH];
        v2i fw4[KH];
#pragma unroll
        for (int kk = 0; kk < KH; ++kk) {
            if (W4) lds_read64_nowait<0>(fw4[kk], wa[kk] + slot * STAGE);
            else lds_read128_nowait<0>(fw[kk], wa[kk] + slot * STAGE);
            lds_read128_nowait<0>(fp[kk], pa[kk] + slot * STAGE);
        }
        wait_lgkm<0>();
#pragma unroll
        for (int kk = 0; kk < KH; ++kk) {
            if (W4) {
                tie(fw4[kk]);
                const unsigned p0 = (unsigned)fw4[kk][0], p1 = (unsigned)fw4[kk][1];
                fw[kk][0] = (int)((p0 << 4) & 0xf0f0f0f0u);
                fw[kk][1] = (int)(p0 & 0xf0f0f0f0u);
                fw[kk][2] = (int)((p1 << 4) & 0xf0f0f0f0u);
                fw[kk][3] = (int)(p1 & 0xf0f0f0f0u);
            } else {
                tie(fw[kk]);
            }
            tie(fp[kk]);
        }
        if (i + S < n)
            issue(wave + (i + S) * NW, slot);
        slot = slot + 1 == S ? 0 : slot + 1;
#pragma unroll
        for (int kk = 0; kk < KH; ++kk)
            acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(fw[kk], fp[kk], acc, 0, 0, 0);
    }

    // ---- the partial sums meet: lane (l32, lh) holds, for pixel l32, channels 8 g + 4 lh + e in acc[4 g + e]
    __syncthreads();                                       // (every wave has read its last stage; no load is under way)
    int* red = (int*)smem;
#pragma unroll
    for (int g = 0; g < 4; ++g)
        *(v4i*)(red + (wave * 32 + l32) * RP + 8 * g + 4 * lh) = v4i{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
    __syncthreads();
#pragma unroll
    for (int u = 0; u < ITEMS; ++u) {
        const int m = (tid >> 3) + u * (NW * 8);
        v4i v = *(const v4i*)(red + m * RP + (tid & 7) * 4);
#pragma unroll
        for (int w = 1; w < NW; ++w)
            v += *(const v4i*)(red + (w * 32 + m) * RP + (tid & 7) * 4);
        if (pixel[u] < 0)
            continue;
        if (RAW) {
            int r[4];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                r[e] = epi_apply<EPI_RAW>(v[e] + (e == 0 ? ta.x : e == 1 ? ta.y : e == 2 ? ta.z : ta.w), 0, 0, 0, 0, 0, 0, 0, p.epi.relu);
            *(int4*)((int*)p.out + (long long)pixel[u] * p.out_cs + ch) = int4{r[0], r[1], r[2], r[3]};
            continue;
        }
        const int A[4] = {ta.x, ta.y, ta.z, ta.w}, B[4] = {tb.x, tb.y, tb.z, tb.w}, Cc[4] = {tc.x, tc.y, tc.z, tc.w},
                  D[4] = {td.x, td.y, td.z, td.w}, E[4] = {te.x, te.y, te.z, te.w};
        int r[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            int t = W4 ? v[e] >> 4 : v[e];
            if (q.preclamp) t = med3_i32(t, A[e], B[e]);
            r[e] = med3_i32((__mul24(t, Cc[e]) + D[e]) >> E[e], p.epi.lo, p.epi.hi);       // (the bias is inside the tables)
        }
        if (q.res) {
            const unsigned w = other[u] ^ q.res_flip;
            const int XA[4] = {xa.x, xa.y, xa.z, xa.w}, XB[4] = {xb.x, xb.y, xb.z, xb.w}, XC[4] = {xc.x, xc.y, xc.z, xc.w},
                      XD[4] = {xd.x, xd.y, xd.z, xd.w}, XE[4] = {xe.x, xe.y, xe.z, xe.w}, SA[4] = {sa.x, sa.y, sa.z, sa.w},
                      SB[4] = {sb.x, sb.y, sb.z, sb.w}, SC[4] = {sc.x, sc.y, sc.z, sc.w}, SD[4] = {sd.x, sd.y, sd.z, sd.w},
                      SE[4] = {se.x, se.y, se.z, se.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                int o = (int)((w >> (8 * e)) & 0xffu);
                if (q.has_pre) {
                    if (q.pre_clamp) o = med3_i32(o, XA[e], XB[e]);
                    o = med3_i32((__mul24(o, XC[e]) + XD[e]) >> XE[e], q.pre.lo, q.pre.hi);
                }
                int t = r[e] + o;
                if (q.sum_clamp) t = med3_i32(t, SA[e], SB[e]);
                r[e] = med3_i32((__mul24(t, SC[e]) + SD[e]) >> SE[e], q.sum.lo, q.sum.hi);
            }
        }
        if (p.out_dtype == N2D2HIP_I32)
            *(int4*)((int*)p.out + (long long)pixel[u] * p.out_cs + ch) = int4{r[0], r[1], r[2], r[3]};
        else
            *(unsigned*)((signed char*)p.out + (long long)pixel[u] * p.out_cs + ch) = pack_bytes(r[0], r[1], r[2], r[3]) ^ p.out_xor;
    }
}

template <int VALID>
void launch_kind(const ConvPipeArgs& a, bool w4, int grid, hipStream_t stream)
{
    if (a.c.epi.kind == EPI_RAW) {
        if constexpr (VALID == 1)
            N2D2HIP_LAUNCH_T(conv_split_kernel, (VALID, false, true), dim3(grid), dim3(NW * 64), 0, stream, a);
    } else if (w4) {
        N2D2HIP_LAUNCH_T(conv_split_kernel, (VALID, true, false), dim3(grid), dim3(NW * 64), 0, stream, a);
    } else {
        N2D2HIP_LAUNCH_T(conv_split_kernel, (VALID, false, false), dim3(grid), dim3(NW * 64), 0, stream, a);
    }
}

void launch(ConvPipeArgs a, int valid, bool w4, hipStream_t stream)
{
    a.c.niter = a.c.ktot / 128;
    a.cper = a.c.in_cs / 128;
    a.mtiles = (a.c.M + 31) / 32;
    const int tiles = a.mtiles * a.c.ntiles_n;
    a.mlanes = (tiles + 7) / 8;
    magic_div((unsigned)a.mtiles, &a.xcd_mul, &a.xcd_sh);
    magic_div((unsigned)a.cper, &a.cper_mul, &a.cper_sh);
    a.kw_mul = 65536 / a.kW + 1;
    const int grid = 8 * a.mlanes;
    if (valid == 1) launch_kind<1>(a, w4, grid, stream);
    else if (valid == 2) launch_kind<2>(a, w4, grid, stream);
    else launch_kind<0>(a, w4, grid, stream);
}

} // namespace

bool conv_split_takes(const n2d2hip_conv_desc& d, int epi_kind, int valid)
{
    return d.C % 128 == 0 && d.kW * d.kH <= 31 && d.dilX == 1 && d.dilY == 1 && (epi_kind == EPI_I24 || (epi_kind == EPI_RAW && valid == 1));
}

bool conv_split_pays(long long M, int O, int ktot, bool w4, bool sum)
{
    // Tiles a compute unit gets, in quarters.  A work-group's rings are 64 KB (48 KB with packed weights), so that two (three)
    // run side by side; with more the third comes behind them while the pipelined kernel's larger tiles read less per
    // multiplication.  Measured, us, pipelined kernel / this one (256 compute units, weights not in the L2):
    //   3x3 256 -> 256, 14 x 14:  496 tiles 8.3 / 5.8, 592 8.4 / 7.9, 784 8.5 / 9.6;   4-bit: 784 9.3 / 8.2, 984 9.4 / 8.6, 1176 10.4 / 9.9
    //   3x3 512 -> 512, 7 x 7:    128 tiles 12.7 / 6.2, 400 12.9 / 8.6, 592 12.9 / 12.1, 784 13.2 / 15.0;   4-bit: 784 14.8 / 12.8
    //   3x3 128 -> 128, 28 x 28:  490 tiles 6.0 / 4.8;   4-bit: 588 6.1 / 5.1, 784 6.1 / 6.5
    //   1x1 512 -> 128 and 2048 -> 512: 492 tiles 4.1 / 3.8, 128 7.0 / 4.5;   128 -> 512: 400 3.7 / 3.4, 784 3.9 / 5.1
    // A folded sum runs on 64 x 128 tiles there: 1x1 with one, 608 tiles 6.1 / 5.4, 640 7.0 / 6.4, 784 5.2 / 5.7;
    // 4-bit 3x3 with one, 784 (9 steps) 8.4 / 7.3, 1176 (18 steps) 12.4 / 11.0.
    const long long tiles = ((M + 31) / 32) * ((round_up(O, 16) + 31) / 32);
    const int quarters = (w4 ? 12 : 9) + (sum ? 1 : 0) + (w4 && ktot >= 16 * 128 ? 4 : 0);
    return 4 * tiles <= (long long)quarters * num_cus();
}

int conv_split_launch(ConvPipeArgs a, int valid, bool w4, hipStream_t stream)
{
    N2D2HIP_REQUIRE(a.c.epi.kind == EPI_I24 || (a.c.epi.kind == EPI_RAW && valid == 1 && !w4), N2D2HIP_ERR_INVALID, "conv_split: rescale not served");
    launch(a, valid, w4, stream);
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

} // namespace n2d2hip
