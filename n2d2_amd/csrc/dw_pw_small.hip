// A 3x3 depthwise convolution and the 1x1 convolution that reads it, in one launch, for few pixels: MobileNet-v1 on one
// image.  There both launches are mostly their fixed cost (2.5 us of 4 on this chip), and the kernel for many pixels
// (dw_pw.hip), whose work-groups own 128 pixels and all their outputs, would leave most of the chip idle.
//
// A work-group owns 16 pixels x 32 outputs (64 or 128 where there are more images) and computes the depthwise convolution of its
// pixels itself, once per 32 outputs:
// what is computed again is 9 products an element, and shared are the latencies of one launch.  Its waves share the channels,
// a chunk of 64 each (or two, past 512 channels), and work alone until their sums meet in LDS:
//  * the 9 pixels of each output pixel and the chunk's tables go to the wave's own part of LDS by direct loads, 64 contiguous
//    bytes a pixel (16 bytes a lane of scattered pixels, straight to registers, took 10.4 us for 512 -> 512 channels at
//    14 x 14: the address unit takes a cycle for each line a load touches);
//  * the depthwise convolution of 16 channels x 16 pixels is a 16x16x64 instruction a tap row, whose 64 terms are 16 channels
//    at 4 columns (three taps, the fourth weighing 0);
//  * of its result a lane holds 4 channels of one pixel, and the rescaled bytes of 4 channel groups are, as they lie, the
//    pixel operand of the 1x1 convolution's 16x16x64 instruction, whose weights are laid out for that order of the channels.
#include <algorithm>
#include <vector>

#include "common.h"
#include "conv_handle.hpp"
#include "dw_pw.hpp"
#include "epilogue.hpp"
#include "mfma_util.hpp"

namespace n2d2hip {

namespace {

// rows of a chunk's depthwise tables: tap columns as dwords (w[0][kx], w[1][kx], w[2][kx], 0), the rescale, and what only the
// general rescale needs
enum { DWS_W, DWS_C = 3, DWS_D, DWS_E, DWS_BIAS, DWS_A, DWS_B, DWS_ROWS = 12 };
constexpr int OUTS = 32, PIXELS = 16, MAX_PARTS = 8;
constexpr int MAX_BLOCKS = 8;                     // blocks of 16 outputs of a work-group at most
constexpr int TILES_OUTS = 128;                   // a handle of at most so many outputs holds the kernel for many pixels too
constexpr int STAGE_PIXELS = 9 * PIXELS * 64, STAGE = STAGE_PIXELS + DWS_ROWS * 64 * 4;      // bytes of LDS of a wave

struct DwPwSmallArgs {
    const signed char* in;
    signed char* out;
    const int* dwt;               // [chunk][DWS_ROWS][64]
    const signed char* wpw;       // [block of 16 outputs][chunk][lane][16 bytes]
    const int* pwt;               // bias, a, b, c, d, e, each [O]
    const signed char* fill_line; // C bytes of the input's stored 0
    int C, O, nchunks, parts;
    int H, W, OH, OW, stride, padL, padT;
    int ntasks;                   // output pixels
    int first;                    // of those, the launch's first
    unsigned ow_mul, ow_sh, oh_mul, oh_sh;
    unsigned mid_xor, out_xor;
    int dw_lo, dw_hi;
    int pw_kind, pw_lo, pw_hi;
};

// KIND of the depthwise cell's rescale (FAST: EPI_I24 with the bias folded in, no clamp before it, saturating to [0, 255]); GN:
// groups of 16 channels in a chunk; OB: blocks of 16 outputs
template <int KIND, bool FAST, int GN, int OB>
__global__ __launch_bounds__(64 * MAX_PARTS) void dw_pw_small_kernel(const DwPwSmallArgs q)
{
    typedef const v4i __attribute__((address_space(1))) * GlobalQuad;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];       // STAGE bytes a wave
    const int lane = threadIdx.x & 63, p = lane & 15, g = lane >> 4;
    const int part = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    unsigned char* const stage = smem + part * STAGE;

    // the pixel this lane brings 16 bytes of, 4 lanes a pixel; a pixel's 16-channel groups are swizzled so that 16 pixels' bytes
    // of one group lie in different banks
    const int pl = lane >> 2, group = (lane & 3) ^ (pl >> 2 & 3);
    const int task = min(q.first + (int)blockIdx.y * PIXELS + pl, q.ntasks - 1);
    const int t1 = div_magic(task, q.ow_mul, q.ow_sh), ox = task - t1 * q.OW;
    const int b = div_magic(t1, q.oh_mul, q.oh_sh), oy = t1 - b * q.OH;
    const int ix = ox * q.stride - q.padL, iy = oy * q.stride - q.padT;
    const signed char* tap[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        const bool ok = group < GN && (unsigned)(ix + i % 3) < (unsigned)q.W && (unsigned)(iy + i / 3) < (unsigned)q.H;
        tap[i] = (ok ? q.in + ((long long)(b * q.H + iy + i / 3) * q.W + ix + i % 3) * q.C : q.fill_line) + 16 * (group % GN);
    }

    // the matrix of a tap row weighs, for channel p, that channel's bytes only: byte p % 4 of dword p / 4 is w[ky][g]
    const unsigned select = g == 3 ? 0x0c0c0c0cu : 0x0c0c0c0cu & ~(255u << (8 * (p & 3)));
    const unsigned select1 = g == 3 ? 0u : 1u << (8 * (p & 3));
    const int n0 = (int)blockIdx.x * OB;          // first block of 16 outputs
    v4i acc[OB];
#pragma unroll
    for (int o = 0; o < OB; ++o)
        acc[o] = v4i{};
    for (int k = part; k < q.nchunks; k += q.parts) {
        v4i wp[OB];
#pragma unroll
        for (int i = 0; i < 9; ++i)
            __builtin_amdgcn_global_load_lds((gbl_ptr_t)(tap[i] + k * 64), (lds_ptr_t)(stage + i * 1024), 16, 0, 0);
#pragma unroll
        for (int i = 0; i < (FAST ? 2 : 3); ++i)
            __builtin_amdgcn_global_load_lds((gbl_ptr_t)(q.dwt + ((size_t)k * DWS_ROWS + 4 * i) * 64 + 4 * lane),
                                             (lds_ptr_t)(stage + STAGE_PIXELS + i * 1024), 16, 0, 0);
#pragma unroll
        for (int o = 0; o < OB; ++o)
            wp[o] = *(GlobalQuad)(q.wpw + (((size_t)(n0 + o) * q.nchunks + k) * 64 + lane) * 16);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const int* const t = (const int*)(stage + STAGE_PIXELS);
        const unsigned char* const px = stage + ((g < 3 ? g : 2) * PIXELS + p) * 64;
        v4i mid = {};
#pragma unroll
        for (int G = 0; G < GN; ++G) {
            const int* const tg = t + 16 * G + 4 * g;
            const unsigned taps = (unsigned)t[g * 64 + 16 * G + p];              // (the row after the taps for the fourth column)
            const v4i tc = *(const v4i*)(tg + DWS_C * 64), td = *(const v4i*)(tg + DWS_D * 64), te = *(const v4i*)(tg + DWS_E * 64);
            v4i s = {}, ta = {}, tb = {};
            if (!FAST) {
                s = *(const v4i*)(tg + DWS_BIAS * 64);
                ta = *(const v4i*)(tg + DWS_A * 64);
                tb = *(const v4i*)(tg + DWS_B * 64);
            }
#pragma unroll
            for (int ky = 0; ky < 3; ++ky) {
                const v4i f = *(const v4i*)(px + ky * 3 * PIXELS * 64 + ((G ^ (p >> 2 & 3)) << 4));
                const int byte = (int)__builtin_amdgcn_perm(0u, taps, select + ky * select1);
                v4i w;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    w[e] = (p >> 2) == e ? byte : 0;
                s = __builtin_amdgcn_mfma_i32_16x16x64_i8(w, f, s, 0, 0, 0);
            }
            int v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                v[e] = FAST ? (__mul24(s[e], tc[e]) + td[e]) >> te[e]
                            : epi_apply<KIND>(s[e], ta[e], tb[e], tc[e], td[e], te[e], q.dw_lo, q.dw_hi, 0);
            mid[G] = (int)((FAST ? sat_bytes_u8(v[0], v[1], v[2], v[3]) : pack_bytes(v[0], v[1], v[2], v[3])) ^ q.mid_xor);
        }
#pragma unroll
        for (int o = 0; o < OB; ++o)
            acc[o] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wp[o], mid, acc[o], 0, 0, 0);
        if (k + q.parts < q.nchunks)              // the next chunk's loads write what this one's reads have read
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    // the sums of the waves meet where each kept its pixels
#pragma unroll
    for (int o = 0; o < OB; ++o)
        *(v4i*)(stage + (o * 64 + lane) * 16) = acc[o];
    __syncthreads();
    // 16 pixels x 16 outputs a wave: lane (p, g) holds outputs 4 g .. 4 g + 3 of pixel p
    for (int o = part; o < OB; o += q.parts) {
        v4i s = *(const v4i*)(smem + (o * 64 + lane) * 16);
        for (int i = 1; i < q.parts; ++i)
            s += *(const v4i*)(smem + i * STAGE + (o * 64 + lane) * 16);
        const int ch = (n0 + o) * 16 + 4 * g;
        const v4i bias = *(const v4i*)(q.pwt + ch), a = *(const v4i*)(q.pwt + q.O + ch), bb = *(const v4i*)(q.pwt + 2 * q.O + ch);
        const v4i c = *(const v4i*)(q.pwt + 3 * q.O + ch), d = *(const v4i*)(q.pwt + 4 * q.O + ch), e5 = *(const v4i*)(q.pwt + 5 * q.O + ch);
        int v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            v[e] = q.pw_kind == EPI_I24 ? epi_apply<EPI_I24>(s[e] + bias[e], a[e], bb[e], c[e], d[e], e5[e], q.pw_lo, q.pw_hi, 0)
                                        : epi_apply<EPI_I64>(s[e] + bias[e], a[e], bb[e], c[e], 0, e5[e], q.pw_lo, q.pw_hi, 0);
        const int pix = q.first + (int)blockIdx.y * PIXELS + p;
        if (pix < q.ntasks)
            *(unsigned*)(q.out + (long long)pix * q.O + ch) = pack_bytes(v[0], v[1], v[2], v[3]) ^ q.out_xor;
    }
}

template <int KIND, bool FAST>
void launch_groups(const DwPwSmallArgs& a, int blocks, unsigned pixel_groups, hipStream_t stream)
{
    static_assert(MAX_BLOCKS * 1024 <= STAGE, "a wave's sums lie where its pixels were");
    const dim3 grid((unsigned)(a.O / (16 * blocks)), pixel_groups), waves(64 * a.parts);
    if (a.C == 32) N2D2HIP_LAUNCH_T(dw_pw_small_kernel, (KIND, FAST, 2, 2), grid, waves, a.parts * STAGE, stream, a);
    else if (blocks == 2) N2D2HIP_LAUNCH_T(dw_pw_small_kernel, (KIND, FAST, 4, 2), grid, waves, a.parts * STAGE, stream, a);
    else if (blocks == 4) N2D2HIP_LAUNCH_T(dw_pw_small_kernel, (KIND, FAST, 4, 4), grid, waves, a.parts * STAGE, stream, a);
    else N2D2HIP_LAUNCH_T(dw_pw_small_kernel, (KIND, FAST, 4, MAX_BLOCKS), grid, waves, a.parts * STAGE, stream, a);
}

bool integer_bytes(const n2d2hip_act_s* a)
{
    return (a->args.kind == EPI_I24 || a->args.kind == EPI_I64) && a->min_out >= -128 && a->max_out <= 255;
}

long long work_groups(int O, long long pixels, int blocks = OUTS / 16) { return (pixels + PIXELS - 1) / PIXELS * (O / (16 * blocks)); }
// of those, as many as are on the chip at once (by their LDS, 12 KB a wave)
long long on_chip(int C) { return (long long)num_cus() * (163840 / (std::min(MAX_PARTS, (C + 63) / 64) * STAGE)); }
// Blocks of 16 outputs of a work-group: the fewest with which all are on the chip at once.  More outputs share one depthwise convolution, and
// fewer work-groups the chip.  us, 2 / 4 / 8 blocks: 512 -> 512, 14 x 14, one image 4.9 / 5.2 / 5.5, two 8.1 / 5.3 / 5.5, four 14.5 / 9.0 / 5.7.  (Up to 128 outputs the plan's lines
// are those of 32, with the kernel for many pixels behind them.)
int output_blocks(int C, int O, long long pixels)
{
    int blocks = OUTS / 16;
    while (O > TILES_OUTS && C != 32 && blocks < MAX_BLOCKS && O % (32 * blocks) == 0 && work_groups(O, pixels, blocks) > on_chip(C)) blocks *= 2;
    return blocks;
}

// Where both are faster than the cells' own launches: is the kernel for many pixels the faster one?  It gives a work-group 8 x 16
// pixels and all their outputs, up to 256.  us, that kernel / this one: 32 -> 64 channels, 112 x 112 3.6 / 4.8, two images of 48 x 48
// 3.4 / 4.1; 64 -> 128 stride 2, 56 x 56 4.6 / 4.3, two 4.6 / 5.1; 128 -> 128, 4096 pixels 5.1 / 4.7, 5184 5.1 / 5.2, two images of 56 x 56
// 5.2 / 6.7, four 5.3 / 10.0; 64 -> 256, 2304 pixels 4.9 / 4.8, 4096 5.0 / 5.3; 64 -> 512, 1369 4.9 / 4.9, 2304 5.0 / 5.6.
bool tiles_first(int C, int O, long long pixels) { return (C == 32 && O <= TILES_OUTS) || work_groups(O, pixels) > 1024; }

// Is this kernel faster than the cells' own launches?
bool small_wins(int C, int O, long long pixels)
{
    // Where all work-groups are on the chip at once.  us, one launch / two, for one, two, four, eight and sixteen images (* the rule declines):
    //   256 -> 256, 28 x 28   4.7 6.2   5.1 7.0   6.0 7.0   9.8 8.1*  14.6 10.5*
    //   256 -> 512, 14 x 14   4.2 5.8   4.6 5.8   5.1 6.5   6.1 6.8   9.9 7.9*
    //   512 -> 512, 14 x 14   4.9 6.1   5.3 6.3   5.7 7.3   9.7 7.8*  18.0 9.2*
    //   512 -> 1024, 7 x 7    4.8 5.8   4.9 5.9   5.3 6.0   5.7 6.7   9.7 7.4*
    //   1024 -> 1024, 7 x 7   5.9 6.4   6.0 6.5   6.5 6.7   6.9 7.8   12.0 8.9*
    //   128 -> 256, 28 x 28   4.2 5.8   4.7 6.4   5.6 6.6   7.1 7.5   (from 9216 pixels on the kernel for many)
    return work_groups(O, pixels, output_blocks(C, O, pixels)) <= on_chip(C);
}

} // namespace

bool dw_pw_small_takes(const n2d2hip_conv_s* dw, const n2d2hip_conv_s* pw)
{
    const int C = dw->desc.C, O = pw->desc.O;
    return plain_3x3_depthwise(dw) && integer_bytes(dw->act) && plain_1x1(pw->desc) && !pw->depthwise && !pw->sub_inner && !pw->is_fc && pw->desc.C == C
        && pw->in_cs == C && pw->in_dtype == byte_type_of(dw->act) && O % OUTS == 0 && integer_bytes(pw->act) && !pw->sum && pw->ktot >= C && pw->d_bias
        && (int)pw->act->htab.size() >= 5 * pw->act->cpad;
}

} // namespace n2d2hip

using namespace n2d2hip;

struct n2d2hip_dw_pw_small_s {
    n2d2hip_conv_t dw, pw;
    n2d2hip_dw_pw_t tiles;        // the kernel for many pixels, where it takes the pair and there are at most TILES_OUTS outputs, or null
    bool fast;
    int nchunks;
    signed char* d_image;         // 1x1 weights, depthwise tables, 1x1 tables, the stored 0
    size_t dwt_at, pwt_at, fill_at;
};

extern "C" {

int n2d2hip_dw_pw_small_destroy(n2d2hip_dw_pw_small_t h)
{
    if (!h) return N2D2HIP_OK;
    if (h->d_image) (void)hipFree(h->d_image);
    if (h->tiles) n2d2hip_dw_pw_destroy(h->tiles);
    delete h;
    return N2D2HIP_OK;
}

int n2d2hip_dw_pw_small_create(n2d2hip_conv_t dw, n2d2hip_conv_t pw, n2d2hip_dw_pw_small_t* out)
{
    N2D2HIP_REQUIRE(dw && pw && out, N2D2HIP_ERR_INVALID, "dw_pw_small_create: null argument");
    const int C = dw->desc.C, O = pw->desc.O;
    N2D2HIP_REQUIRE(dw_pw_small_takes(dw, pw), N2D2HIP_ERR_UNSUPPORTED,
                    "dw_pw_small_create: needs a 3x3 undilated depthwise convolution of stride 1 or 2 over 32 or a multiple of 64 channels and an "
                    "unpadded 1x1 convolution of stride 1 reading it, to a multiple of 32 channels, both 8-bit with integer rescales and byte "
                    "outputs, the second without a folded sum");
    const int nchunks = (C + 63) / 64;
    std::vector<signed char> w((size_t)pw->opad * pw->ktot);
    std::vector<int> wdw(4 * (size_t)C), bias(O), fold;
    hipError_t e = hipMemcpy(w.data(), pw->d_w, w.size(), hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(wdw.data(), dw->d_wdw, wdw.size() * sizeof(int), hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(bias.data(), pw->d_bias, bias.size() * sizeof(int), hipMemcpyDeviceToHost);
    const bool fast = dw->bias_folded && dw->d_epi_tab && !dw->preclamp && dw->act->args.kind == EPI_I24 && dw->act->args.lo == 0
        && dw->act->args.hi == 255;
    const int cpd = dw->act->cpad, cpp = pw->act->cpad;
    if (fast) {                                   // a - bias, b - bias, c, d + bias * c, e
        fold.resize(5 * (size_t)cpd);
        if (e == hipSuccess) e = hipMemcpy(fold.data(), dw->d_epi_tab, fold.size() * sizeof(int), hipMemcpyDeviceToHost);
    }
    if (e != hipSuccess)
        return fail(N2D2HIP_ERR_HIP, "dw_pw_small_create: reading the cells back failed: %s", hipGetErrorString(e));
    n2d2hip_dw_pw_small_s* h = new n2d2hip_dw_pw_small_s();
    h->dw = dw; h->pw = pw; h->fast = fast; h->nchunks = nchunks; h->d_image = nullptr; h->tiles = nullptr;
    h->dwt_at = (size_t)(O / 16) * nchunks * 1024;
    h->pwt_at = h->dwt_at + (size_t)nchunks * DWS_ROWS * 64 * sizeof(int);
    h->fill_at = h->pwt_at + 6 * (size_t)O * sizeof(int);
    std::vector<signed char> img(h->fill_at + (size_t)nchunks * 64, 0);
    // lane (p, g) of an output block: output p, and in byte 4 * G + i channel 16 * G + 4 * g + i of the chunk
    signed char* to = img.data();
    for (int o0 = 0; o0 < O; o0 += 16)
        for (int c0 = 0; c0 < C; c0 += 64)
            for (int g = 0; g < 4; ++g)
                for (int o = o0; o < o0 + 16; ++o, to += 16)
                    for (int G = 0; G < (C == 32 ? 2 : 4); ++G)
                        memcpy(to + 4 * G, w.data() + (size_t)o * pw->ktot + c0 + 16 * G + 4 * g, 4);
    int* const dwt = (int*)(img.data() + h->dwt_at);
    const std::vector<int>& tab = fast ? fold : dw->act->htab;
    for (int c = 0; c < C; ++c) {
        int* const t = dwt + (size_t)(c / 64) * DWS_ROWS * 64 + c % 64;
        for (int kx = 0; kx < 3; ++kx)
            for (int ky = 0; ky < 3; ++ky)
                t[(DWS_W + kx) * 64] |= (wdw[(size_t)ky * C + c] >> (8 * kx) & 255) << (8 * ky);
        t[DWS_BIAS * 64] = wdw[3 * (size_t)C + c];
        const int rows[5] = {DWS_A, DWS_B, DWS_C, DWS_D, DWS_E};
        for (int r = 0; r < 5; ++r)
            t[rows[r] * 64] = tab[(size_t)r * cpd + c];
    }
    int* const pwt = (int*)(img.data() + h->pwt_at);
    for (int o = 0; o < O; ++o) {
        pwt[o] = bias[o];
        for (int r = 0; r < 5; ++r)
            pwt[(size_t)(r + 1) * O + o] = pw->act->htab[(size_t)r * cpp + o];
    }
    memset(img.data() + h->fill_at, zero_point(dw->in_dtype) ? 0x80 : 0, img.size() - h->fill_at);
    e = hipMalloc((void**)&h->d_image, img.size());
    if (e == hipSuccess) e = hipMemcpy(h->d_image, img.data(), img.size(), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        n2d2hip_dw_pw_small_destroy(h);
        return fail(N2D2HIP_ERR_HIP, "dw_pw_small_create: device upload failed: %s", hipGetErrorString(e));
    }
    if (O <= TILES_OUTS && dw_pw_takes(dw, pw)) {
        const int rc = n2d2hip_dw_pw_create(dw, pw, &h->tiles);
        if (rc != N2D2HIP_OK) {
            h->tiles = nullptr;
            n2d2hip_dw_pw_small_destroy(h);
            return rc;
        }
    }
    *out = h;
    return N2D2HIP_OK;
}

static bool choose_tiles(n2d2hip_dw_pw_small_t h, long long pixels) { return h->tiles && tiles_first(h->dw->desc.C, h->pw->desc.O, pixels); }

int n2d2hip_dw_pw_plan(n2d2hip_conv_t dw, n2d2hip_conv_t pw, int batch, int in_h, int in_w)
{
    int OH, OW;
    if (!dw || !pw || batch <= 0 || n2d2hip_conv_out_dims(&dw->desc, in_h, in_w, &OH, &OW) != N2D2HIP_OK)
        return N2D2HIP_DW_PW_APART;
    const int C = dw->desc.C, O = pw->desc.O;
    const long long pixels = (long long)batch * OH * OW;
    const bool tiles = dw_pw_takes(dw, pw) && dw_pw_wins(C, O, batch, OH, OW), small = dw_pw_small_takes(dw, pw) && small_wins(C, O, pixels);
    if (tiles && (!small || tiles_first(C, O, pixels)))
        return N2D2HIP_DW_PW_TILES;
    return small ? N2D2HIP_DW_PW_SMALL : N2D2HIP_DW_PW_APART;
}

int n2d2hip_dw_pw_small_pays(n2d2hip_dw_pw_small_t h, int batch, int in_h, int in_w)
{
    if (!h || batch <= 0)
        return 0;
    int OH, OW;
    if (n2d2hip_conv_out_dims(&h->dw->desc, in_h, in_w, &OH, &OW) != N2D2HIP_OK)
        return 0;
    const long long pixels = (long long)batch * OH * OW;
    const int C = h->dw->desc.C, O = h->pw->desc.O;
    return choose_tiles(h, pixels) ? dw_pw_wins(C, O, batch, OH, OW) : small_wins(C, O, pixels);
}

int n2d2hip_dw_pw_small_forward(n2d2hip_dw_pw_small_t h, const n2d2hip_tensor* in, const n2d2hip_tensor* out, n2d2hip_stream_t stream_)
{
    hipStream_t stream = (hipStream_t)stream_;
    N2D2HIP_REQUIRE(h && in && out && in->data && out->data, N2D2HIP_ERR_INVALID, "dw_pw_small_forward: null argument");
    const n2d2hip_conv_desc& dd = h->dw->desc;
    const n2d2hip_conv_desc& dp = h->pw->desc;
    int OH, OW;
    const int rc = n2d2hip_conv_out_dims(&dd, in->H, in->W, &OH, &OW);
    if (rc != N2D2HIP_OK)
        return rc;
    const long long pixels = (long long)in->B * OH * OW;
    if (choose_tiles(h, pixels))
        return n2d2hip_dw_pw_forward(h->tiles, in, out, stream_);
    const int out_dtype = byte_type_of(h->pw->act);
    N2D2HIP_REQUIRE(in->layout == N2D2HIP_NHWC && out->layout == N2D2HIP_NHWC && in->halo == 0 && out->halo == 0, N2D2HIP_ERR_UNSUPPORTED,
                    "dw_pw_small_forward: tensors must be NHWC without a border");
    N2D2HIP_REQUIRE(in->dtype == h->dw->in_dtype && in->C == dd.C && in->cs == dd.C, N2D2HIP_ERR_INVALID,
                    "dw_pw_small_forward: input has %d channels (stride %d) of type %d, the depthwise convolution expects %d of type %d", in->C,
                    in->cs, in->dtype, dd.C, h->dw->in_dtype);
    N2D2HIP_REQUIRE(out->B == in->B && out->C == dp.O && out->cs == dp.O && out->H == OH && out->W == OW && out->dtype == out_dtype,
                    N2D2HIP_ERR_INVALID, "dw_pw_small_forward: output must be %dx%dx%dx%d bytes of type %d with a channel stride of %d", in->B,
                    dp.O, OH, OW, out_dtype, dp.O);
    constexpr int SPAN = 65535 * PIXELS;         // pixels of a launch at most
    N2D2HIP_REQUIRE(pixels > 0 && pixels < (1ll << 31) - SPAN && (long long)in->B * in->H * in->W * in->cs < (1ll << 31),
                    N2D2HIP_ERR_UNSUPPORTED, "dw_pw_small_forward: tensor too large");
    DwPwSmallArgs a;
    a.in = (const signed char*)in->data; a.out = (signed char*)out->data;
    a.wpw = h->d_image; a.dwt = (const int*)(h->d_image + h->dwt_at); a.pwt = (const int*)(h->d_image + h->pwt_at);
    a.fill_line = h->d_image + h->fill_at;
    a.C = dd.C; a.O = dp.O; a.nchunks = h->nchunks; a.parts = std::min(MAX_PARTS, h->nchunks);
    a.H = in->H; a.W = in->W; a.OH = OH; a.OW = OW; a.stride = dd.strideX; a.padL = dd.padL; a.padT = dd.padT;
    a.ntasks = (int)pixels;
    magic_div((unsigned)OW, &a.ow_mul, &a.ow_sh);
    magic_div((unsigned)OH, &a.oh_mul, &a.oh_sh);
    a.mid_xor = h->pw->in_dtype == N2D2HIP_U8B ? 0x80808080u : 0u;
    a.out_xor = out_dtype == N2D2HIP_U8B ? 0x80808080u : 0u;
    a.dw_lo = h->dw->act->args.lo; a.dw_hi = h->dw->act->args.hi;
    a.pw_kind = h->pw->act->args.kind; a.pw_lo = h->pw->act->args.lo; a.pw_hi = h->pw->act->args.hi;
    const int blocks = output_blocks(dd.C, dp.O, pixels);
    // (output tiles first: work-groups 8 apart share an XCD, whose L2 then holds an eighth of the 1x1 weights)
    for (a.first = 0; a.first < a.ntasks; a.first += SPAN) {
        const unsigned groups = (unsigned)((std::min(SPAN, a.ntasks - a.first) + PIXELS - 1) / PIXELS);
        if (h->fast) launch_groups<EPI_I24, true>(a, blocks, groups, stream);
        else if (h->dw->act->args.kind == EPI_I24) launch_groups<EPI_I24, false>(a, blocks, groups, stream);
        else launch_groups<EPI_I64, false>(a, blocks, groups, stream);
    }
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

} // extern "C"
