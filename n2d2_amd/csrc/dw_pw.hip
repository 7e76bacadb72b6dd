// A 3x3 depthwise convolution and the 1x1 convolution that reads it, in one launch (the building block of the MobileNets).
// Launched cell by cell, the depthwise output is written by one launch and read back by the next, and at 14 x 14 and
// below both launches are mostly their fixed cost.  Here a work-group takes tiles of 8 rows x 16 columns of output pixels, and
// of a tile one chunk of 64 (or 32) channels a step: the depthwise convolution of the chunk is rescaled to bytes, written to
// LDS as the pixel operand of the 1x1 convolution, of which the chunk is one slice of K, and multiplied there; the depthwise
// output never reaches memory.
//
// The depthwise convolution runs on the matrix cores as well, though its matrix is mostly zeros: of 16 channels x 16 pixels, one
// 16x16x64 instruction a tap row, whose 64 terms are 16 channels at 4 columns (three taps, the fourth weighing 0) and whose
// weights for a channel are zero but for that channel's bytes.  Its pixel operand is 16 bytes of one pixel as they lie in
// memory, read once for the three output rows that use it.  On the vector ALU, 4 outputs took 12 dot products and about 20
// instructions of transposes, borders and addresses.  What is left there are the two rescales, 14 instructions for 4 outputs.
//
// LDS: the input of a chunk (the tile and its border, by loads that go there directly; a pixel outside the image comes from a
// line of the stored 0), the pixel operand, the 1x1 weights and the depthwise tables, each twice: while step n is computed,
// the input of step n + 1 is on its way, and the multiplication is one step behind the depthwise part, so that one barrier a
// step is enough.  A work-group stays for a run of tiles.  All slots of 16 bytes are swizzled by the pixel so that 16
// pixels' slots of one channel group lie in different banks.
//
// Batch of 64, MobileNet-v1's sizes, before (depthwise on the vector ALU, one tile a work-group, no loads ahead) and now, us:
// 32 -> 64 channels at 112 x 112 34.6 and 19.5 (77 MB, 4.0 TB/s: near the rate of a copy), 64 -> 128 from 112 to 56 30.9 and 19.5
// (77 MB), 128 -> 128 at 56 29.4 and 20.7, 128 -> 256 from 56 to 28 26.6 and 15.8, 256 -> 256 at 28 27.7 and 18.4.  The last three
// have less to move (51, 38 and 26 MB); vector ALU and LDS are each about half busy there, and a step's parts wait for
// each other.  Measured and not kept: half of the waves multiplying first (+2 us), the multiplication before the depthwise
// part (0), 4 waves in place of 8 (+1 to 3 us); 16 waves only where a work-group has 256 outputs (-0.5 us).
#include <algorithm>
#include <vector>

#include "common.h"
#include "conv_handle.hpp"
#include "dw_pw.hpp"
#include "epilogue.hpp"
#include "mfma_util.hpp"

namespace n2d2hip {

struct DwPwArgs {
    const signed char* in;    // B x H x W x C bytes
    signed char* out;         // B x OH x OW x O bytes
    const int* dwt;           // depthwise tables: [chunk][DWT_ROWS][KC] ints, see DWT_*
    const signed char* wpw;   // 1x1 weights: [channel tile of 32*NB][chunk][K step of 32][32-channel block][lane][16 bytes]
    const int* pwt;           // 1x1 rescale with the bias folded in: c and e, d, a, b, each [O]
    const signed char* fill_line;   // 16 bytes of the input's stored form of 0
    int C, O;
    int H, W, OH, OW, padL, padT;
    int tw;                   // valid columns of a tile (at most 16)
    int tiles_x, tiles_y, ntiles;
    int per_xcd, per_block, extra_tiles;   // tiles of an XCD; of those, of one work-group; the first so many have one more
    unsigned mid_xor;         // 0x80808080 when the depthwise output is stored as value - 128
    unsigned out_xor;
    int dw_lo, dw_hi;
    int pw_lo, pw_hi;
    unsigned out_bytes;
};

namespace {

// Rows of a chunk's depthwise tables: the tap columns as dwords (w[0][kx], w[1][kx], w[2][kx], 0), the rescale, and what only
// the general rescale needs (the bias with the zero point folded in, and the bounds).
enum { DWT_W, DWT_CE = 3, DWT_D, DWT_BIAS, DWT_A, DWT_B, DWT_USED, DWT_ROWS = 8 };

// 16 bytes a lane from its own address to 16 * lane bytes past LDS offset `lds`, which is the same in all lanes.  As text,
// because the compiler would wait for every such load of the wave before the next LDS read of any buffer.  m0, which holds the
// offset, is an operand: the compiler writes it and knows what is in it.
__device__ __forceinline__ void load_to_lds(const void* src, unsigned lds)
{
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(src), "{m0}"(lds) : "memory");
}

// (acc * c + d) >> e of the rescales on 32 bits.  acc comes from an instruction of the compiler's: it waits for a matrix
// instruction's result before its own instructions only, not before text (so the clamp before this is not med3_i32 either).  c fits 24 bits, of which alone the multiply-add reads: its word carries e in
// the top byte, so that a table costs one LDS read less.
__device__ __forceinline__ int scale24(int acc, int ce, int d)
{
    int r;
    asm("v_ashrrev_i32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_3 src1_sel:DWORD" : "=v"(r) : "v"(ce), "v"(__mul24(acc, ce) + d));
    return r;
}

// What a variant needs of a compute unit.  SINGLE: the layer is one chunk, whose weights and tables stay for all tiles.
template <int S, int KC, int NB, int WAVES, bool SINGLE, bool FAST>
struct DwPwShape {
    static constexpr int TCOLS = S == 1 ? 18 : 33, TROWS = S == 1 ? 10 : 17;        // input pixels of a tile
    static constexpr int IN_LOADS = (TROWS * TCOLS * KC + 1023) / 1024;             // of 1 KB each
    static constexpr int IN_BYTES = IN_LOADS * 1024;
    static_assert(IN_BYTES >= (TROWS * TCOLS + 1) * KC, "the fourth tap of the last pixel, which weighs 0, reads one pixel past the tile");
    static constexpr int A_BYTES = 128 * KC;
    static constexpr int B_BYTES = KC * NB * 32;
    static constexpr int NT = NB * 32;              // output channels of the work-group
    static constexpr int DWT_LOADS = ((FAST ? (int)DWT_BIAS : (int)DWT_USED) * KC * 4 + 1023) / 1024;
    static constexpr int DWT_BYTES = DWT_LOADS * 1024;
    static_assert(DWT_BYTES <= DWT_ROWS * KC * 4, "the loads stay within the chunk's rows");
    static constexpr int A_OFF = 2 * IN_BYTES, B_OFF = A_OFF + 2 * A_BYTES;
    static constexpr int D_OFF = B_OFF + (SINGLE ? 1 : 2) * B_BYTES, T_OFF = D_OFF + (SINGLE ? 1 : 2) * DWT_BYTES;
    static constexpr int PW_ROWS = FAST ? 2 : 4;    // rows of the 1x1 tables that are read
    static constexpr int LDS = T_OFF + PW_ROWS * NT * 4;
    // work-groups on a compute unit: by LDS, and by registers (5 waves a SIMD have 96 each, 4 have 128, 2 have 256)
    static constexpr int MAX_GROUPS = (2 * NB / WAVES == 1 ? 20 : 8) / WAVES;
    static constexpr int GROUPS = 163840 / LDS < MAX_GROUPS ? 163840 / LDS : MAX_GROUPS;
};

// S: stride of the depthwise convolution; KC: channels per chunk (64, or 32 for a 32-channel layer); NB: 32-channel blocks
// of the 1x1 convolution's outputs a work-group computes (blockIdx.y selects which 32 * NB of them); WAVES: 4, 8 or 16.
// FAST: neither cell needs a clamp before its multiply and both saturate to [0, 255]: the depthwise tables c, d, e are then
// the ones with the bias folded in (accumulators start from zero), and both rescales saturate while they pack.
template <int S, int KC, int NB, int WAVES, bool SINGLE, bool FAST>
__global__ __launch_bounds__(64 * WAVES, (DwPwShape<S, KC, NB, WAVES, SINGLE, FAST>::GROUPS * WAVES / 4)) void dw_pw_kernel(const DwPwArgs q)
{
    typedef DwPwShape<S, KC, NB, WAVES, SINGLE, FAST> Z;
    constexpr int THREADS = 64 * WAVES;
    constexpr int PB = 2;                    // a wave multiplies 2 blocks of 32 pixels ...
    constexpr int NBW = NB / (WAVES / 2);    // ... with 1 or 2 blocks of 32 channels
    static_assert(NBW == 1 || NBW == 2, "a wave stores one channel block or a pair");
    constexpr int SL = KC / 16;              // 16-channel groups of a chunk = 16-byte slots of a pixel
    constexpr int RP = WAVES / SL;           // the tile's rows are split over this many sets of waves
    constexpr int ROWS = 8 / RP;             // output rows a wave walks down
    constexpr int KS = KC / 32;
    constexpr int TCOLS = Z::TCOLS, NT = Z::NT;
    __shared__ __attribute__((aligned(16))) unsigned char smem[Z::LDS];
    const unsigned lds0 = (unsigned)(unsigned long long)(lds_ptr_t)smem;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, lh = lane >> 5;

    // blocks 8 apart run on the same XCD: give each XCD a run of consecutive tiles (neighbours share input rows), and each
    // work-group a run of those
    const int xcd = (int)(blockIdx.x & 7), i = (int)(blockIdx.x >> 3);
    const int extra = min(i, q.extra_tiles);
    const int tile0 = xcd * q.per_xcd + i * q.per_block + extra;
    const int ntile = min(q.per_block + (i < q.extra_tiles ? 1 : 0), min((xcd + 1) * q.per_xcd, q.ntiles) - tile0);
    if (ntile <= 0)
        return;
    const int n0 = (int)blockIdx.y * NT;
    const int nchunks = SINGLE ? 1 : q.C / KC;
    const int nsteps = ntile * nchunks;
    struct Tile { int x, y, b; };
    Tile lt = {tile0 % q.tiles_x, (tile0 / q.tiles_x) % q.tiles_y, tile0 / (q.tiles_x * q.tiles_y)};     // the tile that is loaded
    Tile et = lt;                                                                                         // the one that is written
    auto advance = [&](Tile& t) {
        if (++t.x == q.tiles_x) {
            t.x = 0;
            if (++t.y == q.tiles_y) {
                t.y = 0;
                ++t.b;
            }
        }
    };

    // swizzle of a pixel's slots: 16 consecutive pixels of one slot lie in 16 different 16-byte columns of the 64 banks
    auto swizzle = [](int pos) { return (pos / (16 / SL)) & (SL - 1); };

    // ---- input loads: load j of this wave brings slots 64 * (wave + WAVES * j) + lane of the tile.  A row holds its pixels in
    // order (stride 2: the even columns first), a pixel its 16-channel groups swizzled; outside the image the fill is read.
    constexpr int NLD = (Z::IN_LOADS + WAVES - 1) / WAVES;
    int ld_pos[NLD], ld_off[NLD];      // the slot's row (16 bits up) and column, its bytes from the tile's first pixel
    int in_off[NLD];
#pragma unroll
    for (int j = 0; j < NLD; ++j) {
        const unsigned idx = (wave + WAVES * j) * 64 + lane;
        const unsigned pix = idx / SL, slot = idx % SL;
        const unsigned r = pix / TCOLS, pos = pix % TCOLS;
        const int col = S == 1 ? pos : pos < 17 ? 2 * pos : 2 * (pos - 17) + 1;
        ld_pos[j] = (int)r << 16 | col;         // (the last load ends in a row below the tile)
        ld_off[j] = ((int)r * q.W + col) * q.C + ((slot ^ swizzle(pos)) << 4);
    }
    auto place_tile = [&]() {
        const int ix0 = lt.x * q.tw * S - q.padL, iy0 = lt.y * 8 * S - q.padT;
        const int base = ((lt.b * q.H + iy0) * q.W + ix0) * q.C;
#pragma unroll
        for (int j = 0; j < NLD; ++j)
            in_off[j] = (unsigned)(ix0 + (ld_pos[j] & 0xffff)) < (unsigned)q.W && (unsigned)(iy0 + (ld_pos[j] >> 16)) < (unsigned)q.H ? base + ld_off[j] : -1;
    };
    auto issue_tables = [&](int kc, int step) {
        if (wave < Z::DWT_LOADS)
            load_to_lds((const char*)q.dwt + kc * (DWT_ROWS * KC * 4) + wave * 1024 + lane * 16,
                        lds0 + Z::D_OFF + (SINGLE ? 0 : (step & 1) * Z::DWT_BYTES) + wave * 1024);
    };
    int lkc = 0;                             // the chunk that is loaded
    auto issue_input = [&](int step) {
        if (lkc == 0)
            place_tile();
        const unsigned dst = lds0 + (step & 1) * Z::IN_BYTES;
        const signed char* base = q.in + lkc * KC;
#pragma unroll
        for (int j = 0; j < NLD; ++j)
            if (wave + WAVES * j < Z::IN_LOADS)
                load_to_lds(in_off[j] >= 0 ? base + in_off[j] : q.fill_line, dst + (wave + WAVES * j) * 1024);
        if (!SINGLE)
            issue_tables(lkc, step);
        if (++lkc == nchunks) {
            lkc = 0;
            advance(lt);
        }
    };
    auto issue_weights = [&](int kc, int step) {     // B_BYTES contiguous bytes, 1 KB per load
        const signed char* src = q.wpw + ((long long)blockIdx.y * nchunks + kc) * Z::B_BYTES + lane * 16;
        const unsigned dst = lds0 + Z::B_OFF + (SINGLE ? 0 : (step & 1) * Z::B_BYTES);
#pragma unroll
        for (int j = 0; j < (Z::B_BYTES / 1024 + WAVES - 1) / WAVES; ++j) {
            const int c = wave + WAVES * j;
            if (c < Z::B_BYTES / 1024)
                load_to_lds(src + c * 1024, dst + c * 1024);
        }
    };
    issue_input(0);
    if (SINGLE) {
        issue_weights(0, 0);
        issue_tables(0, 0);
    }

    // ---- depthwise side: this wave's 16 channels and rows; lane (p, g): output column p, tap column g (the fourth tap weighs 0)
    const int cgid = wave % SL, rp = wave / SL;
    const int p = lane & 15, g = lane >> 4;
    // the matrix of a tap row weighs, for channel p, that channel's bytes only: byte p % 4 of dword p / 4 is w[ky][g]
    const unsigned select = g == 3 ? 0x0c0c0c0cu : 0x0c0c0c0cu & ~(255u << (8 * (p & 3)));
    const unsigned select1 = g == 3 ? 0u : 1u << (8 * (p & 3));
    struct Chunk { v4i w[3], ce, d, bias, a, b; };
    auto read_chunk = [&](const int* t, Chunk& k) {
        const int* tc = t + cgid * 16 + 4 * g;
        const unsigned taps = (unsigned)t[DWT_W * KC + g * KC + cgid * 16 + p];      // (the row after them for the fourth)
#pragma unroll
        for (int ky = 0; ky < 3; ++ky) {
            const int byte = (int)__builtin_amdgcn_perm(0u, taps, select + ky * select1);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                k.w[ky][e] = (p >> 2) == e ? byte : 0;
        }
        k.ce = *(const v4i*)(tc + DWT_CE * KC);
        k.d = *(const v4i*)(tc + DWT_D * KC);
        if (!FAST) {
            k.bias = *(const v4i*)(tc + DWT_BIAS * KC);
            k.a = *(const v4i*)(tc + DWT_A * KC);
            k.b = *(const v4i*)(tc + DWT_B * KC);
        }
    };

    // ---- the 1x1 convolution's tables
    int* const tab = (int*)(smem + Z::T_OFF);
    for (int i = tid; i < Z::PW_ROWS * NT; i += THREADS)
        tab[i] = q.pwt[i / NT * q.O + n0 + i % NT];

    const int wm = wave & 1, wn = wave >> 1;     // this wave's 64 pixels and its channel blocks
    v16i acc[PB][NBW];
#pragma unroll
    for (int u = 0; u < PB; ++u)
#pragma unroll
        for (int i = 0; i < NBW; ++i)
            acc[u][i] = v16i{};
    const __amdgpu_buffer_rsrc_t out_rsrc = __builtin_amdgcn_make_buffer_rsrc(q.out, 0, q.out_bytes, 0x00020000);

    const int pos0 = S == 1 ? p + g : (g & 1) * 17 + p + (g >> 1);
    const int in_addr = ((rp * ROWS * S) * TCOLS + pos0) * KC + ((cgid ^ swizzle(pos0)) << 4);
    const int mid_addr = rp * ROWS * 16 * KC + p * KC + ((cgid ^ swizzle(p)) << 4) + 4 * g;       // (16 rows further the swizzle is the same)
    const int m0 = 64 * wm + l32;                // this lane's pixels of the 1x1 convolution: m0 and m0 + 32
    const int pf_addr = m0 * KC;

    bool stored = false;                         // the last iteration stored
    int kc = 0, pkc = 0;                         // chunk of the depthwise part, chunk of the multiplication (one step behind)
    for (int step = 0; step <= nsteps; ++step) {
        // This step's input and the weights of the one before have arrived (a wave's stores were issued last and may be on their
        // way), and every wave is past what it read from the buffers that are filled next.
        if (stored) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(PB * NBW) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" : : : "memory");
        if (step + 1 < nsteps)
            issue_input(step + 1);
        if (step < nsteps) {
            if (!SINGLE)
                issue_weights(kc, step);
            Chunk k;
            read_chunk((const int*)(smem + Z::D_OFF + (SINGLE ? 0 : (step & 1) * Z::DWT_BYTES)), k);
            const unsigned char* ib = smem + (step & 1) * Z::IN_BYTES + in_addr;
            unsigned char* ab = smem + Z::A_OFF + (step & 1) * Z::A_BYTES + mid_addr;
            v4i f[ROWS * S + 3 - S];
#pragma unroll
            for (int r = 0; r < ROWS * S + 3 - S; ++r)
                f[r] = *(const v4i*)(ib + r * TCOLS * KC);
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
                v4i s = FAST ? v4i{} : k.bias;
#pragma unroll
                for (int ky = 0; ky < 3; ++ky)
                    s = __builtin_amdgcn_mfma_i32_16x16x64_i8(k.w[ky], f[S * r + ky], s, 0, 0, 0);
                int v[4];
                unsigned packed;
                if (FAST) {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        v[e] = scale24(s[e], k.ce[e], k.d[e]);
                    packed = sat_bytes_u8(v[0], v[1], v[2], v[3]);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        v[e] = med3_i32(scale24(clamp_i32(s[e], k.a[e], k.b[e]), k.ce[e], k.d[e]), q.dw_lo, q.dw_hi);
                    packed = pack_bytes(v[0], v[1], v[2], v[3]);
                }
                *(unsigned*)(ab + r * 16 * KC) = packed ^ q.mid_xor;
            }
            if (++kc == nchunks)
                kc = 0;
        }
        stored = false;
        if (step == 0)
            continue;
        __builtin_amdgcn_sched_barrier(0);       // (registers: nothing of this part is read early)
        // ---- multiply the chunk before: this wave's 32 pixels against all its channel blocks
        const unsigned char* abuf = smem + Z::A_OFF + ((step - 1) & 1) * Z::A_BYTES;
        const unsigned char* bbuf = smem + Z::B_OFF + (SINGLE ? 0 : ((step - 1) & 1) * Z::B_BYTES);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            v4i pf[PB];
#pragma unroll
            for (int u = 0; u < PB; ++u)
                pf[u] = *(const v4i*)(abuf + pf_addr + u * 32 * KC + (((2 * ks + lh) ^ swizzle(l32)) << 4));
#pragma unroll
            for (int nb = 0; nb < NBW; ++nb) {
                const v4i wf = *(const v4i*)(bbuf + ((ks * NB + wn * NBW + nb) * 64 + lane) * 16);
#pragma unroll
                for (int u = 0; u < PB; ++u)
                    acc[u][nb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wf, pf[u], SINGLE && ks == 0 ? v16i{} : acc[u][nb], 0, 0, 0);
            }
        }
        if (++pkc < nchunks)
            continue;
        pkc = 0;
        stored = true;

        // ---- epilogue: lane (l32, lh) holds, for pixel m0 + 32 * u, channels 32 * (wn * NBW + nb) + 8 * h + 4 * lh + e in
        // acc[u][nb][4 * h + e]
        unsigned qd[PB][NBW][4];
#pragma unroll
        for (int i = 0; i < NBW; ++i) {
            if (!FAST)
                __builtin_amdgcn_sched_barrier(0);
            unsigned pk[PB][4];
#pragma unroll
            for (int h = 0; h < 4; ++h) {
                const int ch = (wn * NBW + i) * 32 + 8 * h + 4 * lh;
                const v4i tce = *(const v4i*)(tab + ch), td = *(const v4i*)(tab + NT + ch);
                v4i ta, tb;
                if (!FAST) {
                    ta = *(const v4i*)(tab + 2 * NT + ch);
                    tb = *(const v4i*)(tab + 3 * NT + ch);
                }
#pragma unroll
                for (int u = 0; u < PB; ++u) {
                    int r[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if (FAST) r[e] = scale24(acc[u][i][4 * h + e], tce[e], td[e]);
                        else r[e] = med3_i32(scale24(clamp_i32(acc[u][i][4 * h + e], ta[e], tb[e]), tce[e], td[e]), q.pw_lo, q.pw_hi);
                    }
                    pk[u][h] = (FAST ? sat_bytes_u8(r[0], r[1], r[2], r[3]) : pack_bytes(r[0], r[1], r[2], r[3])) ^ q.out_xor;
                }
            }
            // exchange between the lane halves: the lower lane owns the block's first 16 channels, the upper one the others
#pragma unroll
            for (int u = 0; u < PB; ++u) {
                const auto s02 = __builtin_amdgcn_permlane32_swap(pk[u][0], pk[u][2], false, false);
                const auto s13 = __builtin_amdgcn_permlane32_swap(pk[u][1], pk[u][3], false, false);
                qd[u][i][0] = s02[0]; qd[u][i][1] = s02[1]; qd[u][i][2] = s13[0]; qd[u][i][3] = s13[1];
            }
        }
#pragma unroll
        for (int u = 0; u < PB; ++u) {
            const int m = m0 + 32 * u, px = m & 15, py = m >> 4;
            const int oxo = et.x * q.tw + px, oyo = et.y * 8 + py;
            const bool pix_ok = px < q.tw && oxo < q.OW && oyo < q.OH;
            // (a store outside the tensor is dropped by its bounds: every wave issues all of them, which the wait above counts)
            const unsigned out_off = pix_ok ? (unsigned)((((et.b * q.OH + oyo) * q.OW + oxo) * q.O) + n0 + wn * NBW * 32 + 16 * NBW * lh) : 0x80000000u;
            typedef unsigned v4u __attribute__((ext_vector_type(4)));
            v4u first, second;
            if constexpr (NBW == 1) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    first[e] = qd[u][0][e];
                __builtin_amdgcn_raw_buffer_store_b128(first, out_rsrc, out_off, 0, 0);
            } else {
                // ... of a pair: the lower lane owns the first block's 32 channels
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const auto xw = __builtin_amdgcn_permlane32_swap(qd[u][0][e], qd[u][1][e], false, false);
                    first[e] = xw[0];
                    second[e] = xw[1];
                }
                __builtin_amdgcn_raw_buffer_store_b128(first, out_rsrc, out_off, 0, 0);
                __builtin_amdgcn_raw_buffer_store_b128(second, out_rsrc, out_off + 16, 0, 0);
            }
        }
        advance(et);
        if (!SINGLE) {
#pragma unroll
            for (int u = 0; u < PB; ++u)
#pragma unroll
                for (int i = 0; i < NBW; ++i)
                    acc[u][i] = v16i{};
        }
    }
}

template <int S, int KC, int NB, int WAVES, bool SINGLE, bool FAST>
void launch_one(DwPwArgs a, int ytiles, hipStream_t stream)
{
    // as many work-groups as the chip holds at a time, each with a run of tiles: their loads overlap the tile before, and
    // tables, addresses and (one chunk) weights are prepared once
    typedef DwPwShape<S, KC, NB, WAVES, SINGLE, FAST> Z;
    const int slots = std::max(1, num_cus() / 8 * Z::GROUPS / ytiles);       // work-groups of an XCD at a time
    a.per_xcd = (a.ntiles + 7) / 8;
    const int groups = std::min(slots, a.per_xcd);
    a.per_block = a.per_xcd / groups;
    a.extra_tiles = a.per_xcd % groups;          // to the first work-groups, each of which shares its unit with a later one
    const dim3 grid((unsigned)(8 * groups), (unsigned)ytiles);
    N2D2HIP_LAUNCH_T(dw_pw_kernel, (S, KC, NB, WAVES, SINGLE, FAST), grid, dim3(64 * WAVES), 0, stream, a);
}

template <int S, int KC, bool SINGLE, bool FAST>
void launch_nb(const DwPwArgs& a, int nb, hipStream_t stream)
{
    const int ytiles = a.O / (nb * 32);
    if (nb == 8) launch_one<S, KC, 8, 16, SINGLE, FAST>(a, ytiles, stream);
    else if (nb == 4) launch_one<S, KC, 4, 8, SINGLE, FAST>(a, ytiles, stream);
    else launch_one<S, KC, 2, 4, SINGLE, FAST>(a, ytiles, stream);
}

template <int S, int KC, bool SINGLE>
void launch_fast(const DwPwArgs& a, bool fast, int nb, hipStream_t stream)
{
    if (fast) launch_nb<S, KC, SINGLE, true>(a, nb, stream); else launch_nb<S, KC, SINGLE, false>(a, nb, stream);
}

template <int S>
void launch_chunks(const DwPwArgs& a, bool fast, int nb, hipStream_t stream)
{
    if (a.C == 32) launch_fast<S, 32, true>(a, fast, nb, stream);
    else if (a.C == 64) launch_fast<S, 64, true>(a, fast, nb, stream);
    else launch_fast<S, 64, false>(a, fast, nb, stream);
}

// columns of a tile: 16, or fewer when that leaves fewer idle columns in the last tile of a row
int tile_columns(int OW)
{
    int best_tw = 16;
    long long best_cols = ((OW + 15) / 16) * 16;
    for (int tw = 15; tw >= 8; --tw) {
        const long long cols = (long long)((OW + tw - 1) / tw) * 16;
        if (cols < best_cols) { best_cols = cols; best_tw = tw; }
    }
    return best_tw;
}

} // namespace

// A work-group goes through its tile's chunks of 64 channels one behind the other, about 1.1 us each, so a launch takes 3 us and
// that for every round of work-groups, while the cells' own launches grow with the pixels from 5 or 6 us on.  us, this launch / the
// cells' own two:
//  * one chunk: 32 -> 64 one pixel 3.0 / 6.0, 32400 4.0 / 8.0; 64 -> 256 4.4 / 6.4 and, 16384, 5.4 / 7.9; 64 -> 512, 32400, 10.6 / 13.3
//  * up to 128 outputs: 128 -> 128 one pixel 4.7 / 5.5; 192 -> 128 5.6 / 6.3; 256 -> 128 one pixel 6.4 / 5.3, 2304 6.8 / 6.9, 8192
//    7.0 / 7.7; 320 -> 128, 2048, 7.7 / 7.7; 384 -> 128, 5184 8.6 / 8.0, 9408 8.7 / 9.5; 512 -> 128, 8192 10.5 / 9.0, 9408 10.5 / 10.8; 768 -> 128, 10000
//    13.9 / 12.9, 16384 14.1 / 15.4; 1024 -> 64, 16384 20.9 / 19.9, 19600 21.0 / 22.1
//  * 256 outputs, whose work-group has the compute unit to itself: 256 -> 256, 6272 8.2 / 8.0, 9408 8.4 / 9.9; 512 -> 256, 8192 11.8 / 9.6,
//    9408 11.9 / 12.0; 1024 -> 256, 12800 21.8 / 19.9.  Two rounds, the second nearly empty: 25872 pixels 256 -> 256 14.0 / 14.0, 512 -> 256
//    21.2 / 19.3; 37632 14.4 / 18.1 and 23.0 / 27.4; 1024 -> 256, 32400 44.9 / 38.5, 40000 45.2 / 47.5
//  * 512 outputs, each tile's depthwise part computed twice: 512 -> 512 at 14 x 14, images: 40 12.7 / 12.3, 48 12.6 / 13.6, 64 (one round)
//    13.0 / 15.4, 65 21.5 / 15.2, 96 21.8 / 21.4, 112 22.6 / 22.1, 128 (two) 22.6 / 24.2, 192 (three) 34.4 / 33.2; at 10 x 10, whose tiles are
//    39 % full, 96 21.1 / 14.0; at 13 x 13, 118 21.7 / 20.6, 128 21.6 / 21.7; 1024 -> 512, 10000 pixels 23.3 / 22.5, 19600 44.0 / 36.0.  (Level ones run as one
//    launch: in MobileNet-v1, 128 images of 193 x 193, that is 383 us where two launches a pair are 395.)
bool dw_pw_wins(int C, int O, int batch, int OH, int OW)
{
    const int chunks = (C + 63) / 64;
    const long long pixels = (long long)batch * OH * OW;
    if (chunks == 1)
        return O <= 512;
    if (O <= 128)
        return pixels >= (chunks <= 3 ? 0 : chunks <= 5 ? 2304 : std::max(9216, 1200 * chunks));
    if (O > 512 || (O == 512 && chunks > 8))
        return false;
    const int tw = tile_columns(OW);
    const long long groups = (long long)batch * ((OH + 7) / 8) * ((OW + tw - 1) / tw) * (O / 256), rounds = (groups + num_cus() - 1) / num_cus();
    if (rounds == 1)
        return pixels >= std::max(9216, 1000 * chunks);
    return O == 512 ? rounds == 2 && pixels >= 20800 : pixels >= rounds * (9600 + 800 * chunks);
}

bool dw_pw_takes(const n2d2hip_conv_s* dw, const n2d2hip_conv_s* pw)
{
    const int C = dw->desc.C, O = pw->desc.O;
    return plain_3x3_depthwise(dw) && dw->act->args.kind == EPI_I24 && dw->act->min_out >= -128 && dw->act->max_out <= 255 && plain_1x1(pw->desc)
        && !pw->sub_inner && pw->desc.C == C && pw->in_cs == C && pw->in_dtype == byte_type_of(dw->act) && (O == 64 || O == 128 || O % 256 == 0)
        && pw->act->args.kind == EPI_I24 && pw->bias_folded && pw->d_epi_tab && pw->act->min_out >= -128 && pw->act->max_out <= 255 && !pw->sum && pw->ktot >= C;
}

} // namespace n2d2hip

using namespace n2d2hip;

struct n2d2hip_dw_pw_s {
    n2d2hip_conv_t dw, pw;
    int nb;                   // 32-channel blocks per work-group
    bool fast;                // neither rescale clamps before its multiply, both saturate to [0, 255]
    signed char* d_w;
    int* d_tab;               // 1x1 tables, [4][O]; 4 ints of the depthwise input's stored 0; depthwise tables by chunk
};

extern "C" {

int n2d2hip_dw_pw_destroy(n2d2hip_dw_pw_t h)
{
    if (!h) return N2D2HIP_OK;
    if (h->d_w) (void)hipFree(h->d_w);
    if (h->d_tab) (void)hipFree(h->d_tab);
    delete h;
    return N2D2HIP_OK;
}

int n2d2hip_dw_pw_create(n2d2hip_conv_t dw, n2d2hip_conv_t pw, n2d2hip_dw_pw_t* out)
{
    N2D2HIP_REQUIRE(dw && pw && out, N2D2HIP_ERR_INVALID, "dw_pw_create: null argument");
    const int C = dw->desc.C, O = pw->desc.O;
    N2D2HIP_REQUIRE(dw_pw_takes(dw, pw), N2D2HIP_ERR_UNSUPPORTED,
                    "dw_pw_create: needs a 3x3 undilated depthwise convolution of stride 1 or 2 over 32 or a multiple of 64 channels and an "
                    "unpadded 1x1 convolution of stride 1 reading it, to 64, 128 or a multiple of 256 channels, both 8-bit with integer "
                    "rescales (32-bit multiply-add) and byte outputs, the second without a folded sum");
    const int kc = C == 32 ? 32 : 64, nb = std::min(O, 256) / 32;
    const int nchunks = C / kc, ks = kc / 32;
    std::vector<signed char> w((size_t)pw->opad * pw->ktot);
    const int cp = pw->act->cpad;
    std::vector<int> tab5(5 * (size_t)cp);
    hipError_t e = hipMemcpy(w.data(), pw->d_w, w.size(), hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(tab5.data(), pw->d_epi_tab, tab5.size() * sizeof(int), hipMemcpyDeviceToHost);
    if (e != hipSuccess)
        return fail(N2D2HIP_ERR_HIP, "dw_pw_create: reading the 1x1 convolution back failed: %s", hipGetErrorString(e));
    // [channel tile][chunk][K step][32-channel block][lane][16 bytes]: lane l holds channel l % 32 of the block,
    // bytes K step * 32 + 16 * (l / 32) .. of the chunk
    auto fragment_image = [&](int blocks) {
        std::vector<signed char> img((size_t)O * C);
        const int tile = blocks * 32;
        for (int t = 0; t < O / tile; ++t)
            for (int c = 0; c < nchunks; ++c)
                for (int s = 0; s < ks; ++s)
                    for (int blk = 0; blk < blocks; ++blk)
                        for (int l = 0; l < 64; ++l)
                            memcpy(img.data() + ((((size_t)(t * nchunks + c) * ks + s) * blocks + blk) * 64 + l) * 16,
                                   w.data() + (size_t)(t * tile + blk * 32 + (l & 31)) * pw->ktot + c * kc + s * 32 + 16 * (l >> 5), 16);
        return img;
    };
    const std::vector<signed char> img = fragment_image(nb);
    // c and e, d, a, b by channel; a cell that needs no clamp before its multiply gets bounds that clamp nothing
    auto with_shift = [](int c, int e) { return (int)(((unsigned)c & 0xffffffu) | (unsigned)e << 24); };
    std::vector<int> tab(4 * (size_t)O);
    for (int o = 0; o < O; ++o) {
        tab[o] = with_shift(tab5[2 * (size_t)cp + o], tab5[4 * (size_t)cp + o]);
        tab[(size_t)O + o] = tab5[3 * (size_t)cp + o];
        tab[2 * (size_t)O + o] = pw->preclamp ? tab5[o] : std::numeric_limits<int>::min();
        tab[3 * (size_t)O + o] = pw->preclamp ? tab5[(size_t)cp + o] : std::numeric_limits<int>::max();
    }
    // 16 bytes of the depthwise input's stored 0 behind them, then the depthwise tables
    tab.insert(tab.end(), 4, zero_point(dw->in_dtype) ? (int)0x80808080u : 0);
    const bool fast = dw->bias_folded && dw->d_epi_tab && !dw->preclamp && dw->act->args.lo == 0 && dw->act->args.hi == 255
        && !pw->preclamp && pw->act->args.lo == 0 && pw->act->args.hi == 255;
    {
        const int cpd = dw->act->cpad;
        std::vector<int> wdw(4 * (size_t)C), rescale = dw->act->htab;      // a, b, c, d, e, each [cpad]
        e = hipMemcpy(wdw.data(), dw->d_wdw, wdw.size() * sizeof(int), hipMemcpyDeviceToHost);
        if (fast && e == hipSuccess) e = hipMemcpy(rescale.data(), dw->d_epi_tab, 5 * (size_t)cpd * sizeof(int), hipMemcpyDeviceToHost);
        if (e != hipSuccess)
            return fail(N2D2HIP_ERR_HIP, "dw_pw_create: reading the depthwise tables back failed: %s", hipGetErrorString(e));
        const size_t base = tab.size();
        tab.resize(base + (size_t)nchunks * DWT_ROWS * kc);
        for (int c = 0; c < C; ++c) {
            int* const t0 = tab.data() + base + (size_t)(c / kc) * DWT_ROWS * kc + c % kc;
            for (int kx = 0; kx < 3; ++kx)
                for (int ky = 0; ky < 3; ++ky)
                    t0[(DWT_W + kx) * kc] |= (wdw[(size_t)ky * C + c] >> (8 * kx) & 255) << (8 * ky);
            t0[DWT_CE * kc] = with_shift(rescale[2 * (size_t)cpd + c], rescale[4 * (size_t)cpd + c]);
            t0[DWT_D * kc] = rescale[3 * (size_t)cpd + c];
            t0[DWT_BIAS * kc] = wdw[3 * (size_t)C + c];
            t0[DWT_A * kc] = rescale[c];
            t0[DWT_B * kc] = rescale[(size_t)cpd + c];
        }
    }
    n2d2hip_dw_pw_s* h = new n2d2hip_dw_pw_s();
    h->dw = dw; h->pw = pw; h->nb = nb; h->fast = fast; h->d_w = nullptr; h->d_tab = nullptr;
    e = hipMalloc((void**)&h->d_w, img.size());
    if (e == hipSuccess) e = hipMemcpy(h->d_w, img.data(), img.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMalloc((void**)&h->d_tab, tab.size() * sizeof(int));
    if (e == hipSuccess) e = hipMemcpy(h->d_tab, tab.data(), tab.size() * sizeof(int), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        n2d2hip_dw_pw_destroy(h);
        return fail(N2D2HIP_ERR_HIP, "dw_pw_create: device upload failed: %s", hipGetErrorString(e));
    }
    *out = h;
    return N2D2HIP_OK;
}

int n2d2hip_dw_pw_pays(n2d2hip_dw_pw_t h, int batch, int in_h, int in_w)
{
    if (!h || batch <= 0)
        return 0;
    int OH, OW;
    if (n2d2hip_conv_out_dims(&h->dw->desc, in_h, in_w, &OH, &OW) != N2D2HIP_OK)
        return 0;
    return dw_pw_wins(h->dw->desc.C, h->pw->desc.O, batch, OH, OW) ? 1 : 0;
}

int n2d2hip_dw_pw_forward(n2d2hip_dw_pw_t h, const n2d2hip_tensor* in, const n2d2hip_tensor* out, n2d2hip_stream_t stream_)
{
    hipStream_t stream = (hipStream_t)stream_;
    N2D2HIP_REQUIRE(h && in && out && in->data && out->data, N2D2HIP_ERR_INVALID, "dw_pw_forward: null argument");
    const n2d2hip_conv_desc& dd = h->dw->desc;
    const n2d2hip_conv_desc& dp = h->pw->desc;
    int OH, OW;
    int rc = n2d2hip_conv_out_dims(&dd, in->H, in->W, &OH, &OW);
    if (rc != N2D2HIP_OK)
        return rc;
    const int out_dtype = byte_type_of(h->pw->act);
    N2D2HIP_REQUIRE(in->layout == N2D2HIP_NHWC && out->layout == N2D2HIP_NHWC && in->halo == 0 && out->halo == 0, N2D2HIP_ERR_UNSUPPORTED,
                    "dw_pw_forward: tensors must be NHWC without a border");
    N2D2HIP_REQUIRE(in->dtype == h->dw->in_dtype && in->C == dd.C && in->cs == dd.C, N2D2HIP_ERR_INVALID,
                    "dw_pw_forward: input has %d channels (stride %d) of type %d, the depthwise convolution expects %d of type %d", in->C,
                    in->cs, in->dtype, dd.C, h->dw->in_dtype);
    N2D2HIP_REQUIRE(out->B == in->B && out->C == dp.O && out->cs == dp.O && out->H == OH && out->W == OW && out->dtype == out_dtype,
                    N2D2HIP_ERR_INVALID, "dw_pw_forward: output must be %dx%dx%dx%d bytes of type %d with a channel stride of %d", in->B, dp.O,
                    OH, OW, out_dtype, dp.O);
    N2D2HIP_REQUIRE((long long)in->B * in->H * in->W * in->cs < (1ll << 31) && (long long)out->B * OH * OW * out->cs < (1ll << 31),
                    N2D2HIP_ERR_UNSUPPORTED, "dw_pw_forward: tensor too large");
    DwPwArgs a;
    a.in = (const signed char*)in->data; a.out = (signed char*)out->data;
    a.wpw = h->d_w; a.pwt = h->d_tab;
    a.fill_line = (const signed char*)(h->d_tab + 4 * dp.O);
    a.dwt = h->d_tab + 4 * dp.O + 4;
    a.dw_lo = h->dw->act->args.lo; a.dw_hi = h->dw->act->args.hi;
    a.C = dd.C; a.O = dp.O;
    a.H = in->H; a.W = in->W; a.OH = OH; a.OW = OW; a.padL = dd.padL; a.padT = dd.padT;
    a.tw = tile_columns(OW);
    a.tiles_x = (OW + a.tw - 1) / a.tw;
    a.tiles_y = (OH + 7) / 8;
    const long long ntiles = (long long)in->B * a.tiles_y * a.tiles_x;
    N2D2HIP_REQUIRE(ntiles < (1 << 28), N2D2HIP_ERR_UNSUPPORTED, "dw_pw_forward: tensor too large");
    a.ntiles = (int)ntiles;
    a.mid_xor = h->pw->in_dtype == N2D2HIP_U8B ? 0x80808080u : 0u;
    a.out_xor = out_dtype == N2D2HIP_U8B ? 0x80808080u : 0u;
    a.pw_lo = h->pw->act->args.lo; a.pw_hi = h->pw->act->args.hi;
    a.out_bytes = (unsigned)((long long)out->B * OH * OW * out->cs);
    if (dd.strideX == 1) launch_chunks<1>(a, h->fast, h->nb, stream);
    else launch_chunks<2>(a, h->fast, h->nb, stream);
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

} // extern "C"
