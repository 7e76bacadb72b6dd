// SAT and LSQ fake-quantization kernels (float32), forward and backward.
// Element-wise work is one coalesced grid-stride pass; the global reductions
// (max |tanh w|, mean, variance, step-size / alpha gradients) are
// wavefront-reduced with cross-lane shuffles, block-reduced through LDS, and
// finished by a one-block kernel over at most PARTIALS block results, so the
// result does not depend on scheduling.  Sums are carried in double.
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "common.h"
#include "epilogue.hpp"
#include "sat_math.hpp"

namespace n2d2hip {

constexpr int PARTIALS = 1024;   // max blocks of a reducing pass
constexpr int QBLOCK = 256;

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        v += __shfl_xor(v, off, 64);
    return v;
}
__device__ __forceinline__ float wave_max(float v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        v = fmaxf(v, __shfl_xor(v, off, 64));
    return v;
}
__device__ __forceinline__ double block_sum(double v)
{
    __shared__ double red[16];
    v = wave_sum(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0.0;
    for (int i = 0; i < (int)(blockDim.x >> 6); ++i) t += red[i];
    return t;
}
// Both sums over the block, with one wait
__device__ __forceinline__ void block_sums(double& a, double& b)
{
    __shared__ double red[16][2];
    a = wave_sum(a);
    b = wave_sum(b);
    if ((threadIdx.x & 63) == 0) { red[threadIdx.x >> 6][0] = a; red[threadIdx.x >> 6][1] = b; }
    __syncthreads();
    a = b = 0.0;
    for (int i = 0; i < (int)(blockDim.x >> 6); ++i) { a += red[i][0]; b += red[i][1]; }
}
__device__ __forceinline__ float block_max(float v)
{
    __shared__ float redm[16];
    v = wave_max(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) redm[threadIdx.x >> 6] = v;
    __syncthreads();
    float t = redm[0];
    for (int i = 1; i < (int)(blockDim.x >> 6); ++i) t = fmaxf(t, redm[i]);
    return t;
}

// A grid's walk over n values: in quads of 16 bytes where the tensors' addresses allow it, the rest one by one.  Memory bounds
// the passes that use it; at 4 bytes a load their at most 1024 blocks had too little in flight (SAT backward of 12.8 M values:
// 40.3 us, now 30.2).  f(number of values as a type, index of the first); a value is read before its place is written, so
// input and output may be one tensor.
template <class F>
__device__ __forceinline__ void for_quads(size_t n, int quads, F f)
{
    const size_t step = (size_t)gridDim.x * QBLOCK, first = (size_t)blockIdx.x * QBLOCK + threadIdx.x, n4 = quads ? n / 4 : 0;
#pragma unroll 2
    for (size_t i = first; i < n4; i += step) f(std::integral_constant<int, 4>{}, i * 4);
    for (size_t i = n4 * 4 + first; i < n; i += step) f(std::integral_constant<int, 1>{}, i);
}
template <int N>
__device__ __forceinline__ void quad_load(float* dst, const float* p, size_t i)
{
    if (N == 4) {
        const float4 v = *(const float4*)(p + i);
        dst[0] = v.x; dst[1] = v.y; dst[2] = v.z; dst[3] = v.w;
    } else {
        dst[0] = p[i];
    }
}
template <int N>
__device__ __forceinline__ void quad_store(float* p, size_t i, const float* v)
{
    if (N == 4) *(float4*)(p + i) = make_float4(v[0], v[1], v[2], v[3]);
    else p[i] = v[0];
}

// ------------------------------------------------------------ SAT weights

// The weights' quantization levels from tanh(w), ref: src/Quantizer/QAT/Kernel/SATQuantizer_Frame_Kernels.cpp:66-238
struct SatLevels {
    int mode;
    float range, tmax, inv_range, full_a, full_b, asym_a, asym_b;
    __device__ SatLevels(float r, int m, float t) : mode(m), range(r), tmax(t)
    {
        if (mode == N2D2HIP_SAT_SYMRANGE || mode == N2D2HIP_SAT_ASYMRANGE || mode == N2D2HIP_SAT_NONE_ASYM)
            range = floorf(range / 2.0f);
        inv_range = 1.0f / range;
        full_a = 1.0f + 0.9998f / range;
        full_b = 0.4999f / range;
        asym_a = 1.0f + 1.0f / (2.0f * range);
        asym_b = 1.0f / (2.0f * range);
    }
    __device__ float operator()(float t) const
    {
        float q;
        switch (mode) {
        case N2D2HIP_SAT_NONE:
            return t / tmax;
        case N2D2HIP_SAT_DEFAULT:
            q = __fmul_rn(0.5f, __fadd_rn(t / tmax, 1.0f));
            q = __fmul_rn(inv_range, rintf(__fmul_rn(q, range)));
            return __fsub_rn(__fmul_rn(q, 2.0f), 1.0f);
        case N2D2HIP_SAT_FULLRANGE:
            q = __fmul_rn(0.5f, __fadd_rn(t / tmax, 1.0f));
            q = __fsub_rn(__fmul_rn(full_a, q), full_b);
            q = __fmul_rn(inv_range, rintf(__fmul_rn(q, range)));
            return __fsub_rn(__fmul_rn(q, 2.0f), 1.0f);
        case N2D2HIP_SAT_SYMRANGE:
            q = t / tmax;
            return __fmul_rn(inv_range, rintf(__fmul_rn(q, range)));
        case N2D2HIP_SAT_ASYMRANGE:
            q = t / tmax;
            q = __fsub_rn(__fmul_rn(asym_a, q), asym_b);
            return __fmul_rn(inv_range, rintf(__fmul_rn(q, range)));
        default:
            q = t / tmax;
            return __fsub_rn(__fmul_rn(asym_a, q), asym_b);
        }
    }
};
// SAT weights of several tensors, in three launches at most: a learning net quantizes the weights of all its cells before a pass,
// most of them few, and a launch each (seven for many weights with scaling) was what bounded them.  16 tensors fit a launch's arguments.
//  * From 1025 (with scaling 8193) to SAT_SELF weights, in the first launch: every block looks for the largest weight of the whole tensor itself, 16
//    bytes a load, and computes 1024 levels.  tanh is taken of that one weight and of the block's own: it does not decrease (tanhf of
//    every positive float compared with the next one's), so the largest weight has the largest tanh.  It ends where reading the tensor from
//    L2 takes as long as the launch that leaves the blocks' maxima to a second one.  us, one block's or two launches / now: 2400 weights
//    4.1 / 3.5, 10080 6.8 / 3.9, 36864 5.8 / 4.6, 65536 5.9 / 5.4; with scaling, three launches 16384 10.0 / 8.9.
//  * Up to 1024, and 8192 with scaling: one block computes the tensor, in the first launch, its tanh in registers (instances by the
//    weights per thread: skipping unused ones inside one instance made the compiler spill).  One compute unit's arithmetic bounds it; from
//    there on many blocks are as fast (with scaling 8192 weights 7.8, 10080 9.4 / 8.5; without 1024 3.2 / 3.4).  So are up to 8192
//    weights that are overwritten by their levels, which another block must not be reading, and those that are only divided by the
//    largest (SAT_NONE, where nothing is quantized), whose launches the log has always had one by one.
//  * More: the first launch leaves each block's max |tanh w|, and every block of the second one takes the maximum of those,
//    at most 256, itself.  The second launch fills the chip, 8 blocks a compute unit, and all deal the weights to the XCDs alike, in
//    runs of 256, so that the weights come from the XCD's own L2 the second time.
//  * With scaling the blocks that computed the levels leave the sums of the levels' differences from the first level and of their squares,
//    in double, and a last launch divides the levels: every block adds the sums up itself.  (One pass for the mean, one for the squares, a
//    block's launch behind each and the division before: 163840 weights 17.4 us, with sums 11.8; 1048576 22.2 / 17.4; 4194304 36.1 / 28.3;
//    16777216 121.5 / 82.3.)  The workspace holds the sums of 448 blocks; from 2 M weights on those are of 1024 threads, which 16777216 need
//    (124.5 with 256; 1048576 18.7 with 1024).
constexpr size_t SAT_SMALL = 8 * 1024;           // weights of one block's tensor at most
constexpr size_t SAT_SELF = 64 * 1024;           // weights among which every block looks for the largest itself
constexpr int SAT_BLOCKS = 256, SAT_BLOCKS2 = 2048;     // blocks of a larger tensor's first, and second or third launch at most
constexpr int SAT_BLOCKS_SUMS = 448;             // of the second where each leaves its sums in the workspace
constexpr size_t SAT_MANY = 2 << 20;             // scaled weights from which their blocks have 1024 threads
constexpr int SAT_ITEMS = 16;
constexpr size_t SAT_SUMS = (SAT_BLOCKS + 4) * sizeof(float);       // place of the blocks' sums, behind their maxima and the first weight's tanh
template <int N>
struct SatBatch {
    n2d2hip_sat_weight_item item[N];
    unsigned first[N + 1], first2[N + 1], first3[N + 1];        // first block of a tensor in each launch
    int count;
};
enum class SatKind { SELF, SMALL, MANY };
__host__ __device__ inline SatKind sat_kind(const n2d2hip_sat_weight_item& t)
{
    const bool in_place = (uintptr_t)t.w < (uintptr_t)(t.wq + t.n) && (uintptr_t)t.wq < (uintptr_t)(t.w + t.n);
    if (!in_place && t.mode != N2D2HIP_SAT_NONE && t.n > (t.apply_scaling ? SAT_SMALL : 1024) && t.n <= SAT_SELF) return SatKind::SELF;
    return t.n <= SAT_SMALL ? SatKind::SMALL : SatKind::MANY;
}

// SAT scaling, ref: SATQuantizer_Frame_Kernels.cpp:244-262: the n levels' mean, their unbiased variance about that mean rounded to
// float, scaling = sqrt(var * outputs_size); from the sums of their differences d from one of them and of d * d, in double
__device__ __forceinline__ float sat_scaling(double sum, double squares, float shift, size_t n, unsigned outputs_size)
{
    const float mean = (float)(sum + (double)n * (double)shift) / (float)n;
    const double e = (double)mean - (double)shift, about = squares - 2.0 * e * sum + (double)n * e * e;
    const float var = (float)(about < 0.0 ? 0.0 : about) / ((float)n - 1.0f);       // (NaN stays)
    return sqrtf(var * (float)outputs_size);
}

template <int K>
__device__ __forceinline__ void sat_weight_small(const n2d2hip_sat_weight_item& t)
{
    const float* __restrict__ w = t.w;
    float* __restrict__ wq = t.wq;
    const int n = (int)t.n;
    __shared__ float first;
    float v[K];
    float m = 0.0f;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int i = k * 1024 + threadIdx.x;
        v[k] = i < n ? tanhf(w[i]) : 0.0f;
        m = fmaxf(m, fabsf(v[k]));
    }
    if (threadIdx.x == 0) first = v[0];
    m = block_max(m);
    const SatLevels level(t.range, t.mode, m);
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = level(v[k]);
    float scaling = 1.0f;
    if (t.apply_scaling) {
        const float shift = level(first);
        double sum = 0.0, squares = 0.0;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const double d = (double)v[k] - (double)shift;
            if (k * 1024 + (int)threadIdx.x < n) {
                sum += d;
                squares += d * d;
            }
        }
        block_sums(sum, squares);
        scaling = sat_scaling(sum, squares, shift, t.n, t.outputs_size);
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int i = k * 1024 + threadIdx.x;
        if (i < n) wq[i] = t.apply_scaling ? v[k] / scaling : v[k];
    }
    if (threadIdx.x == 0) { t.stats[0] = m; t.stats[1] = scaling; }
}
// A block of 1024 threads of those that look for the largest weight themselves: a level a thread
__device__ __forceinline__ void sat_weight_self(const n2d2hip_sat_weight_item& t, unsigned block)
{
    const float* __restrict__ w = t.w;
    const int n = (int)t.n, own = (int)(block * 1024 + threadIdx.x), quads = ((uintptr_t)w & 15) == 0 ? n / 4 : 0;
    const float mine = own < n ? w[own] : 0.0f, zeroth = w[0];
    float m = 0.0f;
#pragma unroll 8
    for (int i = threadIdx.x; i < quads; i += 1024) {
        const float4 v = ((const float4*)w)[i];
        m = fmaxf(m, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
    }
#pragma unroll 4
    for (int i = quads * 4 + threadIdx.x; i < n; i += 1024) m = fmaxf(m, fabsf(w[i]));
    m = tanhf(block_max(m));
    const SatLevels level(t.range, t.mode, m);
    const float q = level(tanhf(mine));
    if (own < n) t.wq[own] = q;
    if (block == 0 && threadIdx.x == 0) { t.stats[0] = m; t.stats[1] = 1.0f; }
    if (!t.apply_scaling) return;
    const float tanh0 = tanhf(zeroth);
    const double d = (double)q - (double)level(tanh0);
    double sum = own < n ? d : 0.0, squares = own < n ? d * d : 0.0;
    block_sums(sum, squares);
    if (threadIdx.x) return;
    ((double2*)((char*)t.workspace + SAT_SUMS))[block] = make_double2(sum, squares);
    if (block == 0) ((float*)t.workspace)[SAT_BLOCKS] = tanh0;
}
template <int N>
__global__ __launch_bounds__(1024) void sat_weight_first_kernel(const SatBatch<N> b)
{
    int k = 0;
    if (N > 1)
        while (k + 1 < b.count && blockIdx.x >= b.first[k + 1]) ++k;
    const n2d2hip_sat_weight_item& t = b.item[k];
    const SatKind kind = sat_kind(t);
    if (kind == SatKind::SELF) {
        sat_weight_self(t, blockIdx.x - b.first[k]);
    } else if (kind == SatKind::SMALL) {
        if (t.n <= 1024) sat_weight_small<1>(t);
        else if (t.n <= 4 * 1024) sat_weight_small<4>(t);
        else sat_weight_small<SAT_SMALL / 1024>(t);
    } else {
        // (blocks 8 apart run on the same XCD: of 8 blocks, a multiple of which there is, each takes every 8th run of 256)
        const unsigned block = blockIdx.x - b.first[k], run = 8 * (4 * (block >> 3) + (threadIdx.x >> 8)) + (block & 7);
        float m = 0.0f;
        for (size_t i = (size_t)run * QBLOCK + (threadIdx.x & (QBLOCK - 1)); i < t.n; i += (size_t)(b.first[k + 1] - b.first[k]) * 1024)
            m = fmaxf(m, fabsf(tanhf(t.w[i])));
        m = block_max(m);
        if (threadIdx.x == 0) ((float*)t.workspace)[block] = m;
        if (block == 0 && threadIdx.x == 0) ((float*)t.workspace)[SAT_BLOCKS] = tanhf(t.w[0]);
    }
}
// A thread's first weight where a tensor's blocks, of 256 or 1024 threads, take every 8th run of 256 from their own on, as the first launch's do
__device__ __forceinline__ size_t sat_first_weight(unsigned block)
{
    return (size_t)(8 * ((blockDim.x >> 8) * (block >> 3) + (threadIdx.x >> 8)) + (block & 7)) * QBLOCK + (threadIdx.x & (QBLOCK - 1));
}
template <int N>
__global__ __launch_bounds__(1024) void sat_weight_second_kernel(const SatBatch<N> b)
{
    int k = 0;
    if (N > 1)
        while (k + 1 < b.count && blockIdx.x >= b.first2[k + 1]) ++k;
    const n2d2hip_sat_weight_item& t = b.item[k];
    const float* __restrict__ w = t.w;
    float* __restrict__ wq = t.wq;
    const unsigned block = blockIdx.x - b.first2[k];
    const size_t step = (size_t)(b.first2[k + 1] - b.first2[k]) * blockDim.x;
    static_assert(SAT_BLOCKS <= QBLOCK, "a thread takes one block's maximum");
    const float m = block_max(threadIdx.x < b.first[k + 1] - b.first[k] ? ((const float*)t.workspace)[threadIdx.x] : 0.0f);
    const SatLevels level(t.range, t.mode, m);
    if (block == 0 && threadIdx.x == 0) { t.stats[0] = m; t.stats[1] = 1.0f; }
    if (!t.apply_scaling) {
        for (size_t i = sat_first_weight(block); i < t.n; i += step) wq[i] = level(tanhf(w[i]));
        return;
    }
    const float shift = level(((const float*)t.workspace)[SAT_BLOCKS]);
    double sum = 0.0, squares = 0.0;
#pragma unroll 4
    for (size_t i = sat_first_weight(block); i < t.n; i += step) {
        const float q = level(tanhf(w[i]));
        const double d = (double)q - (double)shift;
        wq[i] = q;
        sum += d;
        squares += d * d;
    }
    block_sums(sum, squares);
    if (threadIdx.x == 0) ((double2*)((char*)t.workspace + SAT_SUMS))[block] = make_double2(sum, squares);
}

// The division of the levels by their scaling.  The second launch leaves each block's sums; every block of this one adds them up itself
// and divides its share.  (A pass for the sum, one for the squares, a block's launch behind each and the division were five launches.)
template <int N>
__global__ __launch_bounds__(1024) void sat_weight_scale_kernel(const SatBatch<N> b)
{
    int k = 0;
    if (N > 1)
        while (k + 1 < b.count && blockIdx.x >= b.first3[k + 1]) ++k;
    const n2d2hip_sat_weight_item& t = b.item[k];
    float* __restrict__ wq = t.wq;
    const unsigned block = blockIdx.x - b.first3[k];
    const unsigned count = sat_kind(t) == SatKind::SELF ? b.first[k + 1] - b.first[k] : b.first2[k + 1] - b.first2[k];
    const double2* sums = (const double2*)((const char*)t.workspace + SAT_SUMS);
    const float shift = SatLevels(t.range, t.mode, t.stats[0])(((const float*)t.workspace)[SAT_BLOCKS]);
    double sum = 0.0, squares = 0.0;
    for (unsigned i = threadIdx.x; i < count; i += blockDim.x) {
        const double2 v = sums[i];
        sum += v.x;
        squares += v.y;
    }
    block_sums(sum, squares);
    const float scaling = sat_scaling(sum, squares, shift, t.n, t.outputs_size);
    if (block == 0 && threadIdx.x == 0) t.stats[1] = scaling;
    for (size_t i = sat_first_weight(block); i < t.n; i += (size_t)(b.first3[k + 1] - b.first3[k]) * blockDim.x) wq[i] = wq[i] / scaling;
}

// ref: SATQuantizer_Frame_Kernels.cpp:349-404
template <int N>
struct SatGradBatch {
    n2d2hip_sat_weight_grad_item item[N];
    float mode_factor[N];                        // slope of the quantizer's line, 0: none
    unsigned first[N + 1];
    int count;
};
template <int N>
__global__ __launch_bounds__(QBLOCK) void sat_weight_backward_kernel(const SatGradBatch<N> b)
{
    int k = 0;
    if (N > 1)
        while (k + 1 < b.count && blockIdx.x >= b.first[k + 1]) ++k;
    const n2d2hip_sat_weight_grad_item& t = b.item[k];
    const float* __restrict__ dq = t.diff_wq;
    const float* __restrict__ w = t.w;
    float* __restrict__ dw = t.diff_w;
    const float mode_factor = b.mode_factor[k], inv_factor = sat_weight_inv_factor(t);
    for (size_t i = (size_t)(blockIdx.x - b.first[k]) * QBLOCK + threadIdx.x; i < t.n; i += (size_t)(b.first[k + 1] - b.first[k]) * QBLOCK)
        dw[i] = sat_weight_gradient(w[i], dq[i], inv_factor, mode_factor);
}

// -------------------------------------------------------- SAT activations

// ref: SATQuantizer_Frame_Kernels.cpp:268-322 (std::round: half away from zero)
__global__ __launch_bounds__(QBLOCK) void sat_act_forward_kernel(float* __restrict__ x, float* __restrict__ fp, size_t n, float range,
                                                                 const float* __restrict__ alpha)
{
    const float a = fabsf(alpha[0]);
    for (size_t i = (size_t)blockIdx.x * QBLOCK + threadIdx.x; i < n; i += (size_t)gridDim.x * QBLOCK) {
        const float v = x[i];
        if (fp) fp[i] = v;
        x[i] = sat_quantize(v, range, a);
    }
}

// result[0] = (sum + beta * result[0]) * scale
struct Accumulate {
    float beta, scale;
    float* result;
    __device__ void operator()(double s) const
    {
        float acc = (float)s;
        if (beta != 0.0f)
            acc = __fadd_rn(acc, __fmul_rn(beta, result[0]));
        result[0] = __fmul_rn(acc, scale);
    }
};
// The end of a reducing pass: a single block (up to ONE_BLOCK values: a second launch would take longer than the rest of its
// loop) accumulates by itself, several leave their sums to accumulate_final
constexpr size_t ONE_BLOCK = 4096;
__device__ __forceinline__ void end_of_pass(double s, double* __restrict__ partial, const Accumulate& acc)
{
    s = block_sum(s);
    if (threadIdx.x) return;
    if (gridDim.x == 1) acc(s);
    else partial[blockIdx.x] = s;
}

// The inputs of a sum whose outputs the quantizer follows: each receives w times what passes the quantizer, + beta times what is there
struct SumGrads {
    float* dx[N2D2HIP_ELEMWISE_F32_MAX_INPUTS];
    float w[N2D2HIP_ELEMWISE_F32_MAX_INPUTS], beta[N2D2HIP_ELEMWISE_F32_MAX_INPUTS];
    int n;
};
// ref: SATQuantizer_Frame_Kernels.cpp:410-448; the alpha-gradient terms are summed instead of stored.  Memory bounds it.  SUM: the sum's
// inputs receive theirs in the same pass, which read the gradient again (64 x 64 x 32 x 32, two inputs, us: this and one pass for each
// input 11.4 + 5.5 + 5.5, now 19.7).
template <bool SUM>
__global__ __launch_bounds__(QBLOCK) void sat_act_backward_kernel(const float* dy, const float* __restrict__ fp,
                                                                  float* dx, size_t n, float range,
                                                                  const float* __restrict__ alpha, double* __restrict__ partial, int quads, Accumulate accumulate, SumGrads sum)
{
    const float a = fabsf(alpha[0]);
    double s = 0.0;
    for_quads(n, quads, [&](auto k, size_t i) {
        constexpr int N = decltype(k)::value;
        float x[N], g[N], d[N];
        quad_load<N>(x, fp, i);
        quad_load<N>(g, dy, i);
#pragma unroll
        for (int j = 0; j < N; ++j) {
            s += (double)__fmul_rn(sat_alpha_slope(x[j], range, a), g[j]);
            d[j] = __fmul_rn(sat_input_slope(x[j], a), g[j]);
        }
        quad_store<N>(dx, i, d);
        if constexpr (SUM) {
#pragma unroll
            for (int m = 0; m < N2D2HIP_ELEMWISE_F32_MAX_INPUTS; ++m) {
                if (m >= sum.n) break;
                float o[N];              // (an input that is there twice is read as its first part left it)
                if (sum.beta[m] != 0.0f) quad_load<N>(o, sum.dx[m], i);
#pragma unroll
                for (int j = 0; j < N; ++j) {
                    const float t = __fmul_rn(sum.w[m], d[j]);
                    o[j] = sum.beta[m] != 0.0f ? __fadd_rn(t, __fmul_rn(sum.beta[m], o[j])) : t;
                }
                quad_store<N>(sum.dx[m], i, o);
            }
        }
    });
    end_of_pass(s, partial, accumulate);
}
__global__ __launch_bounds__(QBLOCK) void accumulate_final(const double* __restrict__ partial, int count, Accumulate acc)
{
    double s = 0.0;
    for (int i = threadIdx.x; i < count; i += QBLOCK) s += partial[i];
    s = block_sum(s);
    if (threadIdx.x == 0) acc(s);
}

// -------------------------------------------------------------------- LSQ

// ref: LSQQuantizerCell_Frame.cpp:194-208, LSQQuantizerActivation_Frame.cpp:131-141
__global__ __launch_bounds__(QBLOCK) void lsq_forward_kernel(const float* __restrict__ x, float* __restrict__ xq, size_t n,
                                                             const float* __restrict__ step, int lo, int hi)
{
    const float s = step[0];
    const float lob = __fmul_rn((float)lo, s), hib = __fmul_rn((float)hi, s);
    for (size_t i = (size_t)blockIdx.x * QBLOCK + threadIdx.x; i < n; i += (size_t)gridDim.x * QBLOCK) {
        const float q = x[i] / s;
        xq[i] = (q <= (float)lo) ? lob : (q >= (float)hi) ? hib : __fmul_rn(round_half_away(q), s);
    }
}
// ref: LSQQuantizerCell_Frame.cpp:234-303, LSQQuantizerActivation_Frame.cpp:193-262
__global__ __launch_bounds__(QBLOCK) void lsq_backward_kernel(const float* dq, const float* __restrict__ fp,
                                                              float* dfp, size_t n, const float* __restrict__ step,
                                                              int lo, int hi, double* __restrict__ partial, int quads, Accumulate accumulate)
{
    const float s = step[0];
    double acc = 0.0;
    for_quads(n, quads, [&](auto k, size_t i) {
        constexpr int N = decltype(k)::value;
        float x[N], g[N], d[N];
        quad_load<N>(x, fp, i);
        quad_load<N>(g, dq, i);
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const float q = x[j] / s;
            const bool below = q <= (float)lo, above = q >= (float)hi;
            d[j] = __fmul_rn(g[j], (below || above) ? 0.0f : 1.0f);
            const float term = below ? (float)lo : above ? (float)hi : __fsub_rn(round_half_away(q), q);
            acc += (double)__fmul_rn(term, g[j]);
        }
        quad_store<N>(dfp, i, d);
    });
    end_of_pass(acc, partial, accumulate);
}

int sat_weight_grad_check(const n2d2hip_sat_weight_grad_item& t)
{
    N2D2HIP_REQUIRE(t.diff_wq && t.w && t.diff_w && t.stats, N2D2HIP_ERR_INVALID, "sat_weight_backward: null argument");
    N2D2HIP_REQUIRE(t.n > 0, N2D2HIP_ERR_INVALID, "sat_weight_backward: empty tensor");
    N2D2HIP_REQUIRE(t.mode >= N2D2HIP_SAT_NONE && t.mode <= N2D2HIP_SAT_NONE_ASYM, N2D2HIP_ERR_INVALID, "sat_weight_backward: bad mode %d", t.mode);
    return N2D2HIP_OK;
}

} // namespace n2d2hip

using namespace n2d2hip;

namespace {
int blocks_for(size_t n)
{
    size_t b = (n + QBLOCK - 1) / QBLOCK;
    return (int)std::max<size_t>(1, std::min<size_t>(b, PARTIALS));
}
int quads_of(const float* a, const float* b, const float* c) { return (((size_t)a | (size_t)b | (size_t)c) & 15) == 0; }
unsigned ew_grid(size_t n)
{
    size_t b = (n + QBLOCK - 1) / QBLOCK;
    return (unsigned)std::max<size_t>(1, std::min<size_t>(b, 256 * 32));
}
} // namespace

// Scratch of the entry point that allocates nothing: the block partials and the mean of the SAT weight quantizer's
// reductions.  Every GPU the library runs on holds its own copy of this array until the process ends.  In host code the
// array's name is only a handle for hipGetSymbolAddress, never a device address.
constexpr size_t STATIC_SCRATCH_BYTES = (size_t)PARTIALS * sizeof(double) + 256;
static __device__ __align__(256) unsigned char scratch[STATIC_SCRATCH_BYTES];

namespace {
constexpr int MAX_DEVICES = 64;
std::mutex scratch_mutex;
void* scratch_ptr[MAX_DEVICES] = {};     // device address of `scratch` on each device, looked up once per device

// Device address of the current device's copy of `scratch`; no allocation.
int static_scratch(void** ptr)
{
    int dev = 0;
    N2D2HIP_HIP_CHECK(hipGetDevice(&dev));
    N2D2HIP_REQUIRE(dev >= 0 && dev < MAX_DEVICES, N2D2HIP_ERR_UNSUPPORTED, "static scratch: device ordinal %d (at most %d devices)", dev, MAX_DEVICES);
    std::lock_guard<std::mutex> lock(scratch_mutex);
    if (!scratch_ptr[dev]) {
        void* p = nullptr;
        N2D2HIP_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        N2D2HIP_REQUIRE(p != nullptr, N2D2HIP_ERR_HIP, "static scratch: hipGetSymbolAddress returned a null address");
        scratch_ptr[dev] = p;
    }
    *ptr = scratch_ptr[dev];
    return N2D2HIP_OK;
}
} // namespace

// The launches of up to SAT_ITEMS tensors' SAT weight quantizers, each over a workspace of n2d2hip_quantizer_workspace_bytes().
template <int N>
static void sat_weight_launch(const n2d2hip_sat_weight_item* items, int count, hipStream_t st)
{
    SatBatch<N> b = {};
    b.count = count;
    int threads = QBLOCK;
    for (int i = 0; i < count; ++i)
        if (items[i].apply_scaling && items[i].n >= SAT_MANY) threads = 1024;
    const auto blocks = [&](size_t n, int most) {
        return (unsigned)std::min<size_t>(threads == QBLOCK ? (n + QBLOCK - 1) / QBLOCK : (n + 8191) / 8192 * 8, most);
    };
    for (int i = 0; i < count; ++i) {
        const size_t n = items[i].n;
        const SatKind kind = sat_kind(items[i]);
        const bool scaled = items[i].apply_scaling && kind != SatKind::SMALL;
        b.item[i] = items[i];
        b.first[i + 1] = b.first[i] + (kind == SatKind::SMALL ? 1u : kind == SatKind::SELF ? (unsigned)((n + 1023) / 1024)
                                                                                           : (unsigned)std::min<size_t>((n + 8191) / 8192 * 8, SAT_BLOCKS));
        b.first2[i + 1] = b.first2[i] + (kind != SatKind::MANY ? 0u : blocks(n, scaled ? SAT_BLOCKS_SUMS : SAT_BLOCKS2 * QBLOCK / threads));
        b.first3[i + 1] = b.first3[i] + (scaled ? blocks(n, SAT_BLOCKS2 * QBLOCK / threads) : 0u);
    }
    static_assert(SAT_SUMS % sizeof(double2) == 0 && SAT_SUMS + SAT_BLOCKS_SUMS * sizeof(double2) <= (size_t)PARTIALS * sizeof(double) + 256,
                  "a workspace holds the maxima and the sums");
    static_assert((SAT_SELF + 1023) / 1024 <= SAT_BLOCKS_SUMS, "of the blocks that look for the largest weight themselves too");
    N2D2HIP_LAUNCH_T(sat_weight_first_kernel, (N), dim3(b.first[count]), dim3(1024), 0, st, b);
    if (b.first2[count])
        N2D2HIP_LAUNCH_T(sat_weight_second_kernel, (N), dim3(b.first2[count]), dim3(threads), 0, st, b);
    if (b.first3[count])
        N2D2HIP_LAUNCH_T(sat_weight_scale_kernel, (N), dim3(b.first3[count]), dim3(threads), 0, st, b);
}

template <int N>
static void sat_weight_backward_launch(const n2d2hip_sat_weight_grad_item* items, int count, hipStream_t st)
{
    SatGradBatch<N> b = {};
    b.count = count;
    for (int i = 0; i < count; ++i) {
        const n2d2hip_sat_weight_grad_item& t = items[i];
        b.item[i] = t;
        b.first[i + 1] = b.first[i] + ew_grid(t.n);
        b.mode_factor[i] = sat_weight_mode_factor(t);
    }
    hipLaunchKernelGGL(sat_weight_backward_kernel<N>, dim3(b.first[count]), dim3(QBLOCK), 0, st, b);
}

extern "C" {

size_t n2d2hip_quantizer_workspace_bytes(size_t) { return (size_t)PARTIALS * sizeof(double) + 256; }

static int sat_weight_forward_impl(const char* who, const n2d2hip_sat_weight_item* items, int count, hipStream_t st)
{
    for (int i = 0; i < count; ++i) {
        const n2d2hip_sat_weight_item& t = items[i];
        N2D2HIP_REQUIRE(t.n > 0, N2D2HIP_ERR_INVALID, "%s: empty tensor", who);
        N2D2HIP_REQUIRE(t.mode >= N2D2HIP_SAT_NONE && t.mode <= N2D2HIP_SAT_NONE_ASYM, N2D2HIP_ERR_INVALID, "%s: bad mode %d", who, t.mode);
        N2D2HIP_REQUIRE(t.range >= 1.0f, N2D2HIP_ERR_INVALID, "%s: range %g", who, (double)t.range);
        N2D2HIP_REQUIRE(!t.apply_scaling || t.n > 1, N2D2HIP_ERR_INVALID, "%s: SAT scaling needs more than one weight", who);
    }
    for (int i = 0; i < count; i += SAT_ITEMS) {
        const int nb = std::min(count - i, SAT_ITEMS);
        if (nb == 1) sat_weight_launch<1>(items + i, nb, st);
        else sat_weight_launch<SAT_ITEMS>(items + i, nb, st);
    }
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

int n2d2hip_sat_weight_forward_batch(const n2d2hip_sat_weight_item* items, int count, n2d2hip_stream_t stream_)
{
    N2D2HIP_REQUIRE(items && count > 0, N2D2HIP_ERR_INVALID, "sat_weight_forward_batch: bad argument");
    for (int i = 0; i < count; ++i) {
        N2D2HIP_REQUIRE(items[i].w && items[i].wq && items[i].stats && items[i].workspace, N2D2HIP_ERR_INVALID, "sat_weight_forward_batch: null argument");
        N2D2HIP_REQUIRE(items[i].workspace_bytes >= n2d2hip_quantizer_workspace_bytes(items[i].n), N2D2HIP_ERR_WORKSPACE,
                        "sat_weight_forward_batch: workspace of %zu bytes needed", n2d2hip_quantizer_workspace_bytes(items[i].n));
    }
    return sat_weight_forward_impl("sat_weight_forward_batch", items, count, (hipStream_t)stream_);
}

int n2d2hip_sat_weight_forward(const float* w, float* wq, size_t n, float range, int mode, int apply_scaling,
                               unsigned outputs_size, float* stats, void* workspace, size_t workspace_bytes, n2d2hip_stream_t stream_)
{
    N2D2HIP_REQUIRE(w && wq && stats && workspace, N2D2HIP_ERR_INVALID, "sat_weight_forward: null argument");
    N2D2HIP_REQUIRE(workspace_bytes >= n2d2hip_quantizer_workspace_bytes(n), N2D2HIP_ERR_WORKSPACE, "sat_weight_forward: workspace of %zu bytes needed",
                    n2d2hip_quantizer_workspace_bytes(n));
    const n2d2hip_sat_weight_item item = {w, wq, n, range, mode, apply_scaling, outputs_size, stats, workspace, workspace_bytes};
    return sat_weight_forward_impl("sat_weight_forward", &item, 1, (hipStream_t)stream_);
}

int n2d2hip_sat_weight_forward_static(const float* w, float* wq, size_t n, float range, int mode, int apply_scaling,
                                      unsigned outputs_size, float* stats, n2d2hip_stream_t stream_)
{
    N2D2HIP_REQUIRE(w && wq && stats, N2D2HIP_ERR_INVALID, "sat_weight_forward_static: null argument");
    N2D2HIP_REQUIRE(n <= (size_t)N2D2HIP_SAT_STATIC_MAX_WEIGHTS, N2D2HIP_ERR_UNSUPPORTED,
                    "sat_weight_forward_static: %zu weights, at most %zu are served from the static scratch; use n2d2hip_sat_weight_forward",
                    n, (size_t)N2D2HIP_SAT_STATIC_MAX_WEIGHTS);
    static_assert(STATIC_SCRATCH_BYTES >= (size_t)PARTIALS * sizeof(double) + sizeof(float), "scratch holds the partials and the mean");
    void* ws = nullptr;
    int rc = static_scratch(&ws);
    if (rc != N2D2HIP_OK)
        return rc;
    // Nothing in the scratch has to start from zero: every pass writes the partials it then reads (the same block count
    // both times), and the mean is written before it is read.
    const n2d2hip_sat_weight_item item = {w, wq, n, range, mode, apply_scaling, outputs_size, stats, ws, STATIC_SCRATCH_BYTES};
    return sat_weight_forward_impl("sat_weight_forward_static", &item, 1, (hipStream_t)stream_);
}

int n2d2hip_sat_weight_backward_batch(const n2d2hip_sat_weight_grad_item* items, int count, n2d2hip_stream_t stream_)
{
    N2D2HIP_REQUIRE(items && count > 0, N2D2HIP_ERR_INVALID, "sat_weight_backward: bad argument");
    for (int i = 0; i < count; ++i) {
        const int rc = sat_weight_grad_check(items[i]);
        if (rc != N2D2HIP_OK) return rc;
    }
    for (int i = 0; i < count; i += SAT_ITEMS) {
        const int nb = std::min(count - i, SAT_ITEMS);
        if (nb == 1) sat_weight_backward_launch<1>(items + i, nb, (hipStream_t)stream_);
        else sat_weight_backward_launch<SAT_ITEMS>(items + i, nb, (hipStream_t)stream_);
    }
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

int n2d2hip_sat_weight_backward(const float* diff_wq, const float* w, float* diff_w, size_t n, float range, int mode,
                                int apply_scaling, const float* stats, n2d2hip_stream_t stream_)
{
    const n2d2hip_sat_weight_grad_item item = {diff_wq, w, diff_w, n, range, mode, apply_scaling, stats};
    return n2d2hip_sat_weight_backward_batch(&item, 1, stream_);
}

int n2d2hip_sat_act_forward(float* x, float* fp_copy, size_t n, float range, const float* alpha, n2d2hip_stream_t stream_)
{
    N2D2HIP_REQUIRE(x && alpha, N2D2HIP_ERR_INVALID, "sat_act_forward: null argument");
    N2D2HIP_REQUIRE(n > 0, N2D2HIP_ERR_INVALID, "sat_act_forward: empty tensor");
    hipLaunchKernelGGL(sat_act_forward_kernel, dim3(ew_grid(n)), dim3(QBLOCK), 0, (hipStream_t)stream_, x, fp_copy, n, range, alpha);
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

int n2d2hip_sat_act_backward(const float* diff_in, const float* fp_x, float* diff_out, size_t n, float range, const float* alpha,
                             float beta, float* diff_alpha, void* workspace, size_t workspace_bytes, n2d2hip_stream_t stream_)
{
    hipStream_t st = (hipStream_t)stream_;
    N2D2HIP_REQUIRE(diff_in && fp_x && diff_out && alpha && diff_alpha && workspace, N2D2HIP_ERR_INVALID, "sat_act_backward: null argument");
    N2D2HIP_REQUIRE(n > 0, N2D2HIP_ERR_INVALID, "sat_act_backward: empty tensor");
    N2D2HIP_REQUIRE(workspace_bytes >= n2d2hip_quantizer_workspace_bytes(n), N2D2HIP_ERR_WORKSPACE, "sat_act_backward: workspace of %zu bytes needed",
                    n2d2hip_quantizer_workspace_bytes(n));
    const int nb = n <= ONE_BLOCK ? 1 : blocks_for(n);
    const Accumulate acc = {beta, 1.0f, diff_alpha};
    double* partial = (double*)workspace;
    hipLaunchKernelGGL(sat_act_backward_kernel<false>, dim3(nb), dim3(QBLOCK), 0, st, diff_in, fp_x, diff_out, n, range, alpha, partial,
                       quads_of(diff_in, fp_x, diff_out), acc, SumGrads{});
    if (nb > 1) hipLaunchKernelGGL(accumulate_final, dim3(1), dim3(QBLOCK), 0, st, (const double*)partial, nb, acc);
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

int n2d2hip_elemwise_sum_f32_backward_sat(int nb_inputs, size_t n, const float* weights, const float* betas, float* const* diff_x, float* diff_y,
                                          const float* full_precision, float range, const float* alpha, float beta_alpha, float* diff_alpha,
                                          void* workspace, size_t workspace_bytes, n2d2hip_stream_t stream_)
{
    hipStream_t st = (hipStream_t)stream_;
    const char* who = "n2d2hip_elemwise_sum_f32_backward_sat";
    N2D2HIP_REQUIRE(nb_inputs >= 0 && (nb_inputs == 0 || (weights && betas && diff_x)) && diff_y && full_precision && alpha && diff_alpha && workspace && n > 0
                        && full_precision != diff_y,
                    N2D2HIP_ERR_INVALID, "%s: bad argument", who);
    N2D2HIP_REQUIRE(nb_inputs <= N2D2HIP_ELEMWISE_F32_MAX_INPUTS, N2D2HIP_ERR_UNSUPPORTED, "%s: at most %d inputs", who, N2D2HIP_ELEMWISE_F32_MAX_INPUTS);
    N2D2HIP_REQUIRE(workspace_bytes >= n2d2hip_quantizer_workspace_bytes(n), N2D2HIP_ERR_WORKSPACE, "%s: workspace of %zu bytes needed", who,
                    n2d2hip_quantizer_workspace_bytes(n));
    SumGrads sum = {};
    sum.n = nb_inputs;
    int quads = quads_of(diff_y, full_precision, nullptr);
    for (int k = 0; k < nb_inputs; ++k) {
        N2D2HIP_REQUIRE(diff_x[k], N2D2HIP_ERR_INVALID, "%s: input %d is null", who, k);
        sum.dx[k] = diff_x[k];
        sum.w[k] = weights[k];
        sum.beta[k] = betas[k];
        quads &= quads_of(diff_x[k], nullptr, nullptr);
    }
    const int nb = n <= ONE_BLOCK ? 1 : blocks_for(n);
    const Accumulate acc = {beta_alpha, 1.0f, diff_alpha};
    double* partial = (double*)workspace;
    hipLaunchKernelGGL(sat_act_backward_kernel<true>, dim3(nb), dim3(QBLOCK), 0, st, diff_y, full_precision, diff_y, n, range, alpha, partial, quads, acc, sum);
    if (nb > 1) hipLaunchKernelGGL(accumulate_final, dim3(1), dim3(QBLOCK), 0, st, (const double*)partial, nb, acc);
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

int n2d2hip_lsq_forward(const float* x, float* xq, size_t n, const float* step, int lo, int hi, n2d2hip_stream_t stream_)
{
    N2D2HIP_REQUIRE(x && xq && step, N2D2HIP_ERR_INVALID, "lsq_forward: null argument");
    N2D2HIP_REQUIRE(n > 0 && lo < hi, N2D2HIP_ERR_INVALID, "lsq_forward: empty tensor or empty range [%d,%d]", lo, hi);
    hipLaunchKernelGGL(lsq_forward_kernel, dim3(ew_grid(n)), dim3(QBLOCK), 0, (hipStream_t)stream_, x, xq, n, step, lo, hi);
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

int n2d2hip_lsq_backward(const float* diff_q, const float* fp_x, float* diff_fp, size_t n, const float* step, int lo, int hi,
                         float grad_scale, float beta, float* diff_step, void* workspace, size_t workspace_bytes, n2d2hip_stream_t stream_)
{
    hipStream_t st = (hipStream_t)stream_;
    N2D2HIP_REQUIRE(diff_q && fp_x && diff_fp && step && diff_step && workspace, N2D2HIP_ERR_INVALID, "lsq_backward: null argument");
    N2D2HIP_REQUIRE(n > 0 && lo < hi, N2D2HIP_ERR_INVALID, "lsq_backward: empty tensor or empty range [%d,%d]", lo, hi);
    N2D2HIP_REQUIRE(workspace_bytes >= n2d2hip_quantizer_workspace_bytes(n), N2D2HIP_ERR_WORKSPACE, "lsq_backward: workspace of %zu bytes needed",
                    n2d2hip_quantizer_workspace_bytes(n));
    const int nb = n <= ONE_BLOCK ? 1 : blocks_for(n);
    const Accumulate acc = {beta, grad_scale, diff_step};
    double* partial = (double*)workspace;
    hipLaunchKernelGGL(lsq_backward_kernel, dim3(nb), dim3(QBLOCK), 0, st, diff_q, fp_x, diff_fp, n, step, lo, hi, partial,
                       quads_of(diff_q, fp_x, diff_fp), acc);
    if (nb > 1) hipLaunchKernelGGL(accumulate_final, dim3(1), dim3(QBLOCK), 0, st, (const double*)partial, nb, acc);
    N2D2HIP_HIP_CHECK(hipGetLastError());
    return N2D2HIP_OK;
}

} // extern "C"
