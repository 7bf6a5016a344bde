// hadamard_kernels.hip -- the block-128 transforms of the incoherence step
// (had_left and had_right, quantize.py:134-145), with the channel scales of
// to_inner and from_inner (quantize.py:148-163) folded in where both sides are
// transformed.
//
// Every output is one fp32 fused multiply-add chain over its 128 products in
// ascending order, from zero, as torch's CPU sgemm evaluates the reference's
// matmul (measured bit for bit against an fmaf chain).  That order leaves the
// matrix cores one product per output and instruction: v_mfma_f32_32x32x1f32
// (two 32x32 blocks, k = 1) adds each product to its accumulator with one
// rounding.  It runs 32 multiply-adds a cycle and SIMD, against 16 for the
// v_fma_f32 with a scalar operand that these kernels used before (an SGPR
// operand puts it at the 4-cycle rate), and takes 2 operand registers per 2048
// multiply-adds.  Bound: those 128 multiply-adds per output (17408x5120:
// 0.15 ms at 2.35 GHz, against 0.13 ms for its 713 MB at 5.5 TB/s).
//
// In had_left and had_right a wave keeps its 32 rows (columns) of the
// multipliers in 128 VGPRs and takes one 64-wide tile after the other; 2 waves
// per SIMD (17408x5120: had_left 0.48 -> 0.26, had_right 0.76 -> 0.24 ms).
// had_both takes both sides of a 128x128 block without leaving the CU.
#include "viterbi_kernels.h"

#pragma clang fp contract(off)

namespace xtq {
namespace {

typedef float v32f __attribute__((ext_vector_type(32)));
typedef float f32x4_t __attribute__((ext_vector_type(4), aligned(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

// Most workgroups of a launch, two (had_both: one) for each of the MI355X's 256
// CUs; they take the tiles in turn, so any number of CUs is right.
constexpr int kHadGroups = 512;
constexpr int kHadBothGroups = 256;

// Row of accumulator register v in its 32x32 block, for the lane's half.
__device__ __forceinline__ int acc_row(int v, int ln) {
    return 8 * ((v >> 2) & 3) + 4 * (ln >> 5) + (v & 3);
}

// out[128b + r][c] = sum_t ht[t][r] x[128b + t][c].  Workgroup: one 128-row
// block of 64 columns at a time, wave w its output rows 32w .. 32w+31.  The
// tile waits in LDS (every wave reads all of it), the next one's loads in
// flight in registers: 32 KiB per workgroup, which is what hides the HBM
// latency (each wave loading its operands 16 rows ahead, without LDS, took
// twice the time).
__global__ __launch_bounds__(256, 2) void had_left_kernel(const float* __restrict__ ht,
                                                          const float* __restrict__ in,
                                                          float* __restrict__ out, int nblk,
                                                          int cols) {
    __shared__ float tile[128 * 64];
    constexpr int NV = 32;                              // elements per thread and tile
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ln = threadIdx.x & 63;
    float h[128];
#pragma unroll
    for (int t = 0; t < 128; ++t) h[t] = ht[t * 128 + 32 * wv + (ln & 31)];
    const int nct = (cols + 63) / 64, items = nblk * nct;
    float nx[NV];
    // wave w loads rows w, w + 4, ..
    auto load = [&](int item) __attribute__((always_inline)) {
        const int blk = item / nct, c = (item - blk * nct) * 64 + ln;
        const int ci = c < cols ? c : cols - 1;         // a valid column; its sums are not stored
        const float* src = in + ((size_t)blk * 128 + wv) * cols;
#pragma unroll
        for (int i = 0; i < NV; ++i) nx[i] = src[(size_t)(4 * i) * cols + ci];
    };
    if ((int)blockIdx.x < items) load(blockIdx.x);
    for (int item = blockIdx.x; item < items; item += gridDim.x) {
        const int blk = item / nct, c0 = (item - blk * nct) * 64;
        __syncthreads();                                // the previous tile is read
#pragma unroll
        for (int i = 0; i < NV; ++i) tile[(wv + 4 * i) * 64 + ln] = nx[i];
        __syncthreads();
        if (item + (int)gridDim.x < items) load(item + gridDim.x);
        v32f acc;
#pragma unroll
        for (int v = 0; v < 32; ++v) acc[v] = 0.0f;
#pragma unroll
        for (int t = 0; t < 128; ++t)
            acc = __builtin_amdgcn_mfma_f32_32x32x1f32(h[t], tile[t * 64 + ln], acc, 0, 0, 0);
#pragma unroll
        for (int v = 0; v < 32; ++v) {
            const int r = blk * 128 + 32 * wv + acc_row(v, ln);
            const int c = c0 + 32 * (v >> 4) + (ln & 31);
            if (c < cols) out[(size_t)r * cols + c] = acc[v];
        }
    }
}

// out[r][128b + c] = sum_t h[t][c] in[r][128b + t].  Workgroup: 64 rows of one
// 128-column block at a time, wave w its output columns 32w .. 32w+31.  The
// tile waits in LDS at a row stride of 132 floats (16-byte reads of 64 rows
// spread over all banks), the next one's loads in flight in registers.
constexpr int kHrRows = 64;
constexpr int kHrStride = 132;

__global__ __launch_bounds__(256, 2) void had_right_kernel(const float* __restrict__ hm,
                                                           const float* __restrict__ in,
                                                           float* __restrict__ out, int rows,
                                                           int cols) {
    __shared__ __attribute__((aligned(16))) float tile[kHrRows * kHrStride];
    constexpr int NV = kHrRows * 32 / 256;              // float4s per thread and tile
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ln = threadIdx.x & 63;
    float h[128];
#pragma unroll
    for (int t = 0; t < 128; ++t) h[t] = hm[t * 128 + 32 * wv + (ln & 31)];
    const int ncb = cols / 128, items = ((rows + kHrRows - 1) / kHrRows) * ncb;
    f32x4_t nx[NV];
    auto load = [&](int item) __attribute__((always_inline)) {
        const int rt = item / ncb, b = item - rt * ncb;
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int idx = threadIdx.x + 256 * i, rr = kHrRows * rt + (idx >> 5);
            const int r = rr < rows ? rr : rows - 1;    // a valid row; its sums are not stored
            nx[i] = *(const f32x4_t*)(in + (size_t)r * cols + 128 * b + 4 * (idx & 31));
        }
    };
    if ((int)blockIdx.x < items) load(blockIdx.x);
    for (int item = blockIdx.x; item < items; item += gridDim.x) {
        const int rt = item / ncb, b = item - rt * ncb;
        __syncthreads();                                // the previous tile is read
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int idx = threadIdx.x + 256 * i;
            *(v4f*)(tile + (idx >> 5) * kHrStride + 4 * (idx & 31)) = nx[i];
        }
        __syncthreads();
        if (item + (int)gridDim.x < items) load(item + gridDim.x);
        v32f acc;
#pragma unroll
        for (int v = 0; v < 32; ++v) acc[v] = 0.0f;
        const float* row = tile + ln * kHrStride;
#pragma unroll
        for (int t = 0; t < 128; t += 4) {
            const v4f x = *(const v4f*)(row + t);
            acc = __builtin_amdgcn_mfma_f32_32x32x1f32(x.x, h[t], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x1f32(x.y, h[t + 1], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x1f32(x.z, h[t + 2], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x1f32(x.w, h[t + 3], acc, 0, 0, 0);
        }
        const int c = 128 * b + 32 * wv + (ln & 31);
#pragma unroll
        for (int v = 0; v < 32; ++v) {
            const int r = kHrRows * rt + 32 * (v >> 4) + acc_row(v, ln);
            if (r < rows) out[(size_t)r * cols + c] = acc[v];
        }
    }
}

// to_inner and from_inner: both sides of the 128x128 blocks,
//     y = (sum_t h[r][t] x[t][c]) [* mr[row]],  out = (sum_t y[r][t] h[t][c]) [* mc[column]],
// in the products and order of had_left followed by had_right.  DIV (to_inner):
// x = (in / dr[row]) / dc[column], two rounded divisions as torch's; MUL
// (from_inner): the factors in brackets.  The transforms only mix within a
// block, so y never leaves the CU: one 512-thread workgroup per CU holds the
// block and the multipliers in LDS (rows of 132 floats: 16-byte reads down 32
// or 64 rows, and 4-byte reads along a row, spread over all banks), the next
// block's loads in flight in registers.  A wave sums a 32x64 part of y, and
// after the barrier a 64x32 part of the output.  Bound: the 256 multiply-adds
// per output at 32 a cycle and SIMD (17408x5120: 0.30 ms, the traffic of one
// read and one write 0.13 ms), to which the divisions, the LDS round trip and
// the four barriers of a block add.  to_inner + from_inner, against the two
// passes with the scales folded in that this replaces / against separate passes
// for the scales too: 17408x5120 975 / 2965 -> 876 us (876 to 1012 by the
// device's clock), 4096x4096 211 / 460 -> 178, 1024x1024 76 / 104 -> 52 (host
// side of two calls).
template <bool DIV, bool MUL>
__global__ __launch_bounds__(512, 2) void had_both_kernel(
    const float* __restrict__ hm, const float* __restrict__ in, float* __restrict__ out,
    int nrb, int cols, const float* __restrict__ rs, const float* __restrict__ cs) {
    constexpr int S = kHrStride, NV = 128 * 32 / 512;   // float4s per thread and block
    __shared__ __attribute__((aligned(16))) float H[128 * S], T[128 * S];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ln = threadIdx.x & 63;
    const int w32 = 32 * (wv & 3), w64 = 64 * (wv >> 2);
    const int r0 = threadIdx.x >> 5, c4 = 4 * (threadIdx.x & 31);   // loads: rows r0 + 16 i
    const int ncb = cols / 128, items = nrb * ncb;
#pragma unroll
    for (int i = 0; i < NV; ++i)
        *(v4f*)(H + (r0 + 16 * i) * S + c4) = *(const f32x4_t*)(hm + (r0 + 16 * i) * 128 + c4);
    f32x4_t nx[NV];
    auto load = [&](int item) __attribute__((always_inline)) {
        const int rb = item / ncb, b = item - rb * ncb;
        const float* src = in + ((size_t)rb * 128 + r0) * cols + 128 * b + c4;
#pragma unroll
        for (int i = 0; i < NV; ++i) nx[i] = *(const f32x4_t*)(src + (size_t)(16 * i) * cols);
    };
    if ((int)blockIdx.x < items) load(blockIdx.x);
    for (int item = blockIdx.x; item < items; item += gridDim.x) {
        const int rb = item / ncb, b = item - rb * ncb;
        if constexpr (DIV) {
            const f32x4_t d = *(const f32x4_t*)(cs + 128 * b + c4);
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                const float r = rs[rb * 128 + r0 + 16 * i];
                nx[i].x = (nx[i].x / r) / d.x;
                nx[i].y = (nx[i].y / r) / d.y;
                nx[i].z = (nx[i].z / r) / d.z;
                nx[i].w = (nx[i].w / r) / d.w;
            }
        }
        __syncthreads();                                // the previous block is read
#pragma unroll
        for (int i = 0; i < NV; ++i) *(v4f*)(T + (r0 + 16 * i) * S + c4) = nx[i];
        __syncthreads();
        if (item + (int)gridDim.x < items) load(item + gridDim.x);
        v32f acc;
#pragma unroll
        for (int v = 0; v < 32; ++v) acc[v] = 0.0f;
#pragma unroll 8
        for (int t = 0; t < 128; t += 4) {
            const v4f a = *(const v4f*)(H + (w32 + (ln & 31)) * S + t);
            const float* x = T + t * S + w64 + ln;
            acc = __builtin_amdgcn_mfma_f32_32x32x1f32(a.x, x[0], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x1f32(a.y, x[S], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x1f32(a.z, x[2 * S], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x1f32(a.w, x[3 * S], acc, 0, 0, 0);
        }
        __syncthreads();                                // every wave has read the block
#pragma unroll
        for (int v = 0; v < 32; ++v) {
            const int r = w32 + acc_row(v, ln), c = w64 + 32 * (v >> 4) + (ln & 31);
            T[r * S + c] = MUL ? acc[v] * rs[rb * 128 + r] : acc[v];
        }
        __syncthreads();
#pragma unroll
        for (int v = 0; v < 32; ++v) acc[v] = 0.0f;
#pragma unroll 8
        for (int t = 0; t < 128; t += 4) {
            const v4f a = *(const v4f*)(T + (w64 + ln) * S + t);
            const float* x = H + t * S + w32 + (ln & 31);
            acc = __builtin_amdgcn_mfma_f32_32x32x1f32(a.x, x[0], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x1f32(a.y, x[S], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x1f32(a.z, x[2 * S], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x1f32(a.w, x[3 * S], acc, 0, 0, 0);
        }
        const int c = 128 * b + w32 + (ln & 31);
        const float m = MUL ? cs[c] : 1.0f;
#pragma unroll
        for (int v = 0; v < 32; ++v) {
            const int r = 128 * rb + w64 + 32 * (v >> 4) + acc_row(v, ln);
            out[(size_t)r * cols + c] = MUL ? acc[v] * m : acc[v];
        }
    }
}

}  // namespace

hipError_t launch_had_left(const float* ht, const float* in, float* out, int rows, int cols,
                           hipStream_t stream) {
    if (rows <= 0 || cols <= 0) return hipSuccess;
    if (rows % 128 || rows / 128 > 65535) return hipErrorInvalidValue;
    const int nblk = rows / 128;
    const long long items = (long long)nblk * ((cols + 63LL) / 64);
    if (items > INT32_MAX - kHadGroups) return hipErrorInvalidValue;
    const dim3 grid((uint32_t)(items < kHadGroups ? items : kHadGroups));
    hipLaunchKernelGGL(had_left_kernel, grid, dim3(256), 0, stream, ht, in, out, nblk, cols);
    return hipGetLastError();
}

hipError_t launch_had_right(const float* h, const float* in, float* out, int rows, int cols,
                            hipStream_t stream) {
    if (rows <= 0 || cols <= 0) return hipSuccess;
    if (cols % 128) return hipErrorInvalidValue;
    const long long items = ((rows + (long long)kHrRows - 1) / kHrRows) * (cols / 128);
    if (items > INT32_MAX - kHadGroups) return hipErrorInvalidValue;
    const dim3 grid((uint32_t)(items < kHadGroups ? items : kHadGroups));
    hipLaunchKernelGGL(had_right_kernel, grid, dim3(256), 0, stream, h, in, out, rows, cols);
    return hipGetLastError();
}

hipError_t launch_had_both(const float* h, const float* in, float* out, int rows, int cols,
                           const float* row_scale, const float* col_scale, bool divide,
                           hipStream_t stream) {
    if (rows <= 0 || cols <= 0) return hipSuccess;
    if (rows % 128 || cols % 128 || !row_scale || !col_scale) return hipErrorInvalidValue;
    const long long items = (long long)(rows / 128) * (cols / 128);
    if (items > INT32_MAX - kHadBothGroups) return hipErrorInvalidValue;
    const dim3 grid((uint32_t)(items < kHadBothGroups ? items : kHadBothGroups));
    if (divide)
        hipLaunchKernelGGL((had_both_kernel<true, false>), grid, dim3(512), 0, stream, h, in, out,
                           rows / 128, cols, row_scale, col_scale);
    else
        hipLaunchKernelGGL((had_both_kernel<false, true>), grid, dim3(512), 0, stream, h, in, out,
                           rows / 128, cols, row_scale, col_scale);
    return hipGetLastError();
}

}  // namespace xtq
