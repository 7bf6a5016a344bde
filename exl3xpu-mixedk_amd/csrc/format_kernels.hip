// format_kernels.hip -- gfx950 kernels for the EXL3 trellis format: decode,
// pack and unpack (quantize.py:360-415).
//
// A tile is a 256 K-bit stream of 8K 32-bit words, MSB first: symbol t
// (s_t mod 2^K) at bits [tK, (t+1)K), and state t the 16-bit circular window
// that ends with symbol t's bits.  All three kernels move bytes: what bounds
// them is HBM, and their work is arranged so that a lane's fp32 values and
// states move 16 bytes at a time (fp16 values 8) and a wave's are contiguous.
// The trellis, a fifth of the bytes at most, moves in its 4-byte words.
#include "viterbi_kernels.h"

#pragma clang fp contract(off)

namespace xtq {
namespace {

// Global-memory vectors of the callers' alignment (the element's own): the
// accesses are as wide all the same, gfx950 takes them at any address.
typedef uint32_t u32_t __attribute__((aligned(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4), aligned(4)));
typedef _Float16 f16x4_t __attribute__((ext_vector_type(4), aligned(2)));
typedef int32_t i32x4_t __attribute__((ext_vector_type(4), aligned(4)));
typedef long i64x2_t __attribute__((ext_vector_type(2), aligned(8)));

// Window ending at bit `sh` from the bottom of word lo: (hi:lo) >> sh.
__device__ __forceinline__ uint32_t window(uint32_t hi, uint32_t lo, uint32_t sh) {
    return __builtin_amdgcn_alignbit(hi, lo, sh) & 0xFFFFu;
}

// Codebook value of state s, bit for bit the table's (quantize.py:56-87).
// Computed instead of looked up: 89 M lookups in the 256 KiB table go to L2,
// and took 0.45 ms of a 17408x5120 decode; these take a handful of
// instructions, 1mad's with those of a correctly rounded division.
//   mul1   (1024 + byte sum) c1 + c2 with c1 = 1774/2^18, c2 = -1329/2^7: every
//          term and the sum fit 24 bits, so the fp32 value is exact and only
//          the rounding to fp16 remains, as in the reference's fp64
//   1mad   (byte sum - 510) / 147.800537109375: the divisor is an fp32 number,
//          and one fp32 division gives the bits of the reference's fp64
//          division rounded to fp32 for all 1021 numerators
//   3inst, mcg   the exact sum of two halves, rounded once: an fp16 addition
template <int CODE>
__device__ __forceinline__ float code_value(uint32_t s) {
    if constexpr (CODE == kCodeMul1) {
        const uint32_t h = __builtin_amdgcn_sad_u8(s * 0x83DCD12Du, 0u, 1024u);
        return (float)(_Float16)__builtin_fmaf((float)h, 1774.0f / 262144.0f, -1329.0f / 128.0f);
    } else if constexpr (CODE == kCode1Mad) {
        const uint32_t h = __builtin_amdgcn_sad_u8(s * 34038481u + 76625530u, 0u, 0u);
        return ((float)h - 510.0f) / 147.800537109375f;
    } else {
        uint32_t x = CODE == kCode3Inst ? s * 89226354u + 64248484u : s * 0xCBAC1FEDu;
        x = (x & 0x8FFF8FFFu) ^ 0x3B603B60u;
        const _Float16 lo = __builtin_bit_cast(_Float16, (uint16_t)(x & 0xFFFFu));
        const _Float16 hi = __builtin_bit_cast(_Float16, (uint16_t)(x >> 16));
        return (float)(_Float16)(lo + hi);
    }
}

// decode_trellis (quantize.py:405-415).  A workgroup takes kDecTiles tiles
// side by side; lane l of wave w writes columns 4(l % 4) .. +3 of tile l / 4
// in rows 4w .. 4w+3, so a wave's store is 1 KiB of one output row.  Element
// (r, c) of a tile is symbol t = 32 (c % 8) + 8 ((r % 8) / 2) + 4 (c / 8) +
// 2 (r / 8) + r % 2 (tensor_core_perm, quantize.py:101-118): one column
// further is 32 symbols, K whole words, so the four columns of a lane share
// the bit offset.  The words wait in LDS with one word of padding per 4K (the
// distance between neighbouring lanes), or they would meet in a few banks.
// A 17408x5120 weight at K=4: 528 -> 76 us a call (401 MB, 5.3 TB/s); one
// 256-thread workgroup per tile with a table lookup and a 64-byte store row
// per tile before.
constexpr int kDecTiles = 16;

template <int K, int CODE>
__global__ __launch_bounds__(256) void decode_kernel(const int16_t* __restrict__ trellis, int tn,
                                                     int ng, float* __restrict__ out_f32,
                                                     uint16_t* __restrict__ out_f16) {
    constexpr int TW = 8 * K + 2;                       // words of a tile, padded
    __shared__ uint32_t words[kDecTiles * TW];
    const int a = blockIdx.x / ng, b0 = (blockIdx.x - a * ng) * kDecTiles;
    const int nt = (tn - b0) < kDecTiles ? (tn - b0) : kDecTiles;
    const u32_t* src = (const u32_t*)(trellis + ((size_t)a * tn + b0) * 16 * K);
    for (int i = threadIdx.x; i < nt * 8 * K; i += 256) words[i + i / (4 * K)] = src[i];
    __syncthreads();
    const int l = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int tile = l >> 2, q = l & 3;
    if (tile >= nt) return;
    const uint32_t* tw = words + tile * TW;
    const size_t n = (size_t)tn * 16;
    const int m0 = 4 * (q & 1);                         // c % 8 of the first column
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 4 * wv + i;
        const int t0 = 8 * ((r & 7) >> 1) + 4 * (q >> 1) + 2 * (r >> 3) + (r & 1);
        const int e0 = t0 * K + K - 1;                  // the window's last bit, column c % 8 = 0
        const uint32_t sh = 31u - ((uint32_t)e0 & 31u);
        const int w0 = (e0 >> 5) + K * m0;
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int lo = w0 + K * j, hi = lo > 0 ? lo - 1 : 8 * K - 1;
            v[j] = code_value<CODE>(window(tw[hi + hi / (4 * K)], tw[lo + lo / (4 * K)], sh));
        }
        const size_t idx = (size_t)(16 * a + r) * n + 16 * (size_t)(b0 + tile) + 4 * q;
        if (out_f32) {
            const f32x4_t o = {v[0], v[1], v[2], v[3]};
            *(f32x4_t*)(out_f32 + idx) = o;
        }
        if (out_f16) {
            const f16x4_t o = {(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
            *(f16x4_t*)(out_f16 + idx) = o;
        }
    }
}

// States of a tile from its packed words, one wave per tile: lane l < 8K holds
// word l, and the two words of a window come from their lanes.  S: int32_t, or
// int64_t as the host API's states.  16-byte stores: lane l writes states
// 4l .. 4l+3, or 2l, 2l+1 and 128 + 2l, 128 + 2l + 1.
constexpr int kFmtWaves = 4;                            // tiles per workgroup

template <int K, typename S>
__global__ __launch_bounds__(64 * kFmtWaves) void unpack_kernel(
    const int16_t* __restrict__ trellis, int nt, S* __restrict__ states) {
    const int tile = blockIdx.x * kFmtWaves + (threadIdx.x >> 6), l = threadIdx.x & 63;
    if (tile >= nt) return;
    const uint32_t word = ((const u32_t*)(trellis + (size_t)tile * 16 * K))[l < 8 * K ? l : 0];
    auto state = [&](int t) {
        const int e = t * K + K - 1, lo = e >> 5;
        const uint32_t wl = __shfl(word, lo), wh = __shfl(word, lo > 0 ? lo - 1 : 8 * K - 1);
        return window(wh, wl, 31u - ((uint32_t)e & 31u));
    };
    S* out = states + (size_t)tile * kSteps;
    if constexpr (sizeof(S) == 4) {
        const i32x4_t v = {(int32_t)state(4 * l), (int32_t)state(4 * l + 1),
                           (int32_t)state(4 * l + 2), (int32_t)state(4 * l + 3)};
        *(i32x4_t*)(out + 4 * l) = v;
    } else {
#pragma unroll
        for (int h = 0; h < 256; h += 128) {
            const i64x2_t v = {(long)state(h + 2 * l), (long)state(h + 2 * l + 1)};
            *(i64x2_t*)(out + h + 2 * l) = v;
        }
    }
}

// pack_states (quantize.py:360-378), one wave per tile: lane l joins the 4K
// symbol bits of states 4l .. 4l+3 (16-byte loads), and word lane w < 8K
// gathers the lanes whose bits its 32 cover.
template <int K, typename S>
__global__ __launch_bounds__(64 * kFmtWaves) void pack_kernel(const S* __restrict__ states, int nt,
                                                              int16_t* __restrict__ trellis) {
    constexpr uint32_t M = (1u << K) - 1;
    constexpr int CB = 4 * K;                           // bits per lane
    constexpr int NC = (31 + CB - 1) / CB + 1;          // lanes a word can touch
    const int tile = blockIdx.x * kFmtWaves + (threadIdx.x >> 6), l = threadIdx.x & 63;
    if (tile >= nt) return;
    const S* st = states + (size_t)tile * kSteps + 4 * l;
    uint32_t s[4];
    if constexpr (sizeof(S) == 4) {
        const i32x4_t v = *(const i32x4_t*)st;
#pragma unroll
        for (int i = 0; i < 4; ++i) s[i] = (uint32_t)v[i] & M;
    } else {
        const i64x2_t v0 = *(const i64x2_t*)st, v1 = *(const i64x2_t*)(st + 2);
        s[0] = (uint32_t)v0[0] & M;
        s[1] = (uint32_t)v0[1] & M;
        s[2] = (uint32_t)v1[0] & M;
        s[3] = (uint32_t)v1[1] & M;
    }
    const uint32_t chunk = (((((s[0] << K) | s[1]) << K) | s[2]) << K) | s[3];
    const int w = l < 8 * K ? l : 0, q0 = 32 * w / CB;
    uint32_t word = 0;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        const uint32_t c = __shfl(chunk, (q0 + i) & 63);
        const int up = 32 * w + 32 - CB * (q0 + i + 1);  // chunk's last bit above the word's
        if (up >= 0) word |= c << up;                    // (up < 32: the chunk starts by bit 32w + 31)
        else if (up > -CB) word |= c >> -up;
    }
    if (l < 8 * K) ((u32_t*)(trellis + (size_t)tile * 16 * K))[l] = word;
}

template <int K>
hipError_t decode_k(int code, const int16_t* tr, int tk, int tn, float* of, uint16_t* oh,
                    hipStream_t s) {
    const int ng = (tn - 1) / kDecTiles + 1;
    const dim3 grid((uint32_t)tk * (uint32_t)ng);
    switch (code) {
        case kCodeMul1:
            hipLaunchKernelGGL((decode_kernel<K, kCodeMul1>), grid, dim3(256), 0, s, tr, tn, ng, of, oh);
            break;
        case kCode3Inst:
            hipLaunchKernelGGL((decode_kernel<K, kCode3Inst>), grid, dim3(256), 0, s, tr, tn, ng, of, oh);
            break;
        case kCodeMcg:
            hipLaunchKernelGGL((decode_kernel<K, kCodeMcg>), grid, dim3(256), 0, s, tr, tn, ng, of, oh);
            break;
        case kCode1Mad:
            hipLaunchKernelGGL((decode_kernel<K, kCode1Mad>), grid, dim3(256), 0, s, tr, tn, ng, of, oh);
            break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int K, typename S>
hipError_t pack_k(const S* st, int nt, int16_t* tr, hipStream_t s) {
    hipLaunchKernelGGL((pack_kernel<K, S>), dim3((nt - 1) / kFmtWaves + 1),
                       dim3(64 * kFmtWaves), 0, s, st, nt, tr);
    return hipGetLastError();
}

template <int K, typename S>
hipError_t unpack_k(const int16_t* tr, int nt, S* st, hipStream_t s) {
    hipLaunchKernelGGL((unpack_kernel<K, S>), dim3((nt - 1) / kFmtWaves + 1),
                       dim3(64 * kFmtWaves), 0, s, tr, nt, st);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_decode(int K, int code, const int16_t* trellis, int tk, int tn, float* out_f32,
                         uint16_t* out_f16, hipStream_t stream) {
    if (tk <= 0 || tn <= 0) return hipSuccess;
    switch (K) {
        case 2: return decode_k<2>(code, trellis, tk, tn, out_f32, out_f16, stream);
        case 3: return decode_k<3>(code, trellis, tk, tn, out_f32, out_f16, stream);
        case 4: return decode_k<4>(code, trellis, tk, tn, out_f32, out_f16, stream);
        case 5: return decode_k<5>(code, trellis, tk, tn, out_f32, out_f16, stream);
        case 6: return decode_k<6>(code, trellis, tk, tn, out_f32, out_f16, stream);
        case 7: return decode_k<7>(code, trellis, tk, tn, out_f32, out_f16, stream);
        default: return hipErrorInvalidValue;
    }
}

template <typename S>
hipError_t launch_pack(int K, const S* states, int nt, int16_t* trellis, hipStream_t stream) {
    if (nt <= 0) return hipSuccess;
    switch (K) {
        case 2: return pack_k<2>(states, nt, trellis, stream);
        case 3: return pack_k<3>(states, nt, trellis, stream);
        case 4: return pack_k<4>(states, nt, trellis, stream);
        case 5: return pack_k<5>(states, nt, trellis, stream);
        case 6: return pack_k<6>(states, nt, trellis, stream);
        case 7: return pack_k<7>(states, nt, trellis, stream);
        default: return hipErrorInvalidValue;
    }
}
template hipError_t launch_pack<int32_t>(int, const int32_t*, int, int16_t*, hipStream_t);
template hipError_t launch_pack<int64_t>(int, const int64_t*, int, int16_t*, hipStream_t);

template <typename S>
hipError_t launch_unpack(int K, const int16_t* trellis, int nt, S* states, hipStream_t stream) {
    if (nt <= 0) return hipSuccess;
    switch (K) {
        case 2: return unpack_k<2>(trellis, nt, states, stream);
        case 3: return unpack_k<3>(trellis, nt, states, stream);
        case 4: return unpack_k<4>(trellis, nt, states, stream);
        case 5: return unpack_k<5>(trellis, nt, states, stream);
        case 6: return unpack_k<6>(trellis, nt, states, stream);
        case 7: return unpack_k<7>(trellis, nt, states, stream);
        default: return hipErrorInvalidValue;
    }
}
template hipError_t launch_unpack<int32_t>(int, const int16_t*, int, int32_t*, hipStream_t);
template hipError_t launch_unpack<int64_t>(int, const int16_t*, int, int64_t*, hipStream_t);

}  // namespace xtq
