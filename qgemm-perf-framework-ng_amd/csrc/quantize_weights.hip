// Weight quantizers for gfx950: q4_0 and q4_K, byte-identical to the
// reference's host quantizers llama_reference::quantize_row_q4_0 and
// quantize_row_q4_K (bench/llama_reference/llama_reference.cpp:13-36, 72-111),
// including q4_K's non-upstream scale packing. They are setup kernels: fast
// generation of large weight matrices on the device; the benchmarked paths
// take weights in the reference's byte layout whichever side produced them.
//
// Bit-exactness relies on the same rules as the activation quantizers
// (separately rounded fp32 steps, correctly rounded division, roundf = half
// away from zero, the ggml fp32 -> fp16 routine) plus:
//   * q4_0's scale comes from the first element of largest magnitude (the
//     reference's strict "<" scan, in one lane);
//   * float -> int conversions of values outside the int32 range return
//     INT_MIN, as the reference's x86-64 build does (cvttss2si); they can only
//     occur for degenerate sub-blocks (range far below the offset).
#include <climits>

#include "device_common.h"
#include "kernels.h"

namespace pfng {

namespace {

__device__ __forceinline__ int cvt_i32_x86(float v) {
    return (v >= -2147483648.0f && v < 2147483648.0f) ? (int)v : INT_MIN;
}

// Both kernels give every lane 32 consecutive values (a q4_0 block, a q4_K
// sub-block), so that a block's maxima, divisions and scales are computed once
// instead of by eight lanes each, and no value crosses lanes before it is
// quantized. A wave's 64 x 128 bytes are contiguous in memory; they come in by
// direct-to-LDS loads, whole lines at a time, and each lane reads its 128 bytes
// back. Chunk c of row r lies at slot c ^ (r % 8) of its LDS row (the loads
// permute the chunks within each line), which keeps the 16-byte reads free of
// bank conflicts. With eight lanes per block both kernels were VALU-bound on
// the repeated block arithmetic; 11008 x 4096 (206 MB at 5.8 TB/s now, a
// streaming pass): q4_0 44.7 -> 35.6 us, q4_K 83.0 -> 35.6; 1000 x 1024 2.73 ->
// 2.76 and 4.35 -> 3.19 us; 64 x 256, a handful of waves, 2.30 -> 2.51 and 2.76
// -> 2.90. Workgroups of one wave: with four, 36.3 us and 2.90 / 3.20 at 1000 x
// 1024.
constexpr int kWaveLds = 64 * 128;

// Issues the wave's copies and reads lane l's 32 values (row `first` + l of
// `rows` rows of 32 floats; rows past the end repeat the last).
__device__ __forceinline__ void load_rows32(const float *__restrict__ x, int64_t first, int64_t rows,
                                            uint8_t *lds, int lane, float (&v)[32]) {
    const uint8_t *src = reinterpret_cast<const uint8_t *>(x);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int r = 8 * i + (lane >> 3), c = (lane & 7) ^ (r & 7);
        const int64_t row = first + r < rows ? first + r : rows - 1;
        __builtin_amdgcn_global_load_lds(src + row * 128 + c * 16,
                                         (__attribute__((address_space(3))) void *)(lds + 1024 * i), 16, 0, 0);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const float4 q = *reinterpret_cast<const float4 *>(lds + lane * 128 + ((c ^ (lane & 7)) * 16));
        v[4 * c] = q.x;
        v[4 * c + 1] = q.y;
        v[4 * c + 2] = q.z;
        v[4 * c + 3] = q.w;
    }
}

// Minimum and maximum of 32 values (NaNs ignored, as fminf / fmaxf do) in
// trees of four levels.
__device__ __forceinline__ void min_max32(const float (&v)[32], float &lo, float &hi) {
    float l[11], h[11];
#pragma unroll
    for (int i = 0; i < 10; ++i) {
        l[i] = fminf(fminf(v[3 * i], v[3 * i + 1]), v[3 * i + 2]);
        h[i] = fmaxf(fmaxf(v[3 * i], v[3 * i + 1]), v[3 * i + 2]);
    }
    l[10] = fminf(v[30], v[31]);
    h[10] = fmaxf(v[30], v[31]);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        l[i] = fminf(fminf(l[i], l[i + 3]), l[i + 6]);
        h[i] = fmaxf(fmaxf(h[i], h[i + 3]), h[i + 6]);
    }
    lo = fminf(fminf(fminf(l[0], l[1]), l[2]), fminf(l[9], l[10]));
    hi = fmaxf(fmaxf(fmaxf(h[0], h[1]), h[2]), fmaxf(h[9], h[10]));
}

// kAligned4: the output is 4-byte aligned and leaves as dwords.
template <bool kAligned4>
__global__ __launch_bounds__(64) void quantize_q4_0_kernel(const float *__restrict__ x,
                                                                    uint8_t *__restrict__ y, int64_t nblocks) {
    __shared__ __align__(16) uint8_t buf[kWaveLds];
    const int lane = threadIdx.x;
    const int64_t first = (int64_t)blockIdx.x * 64;
    float v[32];
    load_rows32(x, first, nblocks, buf, lane, v);
    // first element of largest magnitude (the reference's strict "<" scan from
    // 0): the maximum or the minimum, by a scan only where they tie or are NaN
    // (a block of NaNs, which the reference's scan passes over)
    float lo, hi;
    min_max32(v, lo, hi);
    float smax = hi > -lo ? hi : lo;
    if (__any(!(hi > -lo || hi < -lo))) {
        float amax = 0.0f, first_max = 0.0f;
#pragma unroll
        for (int i = 0; i < 32; ++i) {
            const float av = fabsf(v[i]);
            first_max = amax < av ? v[i] : first_max;
            amax = amax < av ? av : amax;
        }
        smax = first_max;
    }
    const float d = smax / -8.0f;
    const float id = d != 0.0f ? 1.0f / d : 0.0f;
    uint32_t qs[4] = {0, 0, 0, 0};  // byte i = q_i | q_(i+16) << 4
#pragma unroll
    for (int i = 0; i < 32; ++i) {
        const int t = (int)(int8_t)(int)add_rn(mul_rn(v[i], id), 8.5f);
        const uint32_t q = (uint32_t)(t < 15 ? t : 15) & 15u;
        qs[(i % 16) / 4] |= q << (8 * (i % 4) + (i < 16 ? 0 : 4));
    }
    // the blocks assembled in the same LDS bytes (their reads are done)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    uint16_t *blk = reinterpret_cast<uint16_t *>(buf) + lane * 9;
    blk[0] = (uint16_t)f32_to_fp16_bits(d);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        blk[1 + 2 * i] = (uint16_t)(qs[i] & 0xffffu);
        blk[2 + 2 * i] = (uint16_t)(qs[i] >> 16);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const int valid = nblocks - first < 64 ? (int)(nblocks - first) : 64;
    uint8_t *out = y + first * 18;
    if constexpr (kAligned4) {  // 64 blocks are 288 dwords; first * 18 is a multiple of 4
        const uint32_t *src = reinterpret_cast<const uint32_t *>(buf);
        uint32_t *dst = reinterpret_cast<uint32_t *>(out);
        const int words = valid * 18 >> 2;
        for (int i = lane; i < words; i += 64) dst[i] = src[i];
        if ((valid & 1) && lane == 0)
            reinterpret_cast<uint16_t *>(out)[valid * 9 - 1] = reinterpret_cast<const uint16_t *>(buf)[valid * 9 - 1];
    } else {
        const uint16_t *src = reinterpret_cast<const uint16_t *>(buf);
        uint16_t *dst = reinterpret_cast<uint16_t *>(out);
        for (int i = lane; i < valid * 9; i += 64) dst[i] = src[i];
    }
}

// x / b correctly rounded, given y = 1 / b correctly rounded: two of
// Markstein's correction steps (the first makes the quotient faithful, the
// second rounds it correctly), 5 operations instead of the 11 of a general
// division. Needs b in [2^-40, 2^40]; a quotient below 2^-40 may be off in its
// last place, which the sum it goes into absorbs.
__device__ __forceinline__ float div_by(float x, float b, float y) {
    float q = x * y;
    q = __builtin_fmaf(__builtin_fmaf(-q, b, x), y, q);
    return __builtin_fmaf(__builtin_fmaf(-q, b, x), y, q);
}

// Lane l quantizes sub-block l % 8 of super-block l / 8 of the wave's eight.
__global__ __launch_bounds__(64) void quantize_q4_K_kernel(const float *__restrict__ x,
                                                                    uint8_t *__restrict__ y, int64_t nblocks) {
    __shared__ __align__(16) uint8_t buf[kWaveLds];
    const int lane = threadIdx.x;
    const int64_t first = (int64_t)blockIdx.x * 8;
    float v[32];
    load_rows32(x, first * 8, nblocks * 8, buf, lane, v);
    float lo, hi;
    min_max32(v, lo, hi);
    const float ls = sub_rn(hi, lo) / 15.0f;
    const float div = ls != 0.0f ? ls : 1.0f;
    const float lm = -lo / div;
    // super-block maxima start from 0, as in the reference
    const float maxs = fmaxf(group_max<8>(ls), 0.0f), maxm = fmaxf(group_max<8>(lm), 0.0f);
    const float ds = maxs / 63.0f, dm = maxm / 63.0f;
    const int si = cvt_i32_x86(roundf(ls / (ds != 0.0f ? ds : 1.0f)));
    const int mi = cvt_i32_x86(roundf(lm / (dm != 0.0f ? dm : 1.0f)));
    const uint32_t s8 = (uint32_t)(si < 63 ? si : 63) & 0xffu;  // uint8_t s[i] = std::min(63, ...)
    const uint32_t m8 = (uint32_t)(mi < 63 ? mi : 63) & 0xffu;
    // values: clamp(round(x / ls + lm), 0, 15)
    uint32_t q[8];
    if (__all(div >= 0x1p-40f && div <= 0x1p+40f)) {
        // trunc(t + (0.5 - 2^-25)) equals roundf(t) on [0, 130] and lies
        // outside [0.5, 15.5) on the same side as t elsewhere (t < 2^31 here)
        const float inv = 1.0f / div;
#pragma unroll
        for (int i = 0; i < 32; ++i) {
            const float t = add_rn(div_by(v[i], div, inv), lm);
            const uint32_t u = (uint32_t)__builtin_amdgcn_fmed3f(add_rn(t, 0x1.fffffep-2f), 0.0f, 15.5f);
            q[i / 4] = i % 4 ? q[i / 4] | u << (8 * (i % 4)) : u;
        }
    } else {
#pragma unroll
        for (int i = 0; i < 32; ++i) {
            int t = cvt_i32_x86(roundf(add_rn(v[i] / div, lm)));
            t = t < 0 ? 0 : (t > 15 ? 15 : t);
            q[i / 4] = i % 4 ? q[i / 4] | (uint32_t)t << (8 * (i % 4)) : (uint32_t)t;
        }
    }
    // qs[32 p + j] = q(2p, j) | q(2p+1, j) << 4: the even lane of a pair takes
    // j < 16, the odd lane the rest
    const int sb = lane & 7;
    const bool odd = sb & 1;
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t got = (uint32_t)xor_shfl<1>((int)(odd ? q[i] : q[4 + i]));
        const uint32_t own = odd ? q[4 + i] : q[i];
        o[i] = odd ? got | own << 4 : own | got << 4;
    }
    // header: d, dmin, 12 bytes of scales / mins with the reference's packing,
    // each lane's bits OR-ed over the super-block's eight lanes
    const int sh = 8 * (sb & 3);
    const bool up = sb >= 4;
    uint32_t w[3] = {up ? (s8 & 3u) << (6 + sh) : s8 << sh, up ? (m8 & 3u) << (6 + sh) : m8 << sh,
                     up ? (((s8 >> 2) | ((m8 >> 2) << 4)) & 0xffu) << sh : 0u};
#pragma unroll
    for (int i = 0; i < 3; ++i)
        w[i] = (uint32_t)butterfly<4>((int)w[i], [](int a, int b) { return a | b; });
    const int64_t block = first + (lane >> 3);
    if (block < nblocks) {
        uint8_t *blk = y + block * 144;
        *reinterpret_cast<uint4 *>(blk + 16 + 16 * sb) = make_uint4(o[0], o[1], o[2], o[3]);
        if (sb == 0)
            *reinterpret_cast<uint4 *>(blk) =
                make_uint4(f32_to_fp16_bits(ds) | (f32_to_fp16_bits(dm) << 16), w[0], w[1], w[2]);
    }
}

}  // namespace

hipError_t launch_quantize_q4_0(const float *x, void *y, int64_t rows, int64_t k, hipStream_t stream) {
    const int64_t nblocks = rows * (k / 32);
    if (nblocks == 0) return hipSuccess;
    const dim3 grid((unsigned)((nblocks + 63) / 64)), block(64);
    if ((reinterpret_cast<uintptr_t>(y) & 3) == 0)
        hipLaunchKernelGGL(quantize_q4_0_kernel<true>, grid, block, 0, stream, x, static_cast<uint8_t *>(y), nblocks);
    else
        hipLaunchKernelGGL(quantize_q4_0_kernel<false>, grid, block, 0, stream, x, static_cast<uint8_t *>(y), nblocks);
    return hipGetLastError();
}

hipError_t launch_quantize_q4_K(const float *x, void *y, int64_t rows, int64_t k, hipStream_t stream) {
    const int64_t nblocks = rows * (k / 256);
    if (nblocks == 0) return hipSuccess;
    hipLaunchKernelGGL(quantize_q4_K_kernel, dim3((unsigned)((nblocks + 7) / 8)), dim3(64), 0, stream, x,
                       static_cast<uint8_t *>(y), nblocks);
    return hipGetLastError();
}

}  // namespace pfng
