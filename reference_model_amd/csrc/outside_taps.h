// CONV2D results whose window leaves the image, on kernels that multiply what lies outside as zeros.
//
// A tap outside the image adds nothing in the reference (tensor_ops.cpp:845-852); zero times the weight is nothing too, unless the weight is infinite or
// NaN.  A workgroup (the patch kernel, the slab kernel and those with resident weights: a wave) that met a sum that is NaN looks at its channels' weights behind its stores, once and with all
// lanes side by side; where one is no number, its waves go over their tiles once more and sum one at a time, without those taps, the results that are NaN,
// whose window leaves the image and whose channel has such a weight.  Every other result keeps the sum it has, and a NaN that came from the image costs
// the look.  us a call on a NaN image, every NaN summed again / so (on finite values): streaming patch fp16 3x3 [7,14,21,200]->288 2600 / 23 (17), bf16
// [16,28,28,256]->64 3679 / 24 (16); GEMM kernel [4,28,28,224]->256 31 (18), bf16 [64,7,7,512]->512 90 (44); patch kernel [2,28,28,256]->250 53 (25); slab
// kernel [8,56,56,64]->64 13.8 (5.9); resident weights fp16 [15,54,65,68]->64 1860 / 32 (24), bf16 [2,79,7,88]->23 276 / 9.4 (5.5); K split bf16 5x5 [2,14,13,200]->40
// 1701 / 35 (15), fp16 stride 2 [9,31,41,240]->32 764 / 16 (8.7).  (A __threadfence() of every wave that met a NaN, before it knew of such a weight: 113 in the place of the 32.)
// (Behind the loop and from arguments read anew it costs the loop a test of the results and no vector register: summed again in the loop, two channel
// tiles a wave of conv_taps.hip fall from four waves a SIMD to two.  On finite values, over 15 layers of the GEMM kernel 1.002 of the time
// without any of this, over 77 of the patch kernel 0.994, where arguments kept by way of LDS spare the loop's scalars; with its scalars kept across the stores bf16
// [4,71,71,280]->136 58.2 / 63.4, so 56.3.  A workgroup's barrier in the patch kernel: layers of short rounds 2 to 4 % more.)
#pragma once
#include <type_traits>

#include "tmi_mfma.h"

namespace tmi
{

struct OutsideTaps
{
    const uint8_t *in, *w;
    const void* bias;
    void* out;
    int32_t row_bytes;    // of a pixel's channel vector
    int32_t IH, IW, OC, OH, OW, KH, KW;
    int32_t sy, sx, dy, dx, pad_top, pad_left;
    int32_t bias_len;
};

// The largest of so_far and N sums, or NaN if one of them is: an instruction for two of them, and one test behind the last
template <int N, typename R>
__device__ __forceinline__ float largest_or_nan(float so_far, const R& v)
{
#pragma unroll
    for (int e = 0; e < N; e += 2)
        so_far = __builtin_elementwise_maximum(__builtin_elementwise_maximum(v[e], v[e + 1]), so_far);
    return so_far;
}

// The lane's number, counted and not kept from the kernel's start
__device__ __forceinline__ int lane_counted()
{
    return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
}

// The kernel's arguments from memory: not the values it began with, which would have to be kept
template <typename Args>
__device__ __forceinline__ Args args_read_anew()
{
    auto* args = __builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(args));
    Args a;
    __builtin_memcpy(&a, (const void*)args, sizeof(a));
    return a;
}

// The same, and the workgroup's number, by way of 16 bytes of LDS (written before the first barrier) where scalar registers are short up to the end
__device__ __forceinline__ void keep_place(v4i* place)
{
    if (threadIdx.x == 0)
    {
        const uint64_t args = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
        *place              = v4i{ (int)(uint32_t)args, (int)(uint32_t)(args >> 32), (int)blockIdx.x, 0 };
    }
}
template <typename Args>
__device__ __forceinline__ Args args_kept(const v4i* place, uint32_t& block)
{
    const v4i p      = *place;
    const uint32_t l = (uint32_t)__builtin_amdgcn_readfirstlane(p[0]), h = (uint32_t)__builtin_amdgcn_readfirstlane(p[1]);
    block            = (uint32_t)__builtin_amdgcn_readfirstlane(p[2]);
    static_assert(sizeof(Args) % 4 == 0, "by words");
    const auto* from = (const __attribute__((address_space(4))) uint32_t*)((uint64_t)h << 32 | l);
    uint32_t words[sizeof(Args) / 4];
#pragma unroll
    for (int i = 0; i < (int)sizeof(Args) / 4; i++)
        words[i] = from[i];
    Args a;
    __builtin_memcpy(&a, words, sizeof(a));
    return a;
}

// Whether a word, 16 bytes of weights hold one that is infinite or NaN
template <typename T>
__device__ __forceinline__ bool not_finite(uint32_t word)
{
    constexpr uint32_t EXPONENT = sizeof(T) == 4 ? 0x7f800000u : (std::is_same_v<T, bf16_t> ? 0x7f80u : 0x7c00u);
    return (word & EXPONENT) == EXPONENT || (sizeof(T) < 4 && (word >> 16 & EXPONENT) == EXPONENT);
}
template <typename T>
__device__ __forceinline__ bool not_finite(const v4i& v)
{
    return not_finite<T>((uint32_t)v[0]) || not_finite<T>((uint32_t)v[1]) || not_finite<T>((uint32_t)v[2]) || not_finite<T>((uint32_t)v[3]);
}

// Whether the lane's part of the weights from w on, every parts-th 16 bytes from the part-th on, holds one that is infinite or NaN
template <typename T>
__device__ __forceinline__ bool weights_not_finite(const uint8_t* w, int64_t bytes, int part, int parts)
{
    bool found          = false;
    const int64_t whole = bytes & ~(int64_t)15;
#pragma unroll 8
    for (int64_t at = 16 * part; at < whole; at += 16 * parts)
        found |= not_finite<T>(load16(w + at));
    for (int64_t at = whole + part * (int)sizeof(T); at < bytes; at += parts * (int)sizeof(T))
        found |= not_finite<T>(sizeof(T) == 4 ? *reinterpret_cast<const uint32_t*>(w + at) : (uint32_t)*reinterpret_cast<const uint16_t*>(w + at));
    return found;
}

// Whether a wave of the workgroup met a NaN (largest_or_nan() of its sums) and the weights of the workgroup's channels are not all finite.  For all waves alike, behind their loops;
// words: 2 WAVES words of LDS that no wave uses any more; weights(look): calls look(w, bytes), from arguments read anew where registers are short.
template <typename T, int WAVES, typename Weights>
__device__ __forceinline__ bool met_odd_weights(float largest, int wave, int32_t* words, Weights&& weights)
{
    const int lane   = lane_counted();
    auto in_any_wave = [&](bool flag, int32_t* word) {
        if (lane == 0)
            word[wave] = flag;
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");    // (stores need not have arrived)
        return __any(lane < WAVES && word[lane < WAVES ? lane : 0]) != 0;
    };
    if (__builtin_expect(!in_any_wave(__any(largest != largest), words), 1))
        return false;
    bool odd = false;
    weights([&](const uint8_t* w, int64_t bytes) { odd = weights_not_finite<T>(w, bytes, wave * 64 + lane, WAVES * 64); });
    return in_any_wave(__any(odd), words + WAVES);
}

// The lane's pixel (n, oy, ox), if it is there; of `tiles` tiles of 32 channels the lane holds `each` from channel c0 on, the same for all lanes of a
// half wave.  For whole waves, whose results in g.out are stored and seen by all lanes.
template <typename T>
__device__ __forceinline__ void without_outside_taps(const OutsideTaps& g, bool there, int n, int oy, int ox, int c0, int tiles, int each)
{
    const int lane = lane_counted();
    const int y0 = oy * g.sy - g.pad_top, x0 = ox * g.sx - g.pad_left;
    const bool leaves = there && (y0 < 0 || x0 < 0 || y0 + (g.KH - 1) * g.dy >= g.IH || x0 + (g.KW - 1) * g.dx >= g.IW);
    if (!__any(leaves))
        return;
    T* out               = reinterpret_cast<T*>(g.out) + (leaves ? (((size_t)n * g.OH + oy) * g.OW + ox) * g.OC : 0);
    const uint8_t* image = g.in + (leaves ? (size_t)n * g.IH * g.IW * g.row_bytes : 0);
    const int w_bytes    = g.KH * g.KW * g.row_bytes;
#pragma unroll 1
    for (int k = 0; k < tiles * each; k++)
    {
        const int c = c0 + k / each * 32 + k % each;
        const bool nan = leaves && c < g.OC && load_as_float<T>(out, c) != load_as_float<T>(out, c);
        if (!__any(nan))
            continue;
        const uint8_t* w   = g.w + (size_t)(c < g.OC ? c : 0) * w_bytes;
        const uint64_t odd = __ballot(weights_not_finite<T>(w, w_bytes, lane & 31, 32));
        if (!nan || (lane < 32 ? (uint32_t)odd : (uint32_t)(odd >> 32)) == 0)
            continue;
        float sum = 0.0f;
#pragma unroll 1
        for (int ky = 0; ky < g.KH; ky++)
#pragma unroll 1
            for (int kx = 0; kx < g.KW; kx++, w += g.row_bytes)
            {
                const int y = y0 + ky * g.dy, x = x0 + kx * g.dx;
                if ((uint32_t)y >= (uint32_t)g.IH || (uint32_t)x >= (uint32_t)g.IW)
                    continue;
                const uint8_t* u = image + ((size_t)y * g.IW + x) * g.row_bytes;
#pragma unroll 1
                for (int i = 0; i < g.row_bytes / (int)sizeof(T); i++)
                    sum += load_as_float<T>(u, i) * load_as_float<T>(w, i);
            }
        store_from_float(out + c, sum + load_as_float<T>(g.bias, g.bias_len == 1 ? 0 : c));
    }
}

}    // namespace tmi
