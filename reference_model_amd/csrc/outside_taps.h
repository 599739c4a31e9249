// CONV2D results whose window leaves the image, on kernels that multiply what lies outside as zeros.
//
// A tap outside the image adds nothing in the reference (tensor_ops.cpp:845-852); zero times the weight is nothing too, unless the weight is infinite or
// NaN.  A workgroup that met a sum that is NaN looks at its channels' weights behind its stores, once and with all lanes side by side; where one is no
// number, its waves go over their tiles once more and sum one at a time, without those taps, the results that are NaN, whose window leaves the image and
// whose channel has such a weight.  Every other result keeps the sum it has, and a NaN that came from the image costs the look.  us a call on a NaN
// image, every NaN summed again / so (on finite values): streaming patch fp16 3x3 [7,14,21,200]->288 2600 / 24 (17), bf16 [16,28,28,256]->64 3679 / 24 (16).
// (Behind the loop and from arguments read anew it costs the loop a test of the results and no register: summed again in the loop, two channel tiles
// a wave of conv_taps.hip fall from four waves a SIMD to two.)
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

// Whether one of N sums of any lane is NaN
template <int N, typename R>
__device__ __forceinline__ bool any_nan(const R& v)
{
    bool nan = false;
#pragma unroll
    for (int e = 0; e < N; e += 2)
        nan |= __builtin_isunordered(v[e], v[e + 1]);
    return __any(nan);
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

// Whether the lane's part of the weights from w on, every parts-th 16 bytes from the part-th on, holds one that is infinite or NaN
template <typename T>
__device__ __forceinline__ bool weights_not_finite(const uint8_t* w, int64_t bytes, int part, int parts)
{
    constexpr uint32_t EXPONENT = sizeof(T) == 4 ? 0x7f800000u : (std::is_same_v<T, bf16_t> ? 0x7f80u : 0x7c00u);
    auto odd = [](uint32_t word) { return (word & EXPONENT) == EXPONENT || (sizeof(T) < 4 && (word >> 16 & EXPONENT) == EXPONENT); };
    bool found          = false;
    const int64_t whole = bytes & ~(int64_t)15;
#pragma unroll 4
    for (int64_t at = 16 * part; at < whole; at += 16 * parts)
    {
        const v4i v = load16(w + at);
        found |= odd(v[0]) || odd(v[1]) || odd(v[2]) || odd(v[3]);
    }
    for (int64_t at = whole + part * (int)sizeof(T); at < bytes; at += parts * (int)sizeof(T))
        found |= odd(sizeof(T) == 4 ? *reinterpret_cast<const uint32_t*>(w + at) : *reinterpret_cast<const uint16_t*>(w + at));
    return found;
}

// Whether a wave of the workgroup met a NaN and the weights of the workgroup's channels are not all finite.  For all waves alike, behind their loops;
// words: 2 WAVES words of LDS that no wave uses any more.
template <typename T, int WAVES>
__device__ __forceinline__ bool met_odd_weights(bool met_nan, int32_t* words, const uint8_t* w, int64_t bytes)
{
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    auto in_any_wave = [&](bool flag, int32_t* word) {
        if (lane == 0)
            word[wave] = flag;
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");    // (stores need not have arrived)
        return __any(lane < WAVES && word[lane < WAVES ? lane : 0]) != 0;
    };
    return in_any_wave(met_nan, words) && in_any_wave(__any(weights_not_finite<T>(w, bytes, threadIdx.x, WAVES * 64)), words + WAVES);
}

// The lane's pixel (n, oy, ox), if it is there; of `tiles` tiles of 32 channels the lane holds `each` from channel c0 on, the same for all lanes of a
// half wave.  For whole waves, whose results in g.out are stored and seen by all lanes.
template <typename T>
__device__ __forceinline__ void without_outside_taps(const OutsideTaps& g, bool there, int n, int oy, int ox, int c0, int tiles, int each)
{
    const int lane = threadIdx.x & 63;
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
