// INT16 x INT8 -> INT48 CONV2D on the int8 matrix cores.  An int16 value is 256 h + l + 128 with h its upper byte and l its
// lower byte minus 128, both int8, so a sum of products is
//     sum x w = 256 sum h w + sum l w + 128 sum w
// with each of the first two an int8 matrix product whose int32 accumulator is exact for K <= 65536, and the last one a dot
// product with ones that the weights' way through the registers takes along.  A value of padding is x = 0, whose bytes obey the
// same identity.  Combined in 64 bits in the epilogue, clipped to 48 (tensor_ops.cpp:875-879).
//
// A wave owns 32 pixels x 32 NB channels and takes both operands straight from global memory into the registers the matrix
// instruction reads (lane = pixel or channel lane % 32, 16 channels of half lane / 32 under one tap: 32 bytes of int16 that
// eight v_perm_b32 split into bytes); no LDS, no barrier.  kDepth steps of 32 k are in flight.  Pixels are the rows of the
// result, so that 32 lanes hold neighbouring channels of one pixel and a store instruction writes two runs of 256 bytes.
//
// What bounds it: the lines its loads touch, 32 to an instruction of which 32 bytes each are used before the L1 has let go
// of them: time follows the number of load instructions.  [8,56,56,64]->64 3x3 on one result per lane 1750 us, here 12.2 (10.5 with the
// weights in LDS: conv_i16_taps.hip, which leads on most layers; long reductions over few pixels, whose weights fill the LDS, are this one's).
#include "tmi_mfma.h"

namespace tmi
{

struct ConvI16Args
{
    const int16_t* in;
    const int8_t* w;
    const int64_t* bias;
    int64_t* out;
    int32_t pixels, OC, IC, KW;
    int32_t chunks;    // KH * KW * IC / 16
    int32_t IH, IW, pad_top, pad_left, stride_y, stride_x, dil_y, dil_x;
    int32_t bias_len;
    int32_t n_blocks;    // blocks of 32 NB channels
    FastDiv ow, oh, nb, ic, kw;
};

__device__ __forceinline__ int64_t clip_int48(int64_t v)
{
    const int64_t top = (int64_t(1) << 47) - 1;
    return v > top ? top : (v < -top - 1 ? -top - 1 : v);
}

template <int NB, int DEPTH, int SPLIT>
__global__ __launch_bounds__(256) void conv_i16_kernel(ConvI16Args a)
{
    __shared__ int64_t part[SPLIT > 1 ? 4 : 1][SPLIT > 1 ? 16 * NB : 1][SPLIT > 1 ? 64 : 1];
    const int lane = threadIdx.x & 63, r32 = lane & 31, half = lane >> 5, wave = threadIdx.x >> 6;
    const uint32_t unit = (blockIdx.x * 4 + wave) / SPLIT;    // (pixel tile, channel block), channel blocks of a tile side by side
    const uint32_t pt = fdiv(unit, a.nb), cb = unit - pt * a.nb.d;
    const int p0 = (int)pt * 32, c0 = (int)cb * 32 * NB;
    if (SPLIT == 1 && p0 >= a.pixels)
        return;
    const int all_steps = (a.chunks + 1) >> 1, share = (all_steps + SPLIT - 1) / SPLIT;
    const int first = (wave % SPLIT) * share, steps = all_steps - first < share ? all_steps - first : share;
    const int end   = 2 * (first + share) < a.chunks ? 2 * (first + share) : a.chunks;    // steps past a share add zeros

    // this lane's pixel; one past the last reads the last and is not stored
    const uint32_t pix = (uint32_t)(p0 + r32 < a.pixels ? p0 + r32 : a.pixels - 1);
    const uint32_t t = fdiv(pix, a.ow), n = fdiv(t, a.oh);
    const int y0 = (int)(t - n * a.oh.d) * a.stride_y - a.pad_top, x0 = (int)(pix - t * a.ow.d) * a.stride_x - a.pad_left;
    const int16_t* image = a.in + (int64_t)n * a.IH * a.IW * a.IC;
    const int8_t* wrow[NB];
#pragma unroll
    for (int b = 0; b < NB; b++)
    {
        const int c = c0 + 32 * b + r32;
        wrow[b]     = a.w + (int64_t)(c < a.OC ? c : a.OC - 1) * a.chunks * 16 + 16 * half + 32 * first;
    }

    // position of the lane's next chunk of 16 channels: chunk 2 s + half of step s
    const uint32_t tap0 = fdiv((uint32_t)(32 * first), a.ic), ky0 = fdiv(tap0, a.kw);
    int chunk = 2 * first + half, ic = 32 * first - (int)(tap0 * a.ic.d) + 16 * half, kx = (int)(tap0 - ky0 * a.kw.d);
    int y = y0 + (int)ky0 * a.dil_y, x = x0 + kx * a.dil_x;
    auto wrap = [&]() {
        while (ic >= a.IC)
        {
            ic -= a.IC, x += a.dil_x;
            if (++kx == a.KW)
                kx = 0, x = x0, y += a.dil_y;
        }
    };
    wrap();
    v4i xv[DEPTH][2], wv[DEPTH][NB];
    auto request = [&](int d) {
        const v4i zero = { 0, 0, 0, 0 };
        xv[d][0] = xv[d][1] = zero;
        if (chunk < end && (uint32_t)y < (uint32_t)a.IH && (uint32_t)x < (uint32_t)a.IW)
        {
            const v4i* src = reinterpret_cast<const v4i*>(image + (y * a.IW + x) * a.IC + ic);
            xv[d][0] = src[0], xv[d][1] = src[1];
        }
#pragma unroll
        for (int b = 0; b < NB; b++)
        {
            wv[d][b] = zero;
            if (chunk < end)
                wv[d][b] = *reinterpret_cast<const v4i*>(wrow[b]);
            wrow[b] += 32;
        }
        chunk += 2, ic += 32;
        wrap();
    };

    v16i hi[NB], lo[NB];
    int sum_w[NB];
#pragma unroll
    for (int b = 0; b < NB; b++)
    {
        sum_w[b] = 0;
#pragma unroll
        for (int i = 0; i < 16; i++)
            hi[b][i] = lo[b][i] = 0;
    }
    auto consume = [&](int d) {
        v4i h, l;
#pragma unroll
        for (int i = 0; i < 4; i++)
        {
            const uint32_t u = (uint32_t)xv[d][i >> 1][2 * (i & 1)], v = (uint32_t)xv[d][i >> 1][2 * (i & 1) + 1];
            h[i] = (int)__builtin_amdgcn_perm(v, u, 0x07050301u);
            l[i] = (int)(__builtin_amdgcn_perm(v, u, 0x06040200u) ^ 0x80808080u);
        }
#pragma unroll
        for (int b = 0; b < NB; b++)
        {
            hi[b] = Mma<int8_t>::mma(h, wv[d][b], hi[b]);
            lo[b] = Mma<int8_t>::mma(l, wv[d][b], lo[b]);
            sum_w[b] += dot4_ones(wv[d][b]);
        }
    };

#pragma unroll
    for (int d = 0; d < DEPTH - 1; d++)
        request(d);
    for (int s = 0; s < steps; s += DEPTH)
    {
#pragma unroll
        for (int d = 0; d < DEPTH; d++)
        {
            request((d + DEPTH - 1) % DEPTH);    // of step s + d + DEPTH - 1: nothing but zeros past the last
            consume(d);
        }
    }

    if constexpr (SPLIT > 1)
    {
        // the waves of a tile meet in LDS; each adds up and stores 1 / SPLIT of its results
#pragma unroll
        for (int b = 0; b < NB; b++)
        {
            const int64_t base = 128 * (int64_t)(sum_w[b] + __shfl_xor(sum_w[b], 32));
#pragma unroll
            for (int i = 0; i < 16; i++)
                part[wave][16 * b + i][lane] = base + 256 * (int64_t)hi[b][i] + (int64_t)lo[b][i];
        }
        __syncthreads();
        constexpr int kEach = 16 * NB / SPLIT;
        const int w0        = wave / SPLIT * SPLIT;
        for (int e = 0; e < kEach; e++)
        {
            const int j = (wave % SPLIT) * kEach + e, i = j & 15, c = c0 + 32 * (j >> 4) + r32, p = p0 + 8 * (i >> 2) + 4 * half + (i & 3);
            int64_t v   = 0;
#pragma unroll
            for (int k = 0; k < SPLIT; k++)
                v += part[w0 + k][j][lane];
            if (p < a.pixels && c < a.OC)
                a.out[(int64_t)p * a.OC + c] = clip_int48(a.bias[a.bias_len == 1 ? 0 : c] + v);
        }
        return;
    }
#pragma unroll
    for (int b = 0; b < NB; b++)
    {
        const int c = c0 + 32 * b + r32;
        const int64_t base = c < a.OC ? a.bias[a.bias_len == 1 ? 0 : c] + 128 * (int64_t)(sum_w[b] + __shfl_xor(sum_w[b], 32)) : 0;
#pragma unroll
        for (int i = 0; i < 16; i++)
        {
            const int p = p0 + 8 * (i >> 2) + 4 * half + (i & 3);
            if (p < a.pixels && c < a.OC)
                a.out[(int64_t)p * a.OC + c] = clip_int48(base + 256 * (int64_t)hi[b][i] + (int64_t)lo[b][i]);
        }
    }
}

// Copies of both operands with the channel vectors padded to ICP (a multiple of 16) channels of zeros, in one launch.
__global__ __launch_bounds__(256) void pad_channels_i16_kernel(const int16_t* __restrict__ in, int64_t in_rows, const int8_t* __restrict__ w,
                                                               int64_t w_rows, int32_t IC, FastDiv icp, int16_t* __restrict__ in_out,
                                                               int8_t* __restrict__ w_out, int32_t blocks)
{
    const int64_t n_in = in_rows * icp.d, total = n_in + w_rows * icp.d;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)blocks * 256)
    {
        const bool is_w   = i >= n_in;
        const int64_t j   = is_w ? i - n_in : i;
        const int64_t row = j / icp.d;
        const int c       = (int)(j - row * icp.d);
        if (is_w)
            w_out[j] = c < IC ? w[row * IC + c] : (int8_t)0;
        else
            in_out[j] = c < IC ? in[row * IC + c] : (int16_t)0;
    }
}

// 0: the layer is not this form's; 1: read in place; else the bytes of scratch its padded operands take
size_t conv_i16_mfma_scratch_bytes(const ConvGeom& g, int32_t w_zp)
{
    const int64_t pixels = (int64_t)g.N * g.OH * g.OW, icp = (g.IC + 15) / 16 * 16, K = (int64_t)g.KH * g.KW * icp;
    if (w_zp != 0 || g.IC < 1 || K > 65536 || !fastdiv_exact_up_to((uint64_t)K, (uint32_t)icp) || pixels > INT32_MAX - 64 || (int64_t)g.IH * g.IW * icp > INT32_MAX / 2 ||
        !fastdiv_exact_up_to((uint64_t)pixels, (uint32_t)g.OW) || !fastdiv_exact_up_to((uint64_t)pixels / g.OW, (uint32_t)g.OH))
        return 0;
    const int64_t units = ((pixels + 31) / 32) * ((g.OC + 31) / 32);
    if (!fastdiv_exact_up_to((uint64_t)units + 4, (uint32_t)((g.OC + 31) / 32)) || (int64_t)g.OC * K > INT32_MAX)
        return 0;
    if (icp == g.IC)
        return 1;
    return (size_t)(((int64_t)g.N * g.IH * g.IW * icp * 2 + 255) / 256 * 256 + (int64_t)g.OC * K);
}

const char* launch_conv_i16_mfma(hipStream_t st, const ConvGeom& g, const void* in, const void* w, const void* bias, void* out, void* scratch)
{
    ConvI16Args a{};
    const int32_t icp = (g.IC + 15) / 16 * 16;
    if (icp != g.IC)
    {
        const int64_t in_rows = (int64_t)g.N * g.IH * g.IW, w_rows = (int64_t)g.OC * g.KH * g.KW, total = (in_rows + w_rows) * icp;
        int16_t* in_pad = reinterpret_cast<int16_t*>(scratch);
        int8_t* w_pad   = reinterpret_cast<int8_t*>(scratch) + (in_rows * icp * 2 + 255) / 256 * 256;
        const int64_t blocks = (total + 255) / 256;
        const unsigned grid = (unsigned)(blocks > 8192 ? 8192 : blocks);
        hipLaunchKernelGGL(pad_channels_i16_kernel, dim3(grid), dim3(256), 0, st, (const int16_t*)in, in_rows, (const int8_t*)w, w_rows, g.IC,
                           make_fastdiv((uint32_t)icp), in_pad, w_pad, (int32_t)grid);
        in = in_pad, w = w_pad;
    }
    else if ((((uintptr_t)in | (uintptr_t)w) & 15) != 0)
        return nullptr;
    a.in = (const int16_t*)in, a.w = (const int8_t*)w, a.bias = (const int64_t*)bias, a.out = (int64_t*)out;
    a.pixels = (int32_t)((int64_t)g.N * g.OH * g.OW), a.OC = g.OC, a.IC = icp, a.KW = g.KW, a.chunks = g.KH * g.KW * icp / 16;
    a.IH = g.IH, a.IW = g.IW, a.pad_top = g.pad_top, a.pad_left = g.pad_left;
    a.stride_y = g.stride_y, a.stride_x = g.stride_x, a.dil_y = g.dil_y, a.dil_x = g.dil_x, a.bias_len = g.bias_len;
    a.ic = make_fastdiv((uint32_t)icp), a.kw = make_fastdiv((uint32_t)g.KW);
    a.ow = make_fastdiv((uint32_t)g.OW), a.oh = make_fastdiv((uint32_t)g.OH);
    const int64_t tiles = (a.pixels + 31) / 32;
    // 64 channels to a wave from 512 such units on: a pixel's bytes then serve twice as many products ([8,56,56,64]->64 3x3, 784
    // units: 12.6 us against 16.2 with 32).  Fewer units: 32 channels, and K split over the waves of a workgroup until there
    // are about two waves per SIMD (us split 1 / 2 / 4: [2,14,14,256]->256 3x3 26.5 / 15.9 / 10.2, [1,7,7,512]->512 45.5 / 25.3 /
    // 14.5, [4,28,28,41]->64 9.9 / 8.5 / 6.8, [1,8,8,16]->8 5.7 / 5.2 / 4.5; with many units the split only costs:
    // [16,56,56,64]->64 1x1 9.6 / 13.8 / 16.9).
    const bool two  = g.OC > 32 && tiles * ((g.OC + 63) / 64) >= 512;
    const int nb    = two ? (g.OC + 63) / 64 : (g.OC + 31) / 32;
    const int64_t units = tiles * nb;
    const int steps = (a.chunks + 1) / 2;
    const int split = two ? 1 : (units <= 512 && steps >= 4 ? 4 : (units <= 1024 && steps >= 2 ? 2 : 1));
    a.nb            = make_fastdiv((uint32_t)nb);
    const dim3 grid((unsigned)((units * split + 3) / 4));
    if (two)
        hipLaunchKernelGGL((conv_i16_kernel<2, 3, 1>), grid, dim3(256), 0, st, a);
    else if (split == 4)
        hipLaunchKernelGGL((conv_i16_kernel<1, 4, 4>), grid, dim3(256), 0, st, a);
    else if (split == 2)
        hipLaunchKernelGGL((conv_i16_kernel<1, 4, 2>), grid, dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL((conv_i16_kernel<1, 4, 1>), grid, dim3(256), 0, st, a);
    return "conv2d_mfma_i16_i48";
}

}    // namespace tmi
