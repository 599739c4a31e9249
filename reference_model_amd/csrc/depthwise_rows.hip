// DEPTHWISE_CONV2D int8 with 3x3 or 5x5 taps, stride 1 or 2, no dilation, of any channel count (multiplier 1, weight_zp 0).
//
// A lane owns four consecutive channels of one output column and walks down a strip of output rows.  Of every input row it loads the K
// dwords under its taps once and turns them into K-dimensional operands once: four taps of a row become channel-major by eight byte
// permutes, and a dot product of four bytes per channel takes them in; the fifth tap stays as it was loaded and meets a weight that is
// zero in the other three bytes.  The operands of the last K input rows stay in registers, so that a row costs its loads and permutes
// once and not K times (K / stride).  Consecutive lanes are consecutive channel groups, then columns: a load of a wave is a run of
// NHWC memory.  Channels that are no multiple of four: the last group's dwords run into the next pixel, whose bytes count for nothing, and its
// result is stored byte by byte.  A tap outside the image reads as the input zero point (see depthwise.hip for the identity).
//
// What bounds it: the vector ALU, some 26 instructions a result at 3x3 of which twelve are the RESCALE; a third of that with one pixel a
// lane at 5x5 (depthwise.hip).  us depthwise.hip, or one result per lane where the channels are no whole groups / here, fused RESCALE: 5x5
// [36,132,137,40] 164 / 45, [21,37,34,576] 171 / 26, [1,8,13,16] 7.0 / 3.4, [14,139,139,29] 132 / 23, stride 2 [6,94,94,554] 205 / 29; 3x3
// [10,131,128,40] 16.5 / 11.4, [34,13,18,445] 33 / 11, [5,129,134,33] 28 / 8.4, [5,22,22,65] 4.9 / 3.6.  The matrix-core kernels keep their layers (channels in
// sixteens, 3x3): [11,55,60,160] 7.9 / 11.6, [64,112,112,96] stride 2 25.5 / 28.4; [54,53,58,48] 11.7 / 13.0.
#include <type_traits>

#include "tmi_kernels.h"

namespace tmi
{

struct DwRowsArgs
{
    const int8_t* in;
    const int8_t* w;
    const int32_t* bias;
    void* out;
    uint32_t* flag_word;
    RescaleParams rp;
    int32_t C, IH, IW, OH, OW, pad_top, pad_left, bias_len;
    int32_t groups;       // of four channels
    int32_t rows;         // output rows of a strip
    int32_t lanes;        // N * strips * OW * groups
    int32_t in_last, w_last;    // offsets of the last four bytes
    int32_t za, out_dtype;
    uint32_t per_xcd;     // workgroups / 8
    FastDiv div_groups, div_ow, div_strips;
};

__device__ __forceinline__ int load4(const int8_t* p)    // of no alignment
{
    int v;
    __builtin_memcpy(&v, p, 4);
    return v;
}

template <int K, int S, bool RAGGED, bool RESCALE>
__global__ __launch_bounds__(256) void depthwise_rows_kernel(DwRowsArgs a)
{
    constexpr int Q = K == 3 ? 4 : 5;    // operands of a row: a quad per channel, and the fifth tap
    uint32_t bid = blockIdx.x;
    if (bid < 8 * a.per_xcd)
        bid = (bid & 7) * a.per_xcd + (bid >> 3);    // a run of strips for each L2
    const uint32_t id = bid * 256u + threadIdx.x;
    if (id >= (uint32_t)a.lanes)
        return;
    const uint32_t col = fdiv(id, a.div_groups);
    const int c0       = (int)(id - col * a.div_groups.d) * 4;
    const uint32_t sr  = fdiv(col, a.div_ow);
    const int ox       = (int)(col - sr * a.div_ow.d);
    const int n        = (int)fdiv(sr, a.div_strips), oy0 = (int)(sr - (uint32_t)n * a.div_strips.d) * a.rows;
    const int oy_end   = oy0 + a.rows < a.OH ? oy0 + a.rows : a.OH;
    const int live     = a.C - c0 < 4 ? a.C - c0 : 4;    // channels of the group
    const int za_word  = (a.za & 0xff) * 0x01010101;

    const int x0   = ox * S - a.pad_left;
    int iy         = oy0 * S - a.pad_top;                          // next input row to load
    int off        = ((n * a.IH + iy) * a.IW + x0) * a.C + c0;     // of its first tap
    const int step = a.IW * a.C;
    bool xv[K];
#pragma unroll
    for (int k = 0; k < K; k++)
        xv[k] = (unsigned)(x0 + k) < (unsigned)a.IW;
    auto load_row = [&](int (&d)[K]) {
        const bool yv = (unsigned)iy < (unsigned)a.IH;
#pragma unroll
        for (int k = 0; k < K; k++)
        {
            const bool ok = yv && xv[k];
            const int o   = ok ? off + k * a.C : 0;
            if constexpr (!RAGGED)
                d[k] = *reinterpret_cast<const int*>(a.in + (uint32_t)o);
            else
            {
                // (the last pixel's last group: its dword would end behind the tensor)
                const int at = o < a.in_last ? o : a.in_last;
                d[k]         = (int)((uint32_t)load4(a.in + (uint32_t)at) >> (8 * (o - at)));
            }
            d[k] = ok ? d[k] : za_word;
        }
        iy++, off += step;
    };
    auto quad = [](int d0, int d1, int d2, int d3, int* e) {
        // bytes (c0..c3) of four taps into bytes (tap0..tap3) of a channel
        const int t01_lo = __builtin_amdgcn_perm(d1, d0, 0x05010400), t01_hi = __builtin_amdgcn_perm(d1, d0, 0x07030602);
        const int t23_lo = __builtin_amdgcn_perm(d3, d2, 0x05010400), t23_hi = __builtin_amdgcn_perm(d3, d2, 0x07030602);
        e[0] = __builtin_amdgcn_perm(t23_lo, t01_lo, 0x05040100), e[1] = __builtin_amdgcn_perm(t23_lo, t01_lo, 0x07060302);
        e[2] = __builtin_amdgcn_perm(t23_hi, t01_hi, 0x05040100), e[3] = __builtin_amdgcn_perm(t23_hi, t01_hi, 0x07060302);
    };
    auto operands = [&](const int (&d)[K], int (&e)[Q]) {
        quad(d[0], d[1], d[2], K == 3 ? d[2] : d[3], e);    // (K = 3: the fourth byte meets a zero)
        if constexpr (K == 5)
            e[4] = d[4];
    };

    // the first rows are on their way while the constants are set up
    int first[K][K], next[S][K];
#pragma unroll
    for (int r = 0; r < K; r++)
        load_row(first[r]);

    // ---- per-lane constants ----------------------------------------------------------------------------
    int wq[K][K == 3 ? 4 : 8];
    int wsum[4] = { 0, 0, 0, 0 };
#pragma unroll
    for (int ky = 0; ky < K; ky++)
    {
        int d[K];
#pragma unroll
        for (int k = 0; k < K; k++)
        {
            const int o = (ky * K + k) * a.C + c0;
            if constexpr (!RAGGED)
                d[k] = *reinterpret_cast<const int*>(a.w + o);
            else
            {
                const int at = o < a.w_last ? o : a.w_last;
                d[k]         = (int)((uint32_t)load4(a.w + at) >> (8 * (o - at)));
            }
        }
        quad(d[0], d[1], d[2], K == 3 ? 0 : d[3], wq[ky]);
#pragma unroll
        for (int c = 0; c < 4; c++)
        {
            wsum[c] = __builtin_amdgcn_sdot4(wq[ky][c], 0x01010101, wsum[c], false);
            if constexpr (K == 5)
            {
                wq[ky][4 + c] = d[4] & (0xff << (8 * c));
                wsum[c]       = __builtin_amdgcn_sdot4(wq[ky][4 + c], 0x01010101, wsum[c], false);
            }
        }
    }
    uint32_t flags = 0;
    int32_t corr[4], mul[4] = {}, sh[4] = {}, zp_post[4] = {};
    uint32_t lim[4] = {};
    int64_t rnd_pos[4] = {}, rnd_neg[4] = {};
    bool check = false;    // some channel has a shift below 32: the value range must be tested
#pragma unroll
    for (int c = 0; c < 4; c++)
    {
        const int cc = c < live ? c0 + c : c0;
        corr[c]      = a.bias[a.bias_len == 1 ? 0 : cc] - a.za * wsum[c];
        if constexpr (RESCALE)
        {
            const int i           = a.rp.per_channel ? cc : 0;
            const ChannelScale cs = make_channel_scale(reinterpret_cast<const int32_t*>(a.rp.multiplier)[i], (int32_t)a.rp.shift[i],
                                                       a.rp.double_round != 0, flags);
            // the output zero point rides in the rounding term where that cannot overflow, else it is added last
            const bool fold       = cs.s <= zp_fold_max_shift(a.rp.out_zp);
            const int64_t zp_term = fold ? ((int64_t)a.rp.out_zp << cs.s) : 0;
            zp_post[c]            = fold ? 0 : a.rp.out_zp;
            mul[c] = cs.m, sh[c] = cs.s, lim[c] = cs.lim;
            rnd_pos[c] = cs.rnd_pos + zp_term, rnd_neg[c] = cs.rnd_neg + zp_term;
            check |= cs.lim != 0x80000000u;
        }
    }

    // ---- rows --------------------------------------------------------------------------------------------
    int e[K][Q];
#pragma unroll
    for (int r = 0; r < K; r++)
        operands(first[r], e[r]);
    size_t o = (((size_t)n * a.OH + oy0) * a.OW + ox) * a.C + c0;
    const size_t o_step = (size_t)a.OW * a.C;
    for (int oy = oy0; oy < oy_end; oy += K)
    {
#pragma unroll
        for (int u = 0; u < K; u++)
        {
            if (oy + u >= oy_end)
                break;
            const bool more = oy + u + 1 < oy_end;
            if (more)
#pragma unroll
                for (int s = 0; s < S; s++)
                    load_row(next[s]);    // on their way while this row is computed
            int32_t res[4];
#pragma unroll
            for (int c = 0; c < 4; c++)
            {
                int32_t v = corr[c];
#pragma unroll
                for (int ky = 0; ky < K; ky++)
                {
                    const int r = (u * S + ky) % K;
                    v           = __builtin_amdgcn_sdot4(e[r][c], wq[ky][c], v, false);
                    if constexpr (K == 5)
                        v = __builtin_amdgcn_sdot4(e[r][Q - 1], wq[ky][(4 + c) % (K == 3 ? 4 : 8)], v, false);
                }
                if constexpr (RESCALE)
                {
                    if (check && c < live && (uint32_t)v + lim[c] > 2u * lim[c] - 1u)
                        flags |= TMI_FLAG_SCALE_VALUE;
                    const int64_t pr = (int64_t)v * (int64_t)mul[c] + (v >= 0 ? rnd_pos[c] : rnd_neg[c]);
                    v                = (int32_t)(pr >> sh[c]) + zp_post[c];
                    v                = v < a.rp.lo ? a.rp.lo : v;
                    v                = v > a.rp.hi ? a.rp.hi : v;
                }
                res[c] = v;
            }
            auto each = [&](auto* p) {
                if (live == 4)
                {
                    struct __attribute__((packed)) Four
                    {
                        std::remove_reference_t<decltype(*p)> v[4];
                    } four;
#pragma unroll
                    for (int c = 0; c < 4; c++)
                        four.v[c] = (std::remove_reference_t<decltype(*p)>)res[c];
                    *reinterpret_cast<Four*>(p) = four;
                }
                else
#pragma unroll
                    for (int c = 0; c < 3; c++)
                        if (c < live)
                            p[c] = (std::remove_reference_t<decltype(*p)>)res[c];
            };
            if (!RESCALE || a.out_dtype == TMI_INT32)
                each(reinterpret_cast<int32_t*>(a.out) + o);
            else if (a.out_dtype == TMI_INT8)
                each(reinterpret_cast<int8_t*>(a.out) + o);
            else
                each(reinterpret_cast<int16_t*>(a.out) + o);
            o += o_step;
            if (more)
#pragma unroll
                for (int s = 0; s < S; s++)
                    operands(next[s], e[(u * S + s) % K]);
        }
    }
    raise_flags(a.flag_word, flags);
}

// nullptr: not this form's
const char* launch_depthwise_rows(hipStream_t st, int32_t in_dtype, int32_t out_dtype, const ConvGeom& g, const void* in, const void* w, const void* bias,
                                  int32_t in_zp, int32_t w_zp, const RescaleParams& rp, void* out, uint32_t* flag_word)
{
    if (in_dtype != TMI_INT8 || g.M != 1 || w_zp != 0 || g.IC < 1 || g.KH != g.KW || (g.KH != 3 && g.KH != 5) || g.stride_y != g.stride_x ||
        (g.stride_y != 1 && g.stride_y != 2) || g.dil_y != 1 || g.dil_x != 1 || (rp.enabled && !rp.fast) ||
        (rp.enabled ? out_dtype != TMI_INT8 && out_dtype != TMI_INT16 && out_dtype != TMI_INT32 : out_dtype != TMI_INT32))
        return nullptr;
    const int64_t in_bytes = (int64_t)g.N * g.IH * g.IW * g.IC, w_bytes = (int64_t)g.KH * g.KW * g.IC, groups = (g.IC + 3) / 4;
    const int64_t row = (int64_t)g.IW * g.IC;
    if (in_bytes < 4 || w_bytes < 4 || in_bytes > (1 << 30) || (g.pad_top + 1) * row + (int64_t)g.pad_left * g.IC > (1 << 29) ||
        ((uintptr_t)bias & 3) || (out_dtype == TMI_INT32 && ((uintptr_t)out & 3)) || (out_dtype == TMI_INT16 && ((uintptr_t)out & 1)) ||
        (int64_t)(g.OH + g.KH) * g.stride_y * row > (1 << 30))
        return nullptr;
    // Strips: long ones load and permute a strip's first rows and set its constants up for less, short ones give the chip more waves.  By
    // SIMD: waves (fewer than three are as slow as three) times rows, the set-up being some five rows' worth (5x5: eight); up to three waves a SIMD
    // that is a row a strip.  us for strips of about 2 / 4 / 12 waves a SIMD: 5x5 [62,16,16,56] 5.9 / 7.9 / 7.8, [36,132,137,40] 49 / 43 / 45, 3x3
    // [30,45,45,292] 24.4 / 22.0 / 22.7, [4,116,116,168] 15.1 / 12.6 / 15.4, [58,38,38,22] 7.5 / 7.4 / 9.8.
    const int64_t columns = (int64_t)g.N * g.OW * groups;
    int64_t strips        = g.OH;
    if (columns * g.OH > 3 * 1024 * 64)
    {
        int64_t least = INT64_MAX;
        for (const int s : { 1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24, 32, 48, 64, 128, 256 })
        {
            if (s > g.OH)
                break;
            const int64_t rows = (g.OH + s - 1) / s, waves = ((g.OH + rows - 1) / rows * columns + 63) / 64, each = (waves + 1023) / 1024;
            const int64_t cost = (each < 3 ? 3 : each) * (rows + (g.KH == 3 ? 5 : 8));
            if (cost < least)
                strips = s, least = cost;
        }
    }
    const int64_t rows = (g.OH + strips - 1) / strips;
    strips             = (g.OH + rows - 1) / rows;
    const int64_t lanes = columns * strips;
    if (lanes > (1 << 30) || !fastdiv_exact_up_to((uint64_t)lanes + 256, (uint32_t)groups) || !fastdiv_exact_up_to((uint64_t)lanes / groups + 256, (uint32_t)g.OW) ||
        !fastdiv_exact_up_to((uint64_t)lanes / groups / g.OW + 256, (uint32_t)strips))
        return nullptr;
    DwRowsArgs a{};
    a.in = (const int8_t*)in, a.w = (const int8_t*)w, a.bias = (const int32_t*)bias, a.out = out, a.flag_word = flag_word, a.rp = rp;
    a.C = g.IC, a.IH = g.IH, a.IW = g.IW, a.OH = g.OH, a.OW = g.OW, a.pad_top = g.pad_top, a.pad_left = g.pad_left, a.bias_len = g.bias_len;
    a.groups = (int32_t)groups, a.rows = (int32_t)rows, a.lanes = (int32_t)lanes, a.in_last = (int32_t)(in_bytes - 4), a.w_last = (int32_t)(w_bytes - 4);
    a.za = in_zp, a.out_dtype = out_dtype;
    a.div_groups = make_fastdiv((uint32_t)groups), a.div_ow = make_fastdiv((uint32_t)g.OW), a.div_strips = make_fastdiv((uint32_t)strips);
    const int64_t grid = (lanes + 255) / 256;
    a.per_xcd          = (uint32_t)(grid / 8);
    const bool ragged  = g.IC % 4 != 0 || (((uintptr_t)in | (uintptr_t)w) & 3);
#define TMI_ROWS(K, S, R)                                                                                             \
    if (g.KH == K && g.stride_y == S && ragged == R)                                                                  \
    {                                                                                                                 \
        if (rp.enabled)                                                                                               \
            hipLaunchKernelGGL((depthwise_rows_kernel<K, S, R, true>), dim3((unsigned)grid), dim3(256), 0, st, a);    \
        else                                                                                                          \
            hipLaunchKernelGGL((depthwise_rows_kernel<K, S, R, false>), dim3((unsigned)grid), dim3(256), 0, st, a);   \
    }
    TMI_ROWS(3, 1, false)
    TMI_ROWS(3, 1, true)
    TMI_ROWS(3, 2, false)
    TMI_ROWS(3, 2, true)
    TMI_ROWS(5, 1, false)
    TMI_ROWS(5, 1, true)
    TMI_ROWS(5, 2, false)
    TMI_ROWS(5, 2, true)
#undef TMI_ROWS
    return rp.enabled ? "depthwise_rows_i8_rescale" : "depthwise_rows_i8";
}

}    // namespace tmi
