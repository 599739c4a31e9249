// INT16 x INT8 -> INT48 CONV2D of any channel count whose weights stay in LDS while the pixels stream past them; the split of an int16
// value into two int8 and the arithmetic are those of conv_i16.hip.
//
// K is walked in chunks of 16 channels of one tap, (ky, kx, ic) in order, four chunks a matrix instruction (16 x 16 results, lane = row or
// column lane % 16, chunk lane / 16).  A workgroup of four waves stages the weights of 16 * CT channels once in the order the instructions
// read them, a fragment 1 KB side by side; the last chunk of a tap is filled up with zeros, so whatever the pixel holds behind its
// channels counts for nothing.  Then every wave walks tiles of 16 pixels on its own (SPLIT: the four share a tile's K and meet in LDS):
// a lane loads the 32 bytes of its chunk straight from the image, or from a page of zeros where the tap lies outside, DEPTH steps ahead;
// four lanes side by side hold neighbouring chunks, so a load instruction touches 16 lines where 32 pixels a tile touch 32.  What a chunk
// adds to the pixel's offset and which of the pixel's row and column bits it needs is read from a table in LDS.  Pixels are the rows of
// the result: 16 lanes store 128 neighbouring bytes.
//
// What bounds it: the chain of a call - weights, table, the first tile's pixels on their way while those are staged, a wave's steps, the
// stores - with a tile or two to a wave.  us conv_i16.hip (with its copies where the channels are no whole chunks) / here: [8,56,56,64]->64 3x3
// 12.2 / 10.5 (16 MB; 9.5 without the pixels' loads, 9.7 without the weights', 9.4 without the stores), [23128 pixels,56]->16 3x3 16.0 / 7.4,
// [13464,24]->16 3x3 stride 2 11.4 / 5.2, [7560,312]->32 3x3 20.1 / 14.1, [16646,49]->32 1x1 9.7 / 5.1, [140,33]->64 1x1 6.9 / 3.8, [360,16]->72 3x3
// 4.7 / 3.7; the other way, and so left there: [960,431]->189 3x3 18.7 / 30.8, [930,213]->136 3x3 11.8 / 18.8.
#include <type_traits>

#include "tmi_mfma.h"

namespace tmi
{

struct I16TapsArgs
{
    const uint8_t* in;
    const uint8_t* w;
    const int64_t* bias;
    int64_t* out;
    const uint8_t* zeros;    // 64 bytes
    int32_t P, OC, OH, OW, IH, IW, KW, KH;
    int32_t sy, sx, dy, dx, pad_top, pad_left;
    int32_t IC, pieces;      // chunks of a tap
    int32_t chunks, steps;
    int32_t bias_len, n_pt, groups;    // tiles of 16 pixels; workgroups of a channel block
    int32_t in_last, w_last;           // offsets of the last 16 bytes of the input, of the weights
    int32_t edge_off;                  // a window that begins further on may reach beyond the input's last 32 bytes
    FastDiv div_ow, div_oh, div_pieces, div_kw, div_groups;
};

constexpr int kI16Dead = 1 << 26;    // table entry: no chunk at all

__device__ __forceinline__ int64_t clip48(int64_t v)
{
    const int64_t top = (int64_t(1) << 47) - 1;
    return v > top ? top : (v < -top - 1 ? -top - 1 : v);
}

template <int CT, bool SPLIT>
constexpr int i16_taps_fixed_lds()
{
    return 16 * CT * 8 + 4 * CT * 16 * 4 + (SPLIT ? 4 * CT * 2048 : 0);
}
template <int CT, bool SPLIT>
constexpr int64_t i16_taps_lds(int64_t steps)
{
    return i16_taps_fixed_lds<CT, SPLIT>() + steps * (CT * 1024 + 32);
}

template <int CT, bool SPLIT, bool RAGGED>
__global__ __launch_bounds__(256, 2) void conv_i16_taps_kernel(I16TapsArgs a)
{
    constexpr int DEPTH = 6;
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    int64_t* tab_base = reinterpret_cast<int64_t*>(lds);                        // bias + 128 sum w of a channel
    int* tab_part     = reinterpret_cast<int*>(lds + 16 * CT * 8);              // a wave's part of sum w
    v4i* part         = reinterpret_cast<v4i*>(lds + 16 * CT * 8 + 4 * CT * 16 * 4);
    v2i* tab_chunk    = reinterpret_cast<v2i*>(lds + i16_taps_fixed_lds<CT, SPLIT>());
    uint8_t* wl       = reinterpret_cast<uint8_t*>(tab_chunk + 4 * a.steps);

    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ocb = (int)fdiv(blockIdx.x, a.div_groups), grp = (int)blockIdx.x - ocb * a.groups;
    const int oc0 = ocb * 16 * CT;

    // ---- weights into registers (on their way while the table is written), then LDS: a wave takes fragments of one channel tile ------
    int sum_w          = 0;
    const int ct_w     = wave % CT;                     // (CT 1, 2 or 4: the fragments wave, wave + 4, ... are of one channel tile)
    constexpr int SKIP = 4 / CT, WB = RAGGED ? 8 : 12;    // steps from one fragment of the wave to the next; fragments in flight
    const int w_oc     = oc0 + 16 * ct_w + l16;
    const int w_row    = (w_oc < a.OC ? w_oc : 0) * (a.KH * a.KW) * a.IC;
    v4i wv[WB];
    auto load_weights = [&](int s0) {
#pragma unroll
        for (int u = 0; u < WB; u++)
        {
            const int s = s0 + u * SKIP, c = 4 * s + q;
            if (s >= a.steps)
                continue;
            const bool ok = w_oc < a.OC && c < a.chunks;
            if constexpr (!RAGGED)
                wv[u] = *reinterpret_cast<const v4i*>(a.w + (uint32_t)(ok ? w_row + c * 16 : 0));
            else
            {
                const int cc  = ok ? c : 0;
                const int tap = (int)fdiv((uint32_t)cc, a.div_pieces), piece = cc - tap * a.pieces;
                const int off = w_row + tap * a.IC + piece * 16, at = off <= a.w_last ? off : a.w_last;
                wv[u]         = load16(a.w + (uint32_t)at);
                if (__any(off > at))
                    wv[u] = drop_front(wv[u], off - at);
                wv[u] = keep_bytes(wv[u], a.IC - piece * 16);    // channels of the chunk
            }
            if (!ok)
                wv[u] = v4i{ 0, 0, 0, 0 };
        }
    };
    auto store_weights = [&](int s0) {
#pragma unroll
        for (int u = 0; u < WB; u++)
            if (s0 + u * SKIP < a.steps)
            {
                sum_w += dot4_ones(wv[u]);
                *reinterpret_cast<v4i*>(wl + ((s0 + u * SKIP) * CT + ct_w) * 1024 + lane * 16) = wv[u];
            }
    };
    load_weights(wave / CT);
    const int64_t bias = tid < 16 * CT && oc0 + tid < a.OC ? a.bias[a.bias_len == 1 ? 0 : oc0 + tid] : 0;
    for (int c = tid; c < 4 * a.steps; c += 256)
    {
        v2i e = { 0, kI16Dead };
        if (c < a.chunks)
        {
            const int tap = (int)fdiv((uint32_t)c, a.div_pieces), piece = c - tap * a.pieces;
            const int ky = (int)fdiv((uint32_t)tap, a.div_kw), kx = tap - ky * a.KW;
            e.x = ((ky * a.dy * a.IW + kx * a.dx) * a.IC + piece * 16) * 2;
            e.y = (1 << ky) | (1 << (13 + kx));
        }
        tab_chunk[c] = e;
    }
    __syncthreads();

    // ---- pixels ---------------------------------------------------------------------------------------------------------
    const int share = SPLIT ? (a.steps + 3) / 4 : a.steps, s_first = SPLIT ? wave * share : 0;
    const int s_end = s_first + share < a.steps ? s_first + share : a.steps, n_steps = s_end > s_first ? s_end - s_first : 0;
    const int first_pt = SPLIT ? grp : grp * 4 + wave, pt_step = SPLIT ? a.groups : a.groups * 4;
    const v2i* chunk_q = tab_chunk + 4 * s_first + q;
    const uint8_t* wf  = wl + s_first * CT * 1024 + lane * 16;
    int pix_off = 0, miss = -1;    // offset of the window's first tap; a zero bit per tap row and column inside the image
    bool edge = false;             // RAGGED: the tensor may end inside the 32 bytes of a lane of this tile
    v4i xv[DEPTH][2];
    auto request = [&](int d, int s, auto careful) {
        const v2i e        = chunk_q[4 * s];
        const bool inside  = (e.y & miss) == 0;
        const int off      = pix_off + e.x;
        const uint8_t* src = inside ? a.in + (uint32_t)off : a.zeros;
        if constexpr (!RAGGED)
            xv[d][0] = reinterpret_cast<const v4i*>(src)[0], xv[d][1] = reinterpret_cast<const v4i*>(src)[1];
        else if constexpr (!decltype(careful)::value)
            xv[d][0] = load16(src), xv[d][1] = load16(src + 16);
        else
#pragma unroll
            for (int j = 0; j < 2; j++)
            {
                // (what lies 16 bytes or more past the last load is behind the channels: any value will do)
                const int past = inside && off + 16 * j > a.in_last ? off + 16 * j - a.in_last : 0;
                xv[d][j]       = drop_front(load16(src + 16 * j - past), past & 15);
            }
    };
    auto enter_tile = [&](int pt) {
        int p = pt * 16 + l16;
        p     = p < a.P ? p : a.P - 1;
        const int r = (int)fdiv((uint32_t)p, a.div_ow), ox = p - r * a.OW, n = (int)fdiv((uint32_t)r, a.div_oh), oy = r - n * a.OH;
        const int y0 = oy * a.sy - a.pad_top, x0 = ox * a.sx - a.pad_left;
        pix_off      = ((n * a.IH + y0) * a.IW + x0) * a.IC * 2;
        int in_bits  = 0;
        for (int k = 0; k < a.KH; k++)
            in_bits |= ((unsigned)(y0 + k * a.dy) < (unsigned)a.IH ? 1 : 0) << k;
        for (int k = 0; k < a.KW; k++)
            in_bits |= ((unsigned)(x0 + k * a.dx) < (unsigned)a.IW ? 1 : 0) << (13 + k);
        miss = ~in_bits;
        if constexpr (RAGGED)
            edge = __any(pix_off > a.edge_off);
        auto first_steps = [&](auto careful) {
#pragma unroll
            for (int d = 0; d < DEPTH; d++)
                if (d < n_steps)
                    request(d, d, careful);
        };
        if (RAGGED && edge)
            first_steps(std::true_type{});
        else
            first_steps(std::false_type{});
    };
    if (first_pt < a.n_pt)
        enter_tile(first_pt);
    store_weights(wave / CT);
    for (int s0 = wave / CT + WB * SKIP; s0 < a.steps; s0 += WB * SKIP)
    {
        load_weights(s0);
        store_weights(s0);
    }
    sum_w += __shfl_xor(sum_w, 16);
    sum_w += __shfl_xor(sum_w, 32);
    if (lane < 16)
        tab_part[(wave / CT) * (16 * CT) + 16 * ct_w + lane] = sum_w;
    __syncthreads();
    if (tid < 16 * CT)
    {
        int64_t sum = 0;
#pragma unroll
        for (int k = 0; k < 4 / CT; k++)
            sum += tab_part[k * (16 * CT) + tid];
        tab_base[tid] = bias + 128 * sum;
    }
    __syncthreads();

    for (int pt = first_pt; pt < a.n_pt; pt += pt_step)
    {
        if (pt != first_pt)
            enter_tile(pt);
        v4i hi[CT], lo[CT];
#pragma unroll
        for (int t = 0; t < CT; t++)
            hi[t] = lo[t] = v4i{ 0, 0, 0, 0 };
        auto consume = [&](int d, int s) {
            v4i h, l;
#pragma unroll
            for (int i = 0; i < 4; i++)
            {
                const uint32_t u = (uint32_t)xv[d][i >> 1][2 * (i & 1)], v = (uint32_t)xv[d][i >> 1][2 * (i & 1) + 1];
                h[i] = (int)__builtin_amdgcn_perm(v, u, 0x07050301u);
                l[i] = (int)(__builtin_amdgcn_perm(v, u, 0x06040200u) ^ 0x80808080u);
            }
#pragma unroll
            for (int t = 0; t < CT; t++)
            {
                const v4i b = *reinterpret_cast<const v4i*>(wf + (s * CT + t) * 1024);
                hi[t]       = __builtin_amdgcn_mfma_i32_16x16x64_i8(h, b, hi[t], 0, 0, 0);
                lo[t]       = __builtin_amdgcn_mfma_i32_16x16x64_i8(l, b, lo[t], 0, 0, 0);
            }
        };
        auto walk = [&](auto careful) {
            int s = 0;
            for (; s + 2 * DEPTH <= n_steps; s += DEPTH)    // (whole groups with whole groups behind: no test)
#pragma unroll
                for (int d = 0; d < DEPTH; d++)
                {
                    consume(d, s + d);
                    request(d, s + d + DEPTH, careful);
                }
            for (; s < n_steps; s += DEPTH)
#pragma unroll
                for (int d = 0; d < DEPTH; d++)
                    if (s + d < n_steps)
                    {
                        consume(d, s + d);
                        if (s + d + DEPTH < n_steps)
                            request(d, s + d + DEPTH, careful);
                    }
        };
        if (RAGGED && edge)
            walk(std::true_type{});
        else
            walk(std::false_type{});

        auto store = [&](int t, int i, int64_t v) {
            const int px = pt * 16 + 4 * q + i, c = 16 * t + l16;
            if (px < a.P && oc0 + c < a.OC)
                a.out[(int64_t)px * a.OC + oc0 + c] = clip48(tab_base[c] + v);
        };
        if constexpr (!SPLIT)
        {
#pragma unroll
            for (int t = 0; t < CT; t++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    store(t, i, 256 * (int64_t)hi[t][i] + (int64_t)lo[t][i]);
        }
        else
        {
            // the parts of a tile meet: channel tile by channel tile, a wave adds up row i = wave of every four
#pragma unroll
            for (int t = 0; t < CT; t++)
                part[(wave * CT + t) * 128 + lane] = hi[t], part[(wave * CT + t) * 128 + 64 + lane] = lo[t];
            __syncthreads();
            const int* p4 = reinterpret_cast<const int*>(part);
#pragma unroll
            for (int t = 0; t < CT; t++)
            {
                int h = 0, l = 0;
#pragma unroll
                for (int k = 0; k < 4; k++)
                {
                    const int* from = p4 + ((k * CT + t) * 128 + lane) * 4 + wave;
                    h += from[0], l += from[256];
                }
                store(t, wave, 256 * (int64_t)h + (int64_t)l);
            }
            __syncthreads();
        }
    }
}

struct I16Form
{
    int ct, split;    // ct 0: none
    double us;
};
// The quickest form by a model fitted to 260 layers of 1x1 ... 3x3 taps on 8 ... 512 channels (each form's times within 6 ... 12 % of it; picked by it a
// layer is 1 ... 2 % from its best form): a call, the staged weights, and per round of workgroups of a CU the steps a wave walks, alone or
// beside the waves of `busy` workgroups, the instructions of its channel tiles and their stores.  Rows: channels of whole chunks, even, odd
// (loads that start between words).
static I16Form i16_taps_form(const ConvGeom& g, int64_t steps)
{
    static const double fit[3][5][6] = {
        // call, staging, chain, step x channel tile, store, step
        { { 3.06, 0.035, 0, 0.147, 0.28, 0 }, { 3.30, 0.023, 0, 0.082, 0.204, 0 }, { 3.36, 0.036, 0, 0.045, 0.207, 0 },
          { 3.12, 0.024, 0.065, 0.132, 0.208, 0 }, { 2.99, 0.019, 0.155, 0.054, 0.211, 0 } },
        { { 3.20, 0.152, 0, 0, 0.525, 0.101 }, { 3.35, 0.061, 0, 0.102, 0.293, 0 }, { 2.65, 0.148, 0, 0.010, 0.333, 0 },
          { 2.72, 0.097, 0.126, 0.058, 0.623, 0 }, { 2.77, 0.085, 0.047, 0.064, 0.362, 0 } },
        { { 3.56, 0.023, 0, 0.414, 0, 0 }, { 3.85, 0.027, 0, 0.233, 0, 0 }, { 3.30, 0.112, 0, 0.093, 0.176, 0 },
          { 2.85, 0.071, 0, 0.516, 0.210, 0 }, { 2.28, 0.053, 0.682, 0, 0.422, 0 } },
    };
    const int64_t n_pt = ((int64_t)g.N * g.OH * g.OW + 15) / 16;
    const auto& rows   = fit[g.IC % 16 == 0 ? 0 : (g.IC % 2 == 0 ? 1 : 2)];
    I16Form best{ 0, 0, 1e30 };
    for (int f = 0; f < 5; f++)    // (four tiles and a split: never the quickest)
    {
        const int ct = 1 << (f % 3), split = f / 3;
        const int64_t lds = steps * (ct * 1024 + 32) + ct * (384 + split * 8192);
        if (lds > 150 * 1024 || (ct > 1 && 8 * ct >= g.OC))
            continue;
        const int64_t blocks = (g.OC + 16 * ct - 1) / (16 * ct), wanted = (split ? n_pt : (n_pt + 3) / 4) * blocks, rounds = (wanted + 255) / 256;
        const int64_t held = lds > 80 * 1024 ? 1 : (lds > 53 * 1024 ? 2 : (lds > 40 * 1024 ? 3 : 4)), busy = rounds < held ? rounds : held;
        const double r = (double)rounds, walked = (double)(split ? (steps + 3) / 4 : steps);
        const auto& c   = rows[f];
        const double us = c[0] + c[1] * (double)(steps * ct) + c[2] * r * walked / (double)busy + c[3] * r * walked * ct + c[4] * r * ct + c[5] * r * walked;
        if (us < best.us)
            best = I16Form{ ct, split, us };
    }
    return best;
}
// The same for conv_i16.hip, with its copies where it needs them (all within 8 %).
static double i16_gather_us(const ConvGeom& g)
{
    const int64_t pixels = (int64_t)g.N * g.OH * g.OW, tiles = (pixels + 31) / 32, steps = ((int64_t)g.KH * g.KW * ((g.IC + 15) / 16) + 1) / 2;
    const bool two = g.OC > 32 && tiles * ((g.OC + 63) / 64) >= 512;
    const int64_t units = tiles * (two ? (g.OC + 63) / 64 : (g.OC + 31) / 32);
    const int64_t split = two ? 1 : (units <= 512 && steps >= 4 ? 4 : (units <= 1024 && steps >= 2 ? 2 : 1)), walked = (steps + split - 1) / split;
    static const double fit[3][6] = { { 3.98, 0.064, 0.093, 0.114, 0.186, 0 }, { 5.84, 0.151, 0.074, 0.166, 0.200, 1.046 }, { 5.93, 0.247, 0.003, 0.092, 0.299, 0.803 } };
    const auto& c                 = fit[g.IC % 16 == 0 ? 0 : (g.IC % 2 == 0 ? 1 : 2)];
    return c[0] + c[1] * (double)walked + c[2] * (double)(units * steps * (two ? 2 : 1)) / 1024 + c[3] * (double)((units * split + 1023) / 1024 * walked) +
           c[4] * (double)(pixels * g.OC) * 8e-6 + c[5] * (double)pixels * g.IC * 2e-6;
}

template <int CT, bool SPLIT, bool RAGGED>
static bool launch_i16_taps(hipStream_t st, I16TapsArgs& a)
{
    const int64_t lds = i16_taps_lds<CT, SPLIT>(a.steps);
    constexpr auto kern = conv_i16_taps_kernel<CT, SPLIT, RAGGED>;
    if (lds > 65536 && !ensure_dynamic_lds<kern>((size_t)lds))
        return false;
    // as many workgroups as the chip holds, for each channel block: the ragged forms' registers, 140 and more, leave three waves a SIMD, and a fourth
    // workgroup of a CU would begin, and stage its weights, when another ends.  us four / three: 1x1 [14,127,114,11]->48 27.7 / 21.6, [30,86,86,40]->16
    // 16.7 / 13.3, 3x3 [32,50,50,20]->164 38.4 / 30.6, [27,82,93,9]->16 22.9 / 18.8; the other way [21,72,72,104]->18 stride 2 12.7 / 13.9
    const int64_t blocks = (a.OC + 16 * CT - 1) / (16 * CT), rounds = SPLIT ? a.n_pt : (a.n_pt + 3) / 4;
    const int64_t held = lds > 80 * 1024 ? 1 : (lds > 53 * 1024 ? 2 : (RAGGED || lds > 40 * 1024 ? 3 : 4)), most = (256 * held + blocks - 1) / blocks;
    const int64_t each = (rounds + most - 1) / most;
    a.groups           = (int32_t)((rounds + each - 1) / each);
    if (!fastdiv_exact_up_to((uint64_t)a.groups * blocks, (uint32_t)a.groups))
        return false;
    a.div_groups = make_fastdiv((uint32_t)a.groups);
    hipLaunchKernelGGL(kern, dim3((unsigned)(a.groups * blocks)), dim3(256), (size_t)lds, st, a);
    return true;
}

// zeros: 64 bytes of them; or_gather: conv_i16.hip may take the layer where it leads.  nullptr: not this form's
const char* launch_conv_i16_taps(hipStream_t st, const ConvGeom& g, const void* in, const void* w, const void* bias, void* out, const void* zeros, bool or_gather)
{
    const int64_t pixels = (int64_t)g.N * g.OH * g.OW, pieces = (g.IC + 15) / 16, chunks = (int64_t)g.KH * g.KW * pieces;
    const int64_t in_bytes = (int64_t)g.N * g.IH * g.IW * g.IC * 2, w_bytes = (int64_t)g.OC * g.KH * g.KW * g.IC;
    // the window's reach beyond the image, twice, stays within 32-bit offsets
    const int64_t reach = ((int64_t)(g.KH - 1) * g.dil_y + g.pad_top + 1) * g.IW * g.IC * 2 + ((int64_t)(g.KW - 1) * g.dil_x + g.pad_left + 1) * g.IC * 2;
    if (g.IC < 1 || g.KH > 13 || g.KW > 13 || chunks * 16 > 65536 || pixels > INT32_MAX - 64 || in_bytes < 16 || w_bytes < 16 || w_bytes > INT32_MAX ||
        in_bytes + 2 * reach > INT32_MAX || (((uintptr_t)in) & 1) || !fastdiv_exact_up_to((uint64_t)pixels, (uint32_t)g.OW) ||
        !fastdiv_exact_up_to((uint64_t)pixels / g.OW, (uint32_t)g.OH) || !fastdiv_exact_up_to((uint64_t)chunks, (uint32_t)pieces) ||
        !fastdiv_exact_up_to((uint64_t)g.KH * g.KW, (uint32_t)g.KW))
        return nullptr;
    I16TapsArgs a{};
    a.in = (const uint8_t*)in, a.w = (const uint8_t*)w, a.bias = (const int64_t*)bias, a.out = (int64_t*)out, a.zeros = (const uint8_t*)zeros;
    a.P = (int32_t)pixels, a.OC = g.OC, a.OH = g.OH, a.OW = g.OW, a.IH = g.IH, a.IW = g.IW, a.KW = g.KW, a.KH = g.KH;
    a.sy = g.stride_y, a.sx = g.stride_x, a.dy = g.dil_y, a.dx = g.dil_x, a.pad_top = g.pad_top, a.pad_left = g.pad_left;
    a.IC = g.IC, a.pieces = (int32_t)pieces, a.chunks = (int32_t)chunks, a.steps = (int32_t)((chunks + 3) / 4);
    a.bias_len = g.bias_len, a.n_pt = (int32_t)((pixels + 15) / 16);
    a.in_last = (int32_t)(in_bytes - 16), a.w_last = (int32_t)(w_bytes - 16);
    // the furthest chunk of a window, from the window's first tap
    const int64_t furthest = (((int64_t)(g.KH - 1) * g.dil_y * g.IW + (int64_t)(g.KW - 1) * g.dil_x) * g.IC + (pieces - 1) * 16) * 2;
    a.edge_off             = (int32_t)(in_bytes - 32 - furthest);
    a.div_ow = make_fastdiv((uint32_t)g.OW), a.div_oh = make_fastdiv((uint32_t)g.OH);
    a.div_pieces = make_fastdiv((uint32_t)pieces), a.div_kw = make_fastdiv((uint32_t)g.KW);
    const bool ragged = g.IC % 16 != 0 || ((((uintptr_t)in | (uintptr_t)w) & 15) != 0);
    const I16Form f   = i16_taps_form(g, a.steps);
    if (!f.ct || (or_gather && i16_gather_us(g) < 1.04 * f.us))
        return nullptr;
    bool ok           = false;
#define TMI_I16(C, S)                                                                                                 \
    if (f.ct == C && f.split == S)                                                                                    \
        ok = ragged ? launch_i16_taps<C, S, true>(st, a) : launch_i16_taps<C, S, false>(st, a);
    TMI_I16(1, 0)
    TMI_I16(2, 0)
    TMI_I16(4, 0)
    TMI_I16(1, 1)
    TMI_I16(2, 1)
#undef TMI_I16
    return ok ? "conv2d_mfma_i16_i48" : nullptr;
}

}    // namespace tmi
