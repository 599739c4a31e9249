// TRANSPOSE_CONV2D int8 -> int32 with a stride, operands read where they lie (tensor_ops.cpp:2138-2187).
//
// out[oy][ox] takes weight tap (ky, kx) from input pixel ((oy - top - ky) / sy, (ox - left - kx) / sx) where those divide evenly, so the output
// pixels of one class (oy % sy, ox % sx) are a CONV2D with stride 1 over the input with the taps of one residue, walked backwards: a
// quarter of the products of the CONV2D over the input with holes at stride 2, and nothing to copy.  Class by class it is the kernel
// with resident weights (see conv_i16_taps.hip): a workgroup of four waves belongs to a class and a block of 16 * CT channels, stages the
// weights of its taps once in fragment order (a fragment 1 KB: 16 channels x four chunks of 16 bytes), and its waves walk tiles of 16 of the
// class's pixels, a lane loading the 16 bytes of its chunk straight from the image, or from the page of input_zp bytes where the tap lies
// outside, DEPTH steps ahead.  Rows of the result are pixels: 16 lanes store 64 neighbouring bytes.
//
// What bounds it: the chain of a call (weights and the first pixels on their way together, a few steps, the stores).  us copies and CONV2D / here,
// stride 2 (class pixels): 3x3 [1968,88]->21 7.3 / 4.7, [273,88]->48 2x2 6.4 / 4.5, [4465,48]->96 2x2 12.7 / 5.7, 4x4 [1368,88]->157 16.3 / 6.7,
// [16632,184]->24 36.8 / 12.1, [4312,208]->48 2x2 15.0 / 5.5, [520,152]->56 3x3 7.4 / 6.6; the slab kernel's layers stay there ([6272,128]->64 3x3
// 7.2 / 7.7: its patch serves all classes).  (These before the arguments came in one trip and a batch of weights in flight: now 0.90 of it over 552 layers.)
#include <algorithm>
#include <type_traits>

#include "tmi_mfma.h"

namespace tmi
{

constexpr int kTconvStrides = 4;    // largest stride

struct TconvAxis
{
    // per residue: the first weight tap, the number of taps, the input position under the first tap of the class's first pixel
    int8_t first[kTconvStrides], taps[kTconvStrides];
    int16_t base[kTconvStrides];
};
struct TconvArgs    // (at most 256 bytes: a larger launch takes the host longer)
{
    const uint8_t* in;
    const uint8_t* w;
    const int32_t* bias;
    int32_t* out;
    const uint8_t* page;     // 16 bytes of input_zp
    TconvAxis y, x;
    int32_t P, OC, OH, OW, IH, IW, KH, KW, sy, sx;    // P: pixels of a class
    int32_t IC, pieces;      // chunks of a tap
    int32_t steps;           // of the class with the most taps
    int32_t bias_len, n_pt, groups, classes;    // tiles of 16 pixels of a class; workgroups of a channel block and class
    int32_t in_last, w_last;           // offsets of the last 16 bytes of the input, of the weights
    int32_t edge_off;                  // a window that begins further on may reach beyond the input's last 16 bytes
    int32_t za;
    uint16_t taps_x_magic[kTconvStrides];    // 65536 / taps, rounded up: exact for the at most 169 taps
    FastDiv div_ow, div_oh, div_pieces, div_groups, div_classes, div_sx;    // (div_ow, div_oh: columns and rows of a class)
};

constexpr int kTconvDead = 1 << 26;    // table entry: no chunk at all

template <int CT>
constexpr int64_t tconv_lds(int64_t steps)
{
    return 16 * CT * 4 + 4 * CT * 16 * 4 + steps * (CT * 1024 + 32);
}

template <int CT, bool RAGGED>
__global__ __launch_bounds__(256, 2) void tconv_taps_kernel(TconvArgs a)
{
    constexpr int DEPTH = 6;
    // The arguments at once.  (Left to the compiler they come where they are used, and the classes' by vector loads: eight trips one after the other
    // before the first operand; [1,7,5,42]->64 2x2 stride 2 4.3 us, so 3.8.)
    asm volatile("" ::"s"(a.in), "s"(a.w), "s"(a.bias), "s"(a.out), "s"(a.page), "s"(a.OC), "s"(a.OH), "s"(a.OW), "s"(a.IH), "s"(a.IW), "s"(a.KH), "s"(a.KW),
                 "s"(a.sy), "s"(a.sx), "s"(a.IC), "s"(a.pieces), "s"(a.groups), "s"(a.classes), "s"(a.w_last), "s"(a.bias_len), "s"(a.P), "s"(a.n_pt));
    asm volatile("" ::"s"(a.div_groups.magic), "s"(a.div_groups.d), "s"(a.div_classes.magic), "s"(a.div_classes.d), "s"(a.div_sx.magic), "s"(a.div_sx.d),
                 "s"(a.div_pieces.magic), "s"(a.div_pieces.d));
    auto entry8  = [](const int8_t (&v)[kTconvStrides], int c) { uint32_t u; __builtin_memcpy(&u, v, 4); return (int)(int8_t)(u >> (8 * c)); };
    auto entry16 = [](const auto& v, int c) { uint64_t u; __builtin_memcpy(&u, v, 8); return (uint32_t)(u >> (16 * c)) & 0xffffu; };
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    int* tab_base  = reinterpret_cast<int*>(lds);                   // bias - input_zp sum w of a channel
    int* tab_part  = reinterpret_cast<int*>(lds + 16 * CT * 4);     // a wave's part of sum w
    v2i* tab_chunk = reinterpret_cast<v2i*>(lds + 16 * CT * 4 + 4 * CT * 16 * 4);
    uint8_t* wl    = reinterpret_cast<uint8_t*>(tab_chunk + 4 * a.steps);

    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int unit = (int)fdiv(blockIdx.x, a.div_groups), grp = (int)blockIdx.x - unit * a.groups;
    const int ocb = (int)fdiv((uint32_t)unit, a.div_classes), cls = unit - ocb * a.classes;
    const int cy = (int)fdiv((uint32_t)cls, a.div_sx), cx = cls - cy * a.sx;
    const int oc0 = ocb * 16 * CT;
    const int taps_y = entry8(a.y.taps, cy), taps_x = entry8(a.x.taps, cx), first_y = entry8(a.y.first, cy), first_x = entry8(a.x.first, cx);
    const int base_y = (int16_t)entry16(a.y.base, cy), base_x = (int16_t)entry16(a.x.base, cx);
    const uint32_t magic_x = entry16(a.taps_x_magic, cx);    // (0: one tap)
    auto row_of = [&](int tap) { return magic_x ? (int)((uint32_t)tap * magic_x >> 16) : tap; };
    const int chunks = taps_y * taps_x * a.pieces, steps = (chunks + 3) >> 2;

    // ---- weights into registers (on their way while the table is written), then LDS: a wave takes fragments of one channel tile ------
    int sum_w          = 0;
    const int ct_w     = wave % CT;                     // (CT 1, 2 or 4: the fragments wave, wave + 4, ... are of one channel tile)
    constexpr int SKIP = 4 / CT, WB = RAGGED ? 8 : 12;    // steps from one fragment of the wave to the next; fragments in flight
    const int w_oc     = oc0 + 16 * ct_w + l16;
    const int w_row    = (w_oc < a.OC ? w_oc : 0) * (a.KH * a.KW) * a.IC;
    v4i wv[WB];
    int wfix[WB];    // RAGGED: what is left of a chunk after the load (bytes before it << 8 | its channels)
    // (a load's result is not looked at here, so that all of a batch are in flight at once: [8,6,5,584]->176 4x4 14.4 us with the fix-ups behind each load, so 11.6)
    auto load_weights = [&](int s0) {
        auto load = [&](int u) {
            const int c   = 4 * (s0 + u * SKIP) + q;
            const bool ok = w_oc < a.OC && c < chunks;
            const int cc  = ok ? c : 0;
            const int tap = (int)fdiv((uint32_t)cc, a.div_pieces), piece = cc - tap * a.pieces;
            const int ty  = row_of(tap), tx = tap - ty * taps_x;
            const int off = w_row + ((first_y + ty * a.sy) * a.KW + first_x + tx * a.sx) * a.IC + piece * 16;
            if constexpr (!RAGGED)
                wv[u] = *reinterpret_cast<const v4i*>(a.w + (uint32_t)off);
            else
            {
                const int at = off <= a.w_last ? off : a.w_last, n = a.IC - piece * 16;
                wv[u]        = load16(a.w + (uint32_t)at);
                wfix[u]      = (off - at) << 8 | (ok ? (n < 16 ? n : 16) : 0);
            }
        };
        if (s0 + (WB - 1) * SKIP < steps)
#pragma unroll
            for (int u = 0; u < WB; u++)
                load(u);
        else
#pragma unroll
            for (int u = 0; u < WB; u++)
                if (s0 + u * SKIP < steps)
                    load(u);
    };
    auto store_weights = [&](int s0) {
#pragma unroll
        for (int u = 0; u < WB; u++)
            if (s0 + u * SKIP < steps)
            {
                if constexpr (RAGGED)
                {
                    if (__any(wfix[u] >> 8))
                        wv[u] = drop_front(wv[u], wfix[u] >> 8);
                    wv[u] = keep_bytes(wv[u], wfix[u] & 255);
                }
                else if (!(w_oc < a.OC && 4 * (s0 + u * SKIP) + q < chunks))
                    wv[u] = v4i{ 0, 0, 0, 0 };
                sum_w += dot4_ones(wv[u]);
                *reinterpret_cast<v4i*>(wl + ((s0 + u * SKIP) * CT + ct_w) * 1024 + lane * 16) = wv[u];
            }
    };
    load_weights(wave / CT);
    const int bias = tid < 16 * CT && oc0 + tid < a.OC ? a.bias[a.bias_len == 1 ? 0 : oc0 + tid] : 0;
    for (int c = tid; c < 4 * steps; c += 256)
    {
        v2i e = { 0, kTconvDead };
        if (c < chunks)
        {
            const int tap = (int)fdiv((uint32_t)c, a.div_pieces), piece = c - tap * a.pieces;
            const int ty = row_of(tap), tx = tap - ty * taps_x;
            e.x = piece * 16 - (ty * a.IW + tx) * a.IC;
            e.y = (1 << ty) | (1 << (13 + tx));
        }
        tab_chunk[c] = e;
    }
    __syncthreads();

    // ---- pixels ---------------------------------------------------------------------------------------------------------
    const int first_pt = grp * 4 + wave, pt_step = a.groups * 4;
    const v2i* chunk_q = tab_chunk + q;
    const uint8_t* wf  = wl + lane * 16;
    int pix_off = 0, miss = -1;    // offset of the window's first tap; a zero bit per tap row and column inside the image
    bool edge = false;             // RAGGED: the tensor may end inside the 16 bytes of a lane of this tile
    int out_pix = 0;               // the lane's pixel in the result, -1: none
    v4i xv[DEPTH];
    auto request = [&](int d, int s, auto careful) {
        const v2i e        = chunk_q[4 * s];
        const bool inside  = (e.y & miss) == 0;
        const int off      = pix_off + e.x;
        const uint8_t* src = inside ? a.in + (uint32_t)off : a.page;
        if constexpr (!RAGGED)
            xv[d] = *reinterpret_cast<const v4i*>(src);
        else if constexpr (!decltype(careful)::value)
            xv[d] = load16(src);
        else
        {
            const int past = inside && off > a.in_last ? off - a.in_last : 0;
            xv[d]          = drop_front(load16(src - past), past);
        }
    };
    auto enter_tile = [&](int pt) {
        int p = pt * 16 + l16;
        p     = p < a.P ? p : a.P - 1;
        const int r = (int)fdiv((uint32_t)p, a.div_ow), x = p - r * (int)a.div_ow.d, n = (int)fdiv((uint32_t)r, a.div_oh), y = r - n * (int)a.div_oh.d;
        const int y0 = y + base_y, x0 = x + base_x;
        pix_off      = ((n * a.IH + y0) * a.IW + x0) * a.IC;
        // (classes are as large as the largest of them: a pixel may lie past the last row or column)
        out_pix      = pt * 16 + l16 < a.P && y * a.sy + cy < a.OH && x * a.sx + cx < a.OW ? (n * a.OH + y * a.sy + cy) * a.OW + x * a.sx + cx : -1;
        int in_bits  = 0;
        for (int k = 0; k < taps_y; k++)
            in_bits |= ((unsigned)(y0 - k) < (unsigned)a.IH ? 1 : 0) << k;
        for (int k = 0; k < taps_x; k++)
            in_bits |= ((unsigned)(x0 - k) < (unsigned)a.IW ? 1 : 0) << (13 + k);
        miss = ~in_bits;
        if constexpr (RAGGED)
            edge = __any(pix_off > a.edge_off);
        auto first_steps = [&](auto careful) {
#pragma unroll
            for (int d = 0; d < DEPTH; d++)
                if (d < steps)
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
    for (int s0 = wave / CT + WB * SKIP; s0 < steps; s0 += WB * SKIP)
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
        int sum = 0;
#pragma unroll
        for (int k = 0; k < 4 / CT; k++)
            sum += tab_part[k * (16 * CT) + tid];
        tab_base[tid] = bias - a.za * sum;
    }
    __syncthreads();

    for (int pt = first_pt; pt < a.n_pt; pt += pt_step)
    {
        if (pt != first_pt)
            enter_tile(pt);
        v4i acc[CT];
#pragma unroll
        for (int t = 0; t < CT; t++)
        {
            const int b = tab_base[16 * t + l16];
            acc[t]      = v4i{ b, b, b, b };
        }
        auto consume = [&](int d, int s) {
#pragma unroll
            for (int t = 0; t < CT; t++)
                acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(xv[d], *reinterpret_cast<const v4i*>(wf + (s * CT + t) * 1024), acc[t], 0, 0, 0);
        };
        auto walk = [&](auto careful) {
            int s = 0;
            for (; s + 2 * DEPTH <= steps; s += DEPTH)    // (whole groups with whole groups behind: no test)
#pragma unroll
                for (int d = 0; d < DEPTH; d++)
                {
                    consume(d, s + d);
                    request(d, s + d + DEPTH, careful);
                }
            for (; s < steps; s += DEPTH)
#pragma unroll
                for (int d = 0; d < DEPTH; d++)
                    if (s + d < steps)
                    {
                        consume(d, s + d);
                        if (s + d + DEPTH < steps)
                            request(d, s + d + DEPTH, careful);
                    }
        };
        if (RAGGED && edge)
            walk(std::true_type{});
        else
            walk(std::false_type{});

#pragma unroll
        for (int i = 0; i < 4; i++)
        {
            const int pix    = __shfl(out_pix, 4 * q + i);
            const int64_t at = (int64_t)pix * a.OC + oc0 + l16;
            if (pix >= 0)
#pragma unroll
                for (int t = 0; t < CT; t++)
                    if (oc0 + 16 * t + l16 < a.OC)
                        a.out[at + 16 * t] = acc[t][i];
        }
    }
}

// Channel tiles of a workgroup, 0: none that fits.  Few of them make many short workgroups, many share a pixel's loads: us 1 / 2 / 4 tiles, 3x3 stride 2 on
// (class pixels): [615,82]->112 6.1 / 6.5 / 8.0, [1196,160]->64 5.6 / 5.8 / 7.1, [1512,24]->240 6.7 / 5.7 / 6.0, 4x4 [1640,24]->248 7.7 / 6.3 / 6.4, 2x2
// [4536,56]->160 8.4 / 7.2 / 6.8, [4465,48]->96 6.4 / 5.7 / 5.8.
static int tconv_form(int64_t oc, int64_t n_pt, int64_t steps, int64_t classes)
{
    int best    = 0;
    double most = 1e30;
    for (int ct = 1; ct <= 4; ct *= 2)
    {
        if (steps * (ct * 1024 + 32) > 149 * 1024 || (ct > 1 && 8 * ct >= oc))
            continue;
        const int64_t rounds = ((n_pt + 3) / 4 * ((oc + 16 * ct - 1) / (16 * ct)) * classes + 255) / 256;
        const double us      = 0.03 * (double)(steps * ct) + (double)rounds * ((double)steps * (0.05 + 0.03 * ct) + 0.15 * ct);
        if (us < most)
            best = ct, most = us;
    }
    return best;
}

template <int CT, bool RAGGED>
static bool launch_tconv(hipStream_t st, TconvArgs& a)
{
    static_assert(sizeof(TconvArgs) <= 256, "see there");
    const int64_t lds = tconv_lds<CT>(a.steps);
    constexpr auto kern = tconv_taps_kernel<CT, RAGGED>;
    if (lds > 65536 && !ensure_dynamic_lds<kern>((size_t)lds))
        return false;
    // as many workgroups as the chip holds, for each channel block and class
    const int64_t units = (int64_t)((a.OC + 16 * CT - 1) / (16 * CT)) * a.classes, rounds = (a.n_pt + 3) / 4;
    const int64_t held = lds > 80 * 1024 ? 1 : (lds > 53 * 1024 ? 2 : (lds > 40 * 1024 ? 3 : 4)), most = (256 * held + units - 1) / units;
    const int64_t each = (rounds + most - 1) / most;
    a.groups           = (int32_t)((rounds + each - 1) / each);
    if (a.groups * units > INT32_MAX || !fastdiv_exact_up_to((uint64_t)a.groups * units, (uint32_t)a.groups) || !fastdiv_exact_up_to((uint64_t)units, (uint32_t)a.classes))
        return false;
    a.div_groups = make_fastdiv((uint32_t)a.groups);
    hipLaunchKernelGGL(kern, dim3((unsigned)(a.groups * units)), dim3(256), (size_t)lds, st, a);
    return true;
}

// page: 16 bytes of input_zp.  nullptr: not this form's
const char* launch_tconv_taps(hipStream_t st, const tmi_tconv_desc_t& d, const void* in, const void* w, const void* bias, int32_t in_zp, void* out, const void* page)
{
    const int sy = d.stride[0], sx = d.stride[1];
    if (d.in_dtype != TMI_INT8 || sy < 1 || sx < 1 || sy > kTconvStrides || sx > kTconvStrides || sy * sx < 2 || d.KH < sy || d.KW < sx || d.KH > 13 * sy ||
        d.KW > 13 * sx || (((uintptr_t)out | (uintptr_t)bias) & 3))
        return nullptr;
    const int64_t rows = (d.OH + sy - 1) / sy, cols = (d.OW + sx - 1) / sx, P = d.N * rows * cols, pieces = (d.IC + 15) / 16;
    const int64_t in_bytes = (int64_t)d.N * d.IH * d.IW * d.IC, w_bytes = (int64_t)d.OC * d.KH * d.KW * d.IC;
    const int64_t taps_y = (d.KH + sy - 1) / sy, taps_x = (d.KW + sx - 1) / sx, chunks = taps_y * taps_x * pieces;
    if (taps_y > 13 || taps_x > 13 || chunks > 4096 || P < 1 || P > (1 << 29) || P * sy * sx > INT32_MAX || in_bytes < 16 || w_bytes < 16 ||
        in_bytes > (1 << 30) || w_bytes > (1 << 30))
        return nullptr;
    TconvArgs a{};
    auto axis = [&](TconvAxis& x, int s, int k, int pad) {
        int64_t far = 0;    // how far a window begins from the class's pixel
        for (int c = 0; c < s; c++)
        {
            const int first = ((c - pad) % s + s) % s, taps = first < k ? (k - first + s - 1) / s : 0, base = (c - pad - first) / s;
            x.first[c] = (int8_t)first, x.taps[c] = (int8_t)taps, x.base[c] = (int16_t)base;
            far = taps < 1 ? INT32_MAX : std::max<int64_t>(far, std::abs((int64_t)base) + taps);
        }
        return far;
    };
    const int64_t far_y = axis(a.y, sy, d.KH, d.out_pad[0]), far_x = axis(a.x, sx, d.KW, d.out_pad[2]);
    if (far_y > 32000 || far_x > 32000 || in_bytes + ((far_y + rows) * d.IW + far_x + cols) * d.IC > INT32_MAX)
        return nullptr;
    a.in = (const uint8_t*)in, a.w = (const uint8_t*)w, a.bias = (const int32_t*)bias, a.out = (int32_t*)out, a.page = (const uint8_t*)page;
    a.P = (int32_t)P, a.OC = d.OC, a.OH = d.OH, a.OW = d.OW, a.IH = d.IH, a.IW = d.IW, a.KH = d.KH, a.KW = d.KW, a.sy = sy, a.sx = sx;
    a.IC = d.IC, a.pieces = (int32_t)pieces, a.steps = (int32_t)((chunks + 3) / 4), a.bias_len = d.bias_len, a.n_pt = (int32_t)((P + 15) / 16);
    a.classes = sy * sx, a.za = in_zp;
    a.in_last = (int32_t)(in_bytes - 16), a.w_last = (int32_t)(w_bytes - 16), a.edge_off = (int32_t)(in_bytes - 16 - (pieces - 1) * 16);
    a.div_ow = make_fastdiv((uint32_t)cols), a.div_oh = make_fastdiv((uint32_t)rows);
    a.div_pieces = make_fastdiv((uint32_t)pieces), a.div_classes = make_fastdiv((uint32_t)a.classes), a.div_sx = make_fastdiv((uint32_t)sx);
    for (int c = 0; c < sx; c++)
        a.taps_x_magic[c] = a.x.taps[c] == 1 ? 0 : (uint16_t)(65536 / a.x.taps[c] + 1);
    if (!fastdiv_exact_up_to((uint64_t)P, a.div_ow.d) || !fastdiv_exact_up_to((uint64_t)P / a.div_ow.d, a.div_oh.d) ||
        !fastdiv_exact_up_to((uint64_t)chunks, (uint32_t)pieces))
        return nullptr;
    const bool ragged = d.IC % 16 != 0 || ((((uintptr_t)in | (uintptr_t)w) & 15) != 0);
    bool ok           = false;
    switch (tconv_form(d.OC, a.n_pt, a.steps, a.classes))
    {
        case 1: ok = ragged ? launch_tconv<1, true>(st, a) : launch_tconv<1, false>(st, a); break;
        case 2: ok = ragged ? launch_tconv<2, true>(st, a) : launch_tconv<2, false>(st, a); break;
        case 4: ok = ragged ? launch_tconv<4, true>(st, a) : launch_tconv<4, false>(st, a); break;
        default: break;
    }
    return ok ? "transpose_conv2d_taps_i8" : nullptr;
}

}    // namespace tmi
