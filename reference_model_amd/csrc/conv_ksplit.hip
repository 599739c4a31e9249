// Small int8 CONV2D layers with taps and a long reduction (3x3 over 128 ... 512 channels on images of 14 x 14 or 7 x 7
// pixels: the last stages of a classification network), with or without the fused RESCALE (+ CLAMP).
//
//   out[n][oy][ox][oc] = sum_{ky,kx,ic} (in[n][oy*sy - pt + ky*dy][ox*sx - pl + kx*dx][ic] - input_zp) * w[oc][ky][kx][ic]
//                        + bias[oc]                                                     (tensor_ops.cpp:828-882)
//
// Such a layer has few output tiles (8 x 14 x 14 pixels x 256 channels: 26 tiles of 128 x 128) and K = 2304 ... 4608, so a
// kernel that gives a workgroup a large tile keeps a tenth of the chip busy.  Here a workgroup of NW waves (4, 8 or 16) owns a
// tile of 32 output channels x 32 pixels and splits the K steps (ky, kx, 32 channels) between its waves; both operands go
// straight from global memory into the registers the matrix instruction reads - the weight rows are K-contiguous as they
// lie, a pixel fragment is 16 bytes of the input pixel under the step's tap, or of the context's page of input_zp bytes
// where that tap falls outside the image - with every load of the tile in flight at once.  Each wave's accumulators start
// from its share of bias - input_zp * sum(w); the partial tiles meet in LDS and the first four waves requantise and store
// a quarter of the tile each (4 consecutive channels per lane).
//
// weight_zp must be 0, IC a multiple of 32, OC a multiple of 8, and K at most 160 steps (16 waves of 10).
//
// Two more forms below take their operands through LDS: 3 x 3 taps on 256, 384 or 512 channels, and 1 x 1 on 512 ... 2048.
#include "tmi_mfma.h"

namespace tmi
{

struct ConvSplitArgs
{
    const uint8_t* in;
    const int8_t* w;
    const int32_t* bias;
    const uint8_t* pad_page;    // 64 bytes of input_zp
    void* out;
    uint32_t* flag_word;
    RescaleParams rp;
    int32_t P, IC, OC;    // output pixels (N * OH * OW), input and output channels
    int32_t IH, IW, OH, OW, KW;
    int32_t sy, sx, dy, dx, pad_top, pad_left;
    int32_t za, bias_len;
    int32_t out_kind;     // 0: int32 accumulators, 1: int8 through the RESCALE, 2: int16 through the RESCALE
    int32_t n_oct, n_pt, n_groups;
    int32_t steps;        // K steps in all = taps * IC / 32
    int32_t spt;          // K steps per tap = IC / 32
    int32_t ksw;          // K steps per wave
    FastDiv div_oct, div_spt, div_kw, div_ow, div_oh;
};

// apply_scale_32 + output_zp + clip (+ CLAMP) from the multiplier and the validated shift (see pointwise.hip)
__device__ __forceinline__ int32_t split_rescale_from_shift(int32_t v, int32_t m, int32_t s, bool double_round, int32_t out_zp,
                                                            int32_t lo, int32_t hi, uint32_t& flags)
{
    if (s <= 31)
    {
        const int32_t high = 1 << (s - 1);
        if (v < -high || v >= high)
            flags |= TMI_FLAG_SCALE_VALUE;
    }
    int64_t round = int64_t(1) << (s - 1);
    if (double_round && s > 31)
        round += v >= 0 ? (int64_t(1) << 30) : -(int64_t(1) << 30);
    const int64_t p = (int64_t)v * (int64_t)m + round;
    int32_t r       = (int32_t)(p >> s) + out_zp;
    r               = r < lo ? lo : r;
    return r > hi ? hi : r;
}

// The requantisation constants of the 32 channels from oct * 32 on, by one wave: the high-word form's, multiplier and shift for
// the general form, and the form word.
template <typename A>
__device__ __forceinline__ void split_tables(const A& a, int oct, int lane, int32_t m_raw, int32_t s_raw, HighWordScale* tab_hw, v2i* tab_ms, int32_t* form_word,
                                             uint32_t& flags)
{
    const int li  = lane & 31;
    const int oc  = oct * 32 + li;
    const bool ok = oc < a.OC;
    const int32_t s_first = __builtin_amdgcn_readfirstlane(s_raw);
    const ChannelScale cs = make_channel_scale(ok ? m_raw : 0, ok ? s_raw : s_first, a.rp.double_round != 0, flags);
    const int s_min       = a.rp.double_round ? 33 : 32;
    // bit 0: the high-word form for all 32 channels; bit 1: no sign test in it (a negative value is clamped away
    // with either rounding term: the result's lower limit is at or above output_zp and no multiplier is negative)
    const int form = (__all(cs.s >= s_min && cs.s <= zp_fold_max_shift(a.rp.out_zp)) ? 1 : 0) |
                     (a.rp.lo >= a.rp.out_zp && __all(cs.m >= 0) ? 2 : 0);
    if (lane < 32)
    {
        tab_ms[li] = v2i{ cs.m, cs.s };
        tab_hw[li] = make_high_word_scale(cs, a.rp.out_zp);
    }
    if (lane == 0)
        *form_word = form;
}

// Requantises and stores the results of channels c0 ... c0 + 3 of the tile for one pixel; `at` is their element offset.
template <typename A>
__device__ __forceinline__ void split_store(const A& a, v4i sum, int c0, size_t at, bool store, int form, const HighWordScale* tab_hw,
                                            const v2i* tab_ms, uint32_t& flags)
{
    if (a.out_kind == 0)
    {
        if (store)
            *reinterpret_cast<v4i*>(reinterpret_cast<int32_t*>(a.out) + at) = sum;
        return;
    }
    const int32_t v_lo = a.rp.lo, v_hi = a.rp.hi;
    int32_t r[4];
#pragma unroll
    for (int j = 0; j < 4; j++)
    {
        const int c = c0 + j;
        if (form & 1)
            r[j] = (a.rp.double_round && !(form & 2)) ? clamp_med3(high_word_rescale64<true>(sum[j], tab_hw[c]), v_lo, v_hi)
                                                      : clamp_med3(high_word_rescale64<false>(sum[j], tab_hw[c]), v_lo, v_hi);
        else
        {
            uint32_t f   = 0;
            const v2i ms = tab_ms[c];
            r[j]         = split_rescale_from_shift(sum[j], ms.x, ms.y, a.rp.double_round != 0, a.rp.out_zp, v_lo, v_hi, f);
            flags |= store ? f : 0u;
        }
    }
    if (a.out_kind == 1)
    {
        const int lo2 = __builtin_amdgcn_perm(r[1], r[0], 0x0c0c0400);
        const int hi2 = __builtin_amdgcn_perm(r[3], r[2], 0x04000c0c);
        if (store)
            *reinterpret_cast<int*>(reinterpret_cast<int8_t*>(a.out) + at) = lo2 | hi2;
    }
    else if (store)
        *reinterpret_cast<v2i*>(reinterpret_cast<int16_t*>(a.out) + at) =
            v2i{ (r[0] & 0xffff) | ((r[1] & 0xffff) << 16), (r[2] & 0xffff) | ((r[3] & 0xffff) << 16) };
}

template <int KS, int NW, bool ZA>
__global__ __launch_bounds__(NW * 64, NW == 16 ? 4 : 2) void conv_ksplit_i8_kernel(ConvSplitArgs a)
{
    // [NW waves x 4 quarters x 64 lanes x 16 bytes][32 x HighWordScale][32 x (m, s)][NW waves x 32 start values][form]
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 31, lh = lane >> 5;
    const uint32_t g = blockIdx.x;
    const int q = (int)fdiv(g, a.div_oct), oct = (int)g - q * a.n_oct;
    const int G = a.n_groups;
    HighWordScale* tab_hw = reinterpret_cast<HighWordScale*>(lds + NW * 4096);
    v2i* tab_ms           = reinterpret_cast<v2i*>(tab_hw + 32);
    int32_t* wave_start   = reinterpret_cast<int32_t*>(tab_ms + 32) + wave * 32;
    int32_t* form_word    = reinterpret_cast<int32_t*>(tab_ms + 32) + NW * 32;
    const int ksw   = a.ksw;
    const int step0 = wave * ksw;    // first K step of the wave's share
    const int nvalid = a.steps - step0 < ksw ? (a.steps - step0 > 0 ? a.steps - step0 : 0) : ksw;    // steps of the share that exist
    const int kbytes = a.steps * 32; // bytes of a weight row

    // ---- pixel fragments: lane (li, lh) holds bytes [16 lh, + 16) of the 32 channels of step s under the step's tap ------
    auto load_pixels = [&](v4i (&fb)[KS], int pt) {
        int p = pt * 32 + li;
        p     = p < a.P ? p : a.P - 1;    // a pixel past the end: the last one again, never stored
        const int row = (int)fdiv((uint32_t)p, a.div_ow);    // n * OH + oy
        const int ox  = p - row * a.OW;
        const int n   = (int)fdiv((uint32_t)row, a.div_oh);
        const int oy  = row - n * a.OH;
        const int iy0 = oy * a.sy - a.pad_top, ix0 = ox * a.sx - a.pad_left;
        const uint8_t* img = a.in + (size_t)n * a.IH * a.IW * a.IC;
        // A wave with one wave on its SIMD issues an instruction every eight clocks or so, so what a step costs is its
        // instruction count: the tap's pixel is worked out once per tap (the wave's first step with divisions, the following
        // taps by stepping: scalar work, the same for all lanes) and a step inside a tap is a load and an addition.
        int tap = (int)fdiv((uint32_t)step0, a.div_spt);
        int cs  = step0 - tap * a.spt;    // which 32 channels of the tap
        int ky  = (int)fdiv((uint32_t)tap, a.div_kw);
        int kx  = tap - ky * a.KW;
        const uint8_t* cur = nullptr;
        uint32_t inc       = 0;
        auto at_tap        = [&]() {
            const int iy = iy0 + ky * a.dy, ix = ix0 + kx * a.dx;
            const bool inside  = (unsigned)iy < (unsigned)a.IH && (unsigned)ix < (unsigned)a.IW;
            const uint32_t off = (uint32_t)((iy * a.IW + ix) * a.IC + cs * 32 + 16 * lh);    // one image is below 2^31 bytes
            cur                = inside ? img + off : a.pad_page + 16 * lh;
            inc                = inside ? 32u : 0u;    // outside the image every step reads the page of input_zp bytes
        };
        at_tap();
#pragma unroll
        for (int s = 0; s < KS; s++)
        {
            if (s < nvalid)    // (a test per step, not a loop exit: the register array keeps constant indices)
            {
                fb[s] = *reinterpret_cast<const v4i*>(cur);
                cur += inc;
                cs++;
                if (cs == a.spt)
                {
                    cs = 0, kx++;
                    if (kx == a.KW)
                        kx = 0, ky++;
                    at_tap();
                }
            }
        }
    };
    v4i fb[KS];
    load_pixels(fb, q);

    // ---- weight fragments: MFMA operand row li is channel 16 * ((li >> 2) & 1) + 4 * (li >> 3) + (li & 3) of the tile -------
    const int wr = 4 * (li & 4) + ((li >> 1) & 12) + (li & 3);
    const int ch = oct * 32 + wr;
    v4i fa[KS];
    {
        // one 32-bit offset per lane; the steps are the instruction's offset field (the weights are below 2^31 bytes)
        const uint32_t woff = (uint32_t)((ch < a.OC ? ch : a.OC - 1) * kbytes + step0 * 32 + 16 * lh);
#pragma unroll
        for (int s = 0; s < KS; s++)
        {
            if (s < nvalid)
                fa[s] = *reinterpret_cast<const v4i*>(a.w + woff + s * 32);
        }
    }
    // (rows past OC are zeroed further down, once, so that no load is waited for before the next one is issued)
    uint32_t flags = 0;
    if (wave == 0)
    {
        if (a.rp.enabled)    // the first wave derives the constants of the tile's 32 channels for all
        {
            const int occ = oct * 32 + li < a.OC ? oct * 32 + li : oct * 32;
            split_tables(a, oct, lane, load_multiplier(a.rp, occ), load_shift(a.rp, occ), tab_hw, tab_ms, form_word, flags);
        }
    }
    if (ch >= a.OC)
    {
#pragma unroll
        for (int s = 0; s < KS; s++)
            fa[s] = v4i{ 0, 0, 0, 0 };
    }
    {
        int32_t b = wave == 0 ? a.bias[a.bias_len == 1 ? 0 : (ch < a.OC ? ch : oct * 32)] : 0;
        if constexpr (ZA)
        {
            int sum = 0;
#pragma unroll
            for (int s = 0; s < KS; s++)
                if (s < nvalid)
                    sum += dot4_ones(fa[s]);
            sum += __builtin_amdgcn_ds_bpermute((lane ^ 32) * 4, sum);
            b = (int32_t)((uint32_t)b - (uint32_t)a.za * (uint32_t)sum);
        }
        if (lh == 0)
            wave_start[wr] = ch < a.OC ? b : 0;
        __builtin_amdgcn_wave_barrier();    // the wave's own LDS accesses complete in order
    }
    // (a tile's start values are read from the wave's table again for every tile: the registers are needed for the loads)
    auto start_values = [&]() {
        int first = 16 * lh;
        asm volatile("" : "+v"(first));    // (hidden from the compiler, which would otherwise keep them across the loop)
        v16i start;
#pragma unroll
        for (int gq = 0; gq < 4; gq++)
        {
            const v4i b4 = *reinterpret_cast<const v4i*>(wave_start + first + 4 * gq);
            start[4 * gq] = b4[0], start[4 * gq + 1] = b4[1], start[4 * gq + 2] = b4[2], start[4 * gq + 3] = b4[3];
        }
        return start;
    };
    const int oc_lane = oct * 32 + 16 * lh + 4 * (wave & 3);    // first of the 4 channels a lane of waves 0 .. 3 stores
    const bool ch_ok  = oc_lane < a.OC;                         // OC is a multiple of 8: the four are in or out together
    for (int pt = q; pt < a.n_pt; pt += G)
    {
        v16i acc = start_values();
#pragma unroll
        for (int s = 0; s < KS; s++)
            if (s < nvalid)
                acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[s], fb[s], acc, 0, 0, 0);
        if (pt + G < a.n_pt)
            load_pixels(fb, pt + G);    // in flight across the exchange and the requantisation
        // the partial tiles meet in LDS: [wave][quarter][lane] of 16 bytes
        if (pt != q)
            __syncthreads();    // every wave has read the tile before
#pragma unroll
        for (int gq = 0; gq < 4; gq++)
            *reinterpret_cast<v4i*>(lds + ((wave * 4 + gq) * 64 + lane) * 16) = v4i{ acc[4 * gq], acc[4 * gq + 1], acc[4 * gq + 2], acc[4 * gq + 3] };
        __syncthreads();    // also publishes the first wave's tables
        if (wave >= 4)
            continue;
        v4i sum = *reinterpret_cast<const v4i*>(lds + ((0 * 4 + wave) * 64 + lane) * 16);
#pragma unroll NW == 16 ? 5 : NW
        for (int w2 = 1; w2 < NW; w2++)
        {
            const v4i o = *reinterpret_cast<const v4i*>(lds + ((w2 * 4 + wave) * 64 + lane) * 16);
            sum.x += o.x, sum.y += o.y, sum.z += o.z, sum.w += o.w;
        }
        const int p      = pt * 32 + li;
        const bool store = p < a.P && ch_ok;
        const size_t at  = (size_t)(p < a.P ? p : 0) * a.OC + (ch_ok ? oc_lane : 0);
        split_store(a, sum, 16 * lh + 4 * wave, at, store, a.rp.enabled ? *form_word : 0, tab_hw, tab_ms, flags);
    }
    raise_flags(a.flag_word, flags);
}

// The same split for 3 x 3 taps on 256, 384 or 512 channels with both operands through the LDS: a workgroup of NW = IC / 32 waves owns 32 output channels
// x a block of TH x TW output pixels of one image (up to 32 * NPT of them); each wave has nine K steps, 288 bytes of every
// weight row.  Weights and input patch are read once, consecutive lanes on consecutive bytes, padding as input_zp bytes.
// What bounds the form above on these layers is its loads: a lane per row makes every load instruction touch 32 lines for 32
// bytes each, and the 70 ... 150 KB of a tile's weights leave the L1 before the next step wants the rest of the line.  Here a
// line is read by one instruction, a pixel once instead of nine times, and what is left is the chain of one workgroup: its
// arguments, one trip to memory, three barriers, the exchange.  us, graph replays, fused RESCALE, form above / this form:
// [8,14,14,256]->256 9.7 / 6.8, [8,28,28,256]->256 stride 2 9.8 / 8.0, [8,7,7,512]->512 11.5 / 8.1, [8,14,14,512]->512 stride 2
// 11.4 / 8.8, [1,14,14,256]->256 7.2 / 5.5, [8,14,14,384]->384 16.2 / 10.7, [16,14,14,256]->256 13.7 / 9.1, [16,7,7,512]->512
// 15.1 / 9.9; with 160, 192 and 320 channels the form above has fewer steps a wave and stays ahead ([8,14,14,160]->160 4.9 / 6.7,
// [8,28,28,192]->192 11.8 / 12.8, [8,14,14,320]->320 8.8 / 10.0).
struct ConvPatchSplitArgs
{
    const uint8_t* in;
    const int8_t* w;
    const int32_t* bias;
    const uint8_t* pad_page;    // 64 bytes of input_zp
    void* out;
    uint32_t* flag_word;
    RescaleParams rp;
    int32_t OC, IH, IW, OH, OW;
    int16_t sy, sx, dy, dx, pad_top, pad_left;
    int32_t bias_len, za;
    int32_t out_kind;     // as above
    int32_t n_blk, n_groups;
    int32_t TH;           // rows of a block (its columns: div_tw.d)
    int32_t chunks;       // 16-byte pieces of a patch
    FastDiv div_oct, div_bx, div_by, div_tw, div_pw;    // by channel tiles, blocks across and down an image, columns of a block, of its patch
};
static_assert(sizeof(ConvPatchSplitArgs) <= 256, "see SlabArgs in conv2d_slab.hip");

template <int NW, int NPT, bool ZA>
__global__ __launch_bounds__(NW * 64, (NW + 3) / 4) void conv_ksplit_patch_kernel(ConvPatchSplitArgs a)
{
    constexpr int KS = 9, IC = NW * 32, NT = NW * 64;
    constexpr int kPieces = 2 * KS, kRow = kPieces * 16 + 16;    // 16-byte pieces of a wave's share of a weight row; its pitch in LDS
    constexpr int CPP = IC / 16, kPitch = IC + 16;               // pieces of a pixel; its pitch: = 16 (mod 32), neighbours of a row in different banks
    // (a block's next row of pixels starts PW - TW pixels further on and meets the banks of the last: 1.6 and 1.5 conflict cycles an LDS
    // instruction measured on 14 x 14 x 256 and 7 x 7 x 512)
    constexpr int NC  = NW >= 14 ? 3 : 4;                        // pieces of the patch a lane has in flight
    // [32 x HighWordScale][32 x (m, s)][NW waves x 32 start values][form] and then the weights of all waves, later
    // [NPT x NW waves x 4 quarters x 64 lanes x 16 bytes][patch]
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    // Every argument the way to the first results needs, in a few wide scalar loads (left to the compiler: forty narrow ones, each
    // waited for where it is used)
    asm volatile("" ::"s"(a.in), "s"(a.w), "s"(a.bias), "s"(a.pad_page), "s"(a.rp.multiplier), "s"(a.rp.shift), "s"(a.OC), "s"(a.IH),
                 "s"(a.IW), "s"(*reinterpret_cast<const uint32_t*>(&a.sy)), "s"(*reinterpret_cast<const uint32_t*>(&a.dy)),
                 "s"(*reinterpret_cast<const uint32_t*>(&a.pad_top)), "s"(a.TH), "s"(a.chunks), "s"(a.div_oct.magic), "s"(a.div_oct.d),
                 "s"(a.div_bx.magic), "s"(a.div_bx.d), "s"(a.div_by.magic), "s"(a.div_by.d), "s"(a.div_tw.d), "s"(a.div_pw.magic),
                 "s"(a.div_pw.d));
    const int tid  = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 31, lh = lane >> 5;
    const uint32_t g = blockIdx.x;
    const int q = (int)fdiv(g, a.div_oct), oct = (int)g - q * (int)a.div_oct.d;
    HighWordScale* tab_hw = reinterpret_cast<HighWordScale*>(lds);
    v2i* tab_ms           = reinterpret_cast<v2i*>(tab_hw + 32);
    int32_t* wave_start   = reinterpret_cast<int32_t*>(tab_ms + 32) + wave * 32;
    int32_t* form_word    = reinterpret_cast<int32_t*>(tab_ms + 32) + NW * 32;
    uint8_t* exch         = reinterpret_cast<uint8_t*>(form_word + 4);
    uint8_t* patch        = exch + NPT * NW * 4096;
    const int TW = (int)a.div_tw.d, PW = (int)a.div_pw.d;
    // MFMA operand row li is channel 16 * ((li >> 2) & 1) + 4 * (li >> 3) + (li & 3) of the tile
    const int wr = 4 * (li & 4) + ((li >> 1) & 12) + (li & 3);
    const int ch = oct * 32 + wr;

    // ---- the first wave's constants, then the weights: the wave's bytes of all 32 rows (a row past OC: the last one again) ----
    int32_t b = 0, m_raw = 0, s_raw = 0;
    if (wave == 0)
    {
        b = a.bias[a.bias_len == 1 ? 0 : (ch < a.OC ? ch : oct * 32)];
        if (a.rp.enabled)
        {
            const int occ = oct * 32 + li < a.OC ? oct * 32 + li : oct * 32;
            m_raw = load_multiplier(a.rp, occ), s_raw = load_shift(a.rp, occ);
        }
    }
    v4i wb[KS];
#pragma unroll
    for (int i = 0; i < KS; i++)
    {
        const int r    = (i * 64 + lane) / kPieces, part = (i * 64 + lane) % kPieces;
        const int from = oct * 32 + r;
        const uint32_t off = mad_u24((uint32_t)(from < a.OC ? from : a.OC - 1), KS * IC, (uint32_t)(wave * KS * 32 + part * 16));
        wb[i] = *reinterpret_cast<const v4i*>(a.w + off);
    }

    // ---- the patch: pieces base + i * NT + tid (past the last one: that one again) -------------------------------------------
    int n = 0, by = 0, bx = 0;    // the block at hand
    auto decode = [&](int blk) {
        const int row = (int)fdiv((uint32_t)blk, a.div_bx);
        bx            = blk - row * (int)a.div_bx.d;
        n             = (int)fdiv((uint32_t)row, a.div_by);
        by            = row - n * (int)a.div_by.d;
    };
    v4i pb[NC];
    int put[NC];    // LDS byte offsets of the pieces
    auto fetch = [&](int base) {
        const int iy0 = by * a.TH * a.sy - a.pad_top, ix0 = bx * TW * a.sx - a.pad_left;
        const int img = n * a.IH;
#pragma unroll
        for (int i = 0; i < NC; i++)
        {
            if (base + i * NT < a.chunks)    // (the same for all lanes)
            {
                int c          = base + i * NT + tid;
                c              = c < a.chunks ? c : a.chunks - 1;
                const int px   = (int)((uint32_t)c / (uint32_t)CPP), part = c - px * CPP;
                const int py   = (int)__umulhi((uint32_t)px, a.div_pw.magic);    // (a patch is at least three pixels wide)
                const int iy = iy0 + py, ix = ix0 + px - py * PW;
                const bool inside  = (unsigned)iy < (unsigned)a.IH && (unsigned)ix < (unsigned)a.IW;
                const uint32_t off = (uint32_t)(((img + iy) * a.IW + ix) * IC + part * 16);    // the input is below 2^31 bytes
                const uint8_t* from = inside ? a.in + off : a.pad_page;
                pb[i]  = *reinterpret_cast<const v4i*>(from);
                put[i] = px * kPitch + part * 16;
            }
        }
    };
    auto place = [&](int base) {
#pragma unroll
        for (int i = 0; i < NC; i++)
            if (base + i * NT < a.chunks)
                *reinterpret_cast<v4i*>(patch + put[i]) = pb[i];
    };
    auto rest = [&]() {    // what one set of registers does not hold
        for (int base = NC * NT; base < a.chunks; base += NC * NT)
        {
            fetch(base);
            place(base);
        }
    };
    decode(q);
    fetch(0);
    asm volatile("" ::"s"(a.out), "s"(a.flag_word), "s"(a.rp.lo), "s"(a.rp.hi), "s"(a.OH), "s"(a.OW), "s"(a.out_kind), "s"(a.n_blk),
                 "s"(a.n_groups), "s"(a.za), "s"(a.div_tw.magic), "s"(a.rp.out_zp));
    // ---- where the wave's steps and the lane's pixels lie in the patch: the same for every block ----------------------------
    int step_at[KS];
    {
        constexpr int spt = NW;    // K steps of a tap
        const int down = a.dy * PW * kPitch, right = a.dx * kPitch;
#pragma unroll
        for (int s = 0; s < KS; s++)
        {
            const int step = wave * KS + s, tap = step / spt, ky = tap / 3;
            step_at[s]     = ky * down + (tap - 3 * ky) * right + (step - tap * spt) * 32;
        }
    }
    uint32_t pixel_at[NPT];
    int sty = 0, stx = 0;    // the pixel of the block whose results this lane stores
#pragma unroll
    for (int t = 0; t < NPT; t++)
    {
        int ty = (int)fdiv((uint32_t)(t * 32 + li), a.div_tw), tx = t * 32 + li - ty * TW;
        if (NPT == 1 || (wave >> 2) == t)
            sty = ty, stx = tx;
        if (ty >= a.TH)
            ty = 0, tx = 0;    // a slot the block does not use: its first pixel again, never stored
        pixel_at[t] = (uint32_t)((ty * a.sy * PW + tx * a.sx) * kPitch + 16 * lh);
    }
    // a lane stores a quarter (4 of 16 channels per half wave) of pixel tile wave / 4
    const int c0      = 16 * lh + 4 * (wave & 3);
    const int oc_lane = oct * 32 + c0;
    const bool ch_ok  = sty < a.TH && oc_lane < a.OC;    // OC is a multiple of 8: the four are in or out together

    // ---- the weights through the wave's own part of the LDS into fragments ---------------------------------------------------
    uint32_t flags = 0;
    v4i fa[KS];
    {
        uint8_t* own = exch + wave * 32 * kRow;
#pragma unroll
        for (int i = 0; i < KS; i++)
            *reinterpret_cast<v4i*>(own + (i * 64 + lane + (i * 64 + lane) / kPieces) * 16) = wb[i];
        __builtin_amdgcn_wave_barrier();    // the wave's own LDS accesses complete in order
#pragma unroll
        for (int s = 0; s < KS; s++)
            fa[s] = *reinterpret_cast<const v4i*>(own + wr * kRow + s * 32 + 16 * lh);
        if (wave == 0 && a.rp.enabled)
            split_tables(a, oct, lane, m_raw, s_raw, tab_hw, tab_ms, form_word, flags);
        if ((oct + 1) * 32 > a.OC)
        {
#pragma unroll
            for (int s = 0; s < KS; s++)
                fa[s] = ch < a.OC ? fa[s] : v4i{ 0, 0, 0, 0 };
        }
        if constexpr (ZA)
        {
            int sum = 0;
#pragma unroll
            for (int s = 0; s < KS; s++)
                sum += dot4_ones(fa[s]);
            sum += __builtin_amdgcn_ds_bpermute((lane ^ 32) * 4, sum);
            b = (int32_t)((uint32_t)b - (uint32_t)a.za * (uint32_t)sum);
        }
        if (lh == 0)
            wave_start[wr] = ch < a.OC ? b : 0;
    }
    __syncthreads();    // every wave has its weights: the patch and the partial tiles take their place
    place(0);
    rest();
    for (int blk = q; blk < a.n_blk; blk += a.n_groups)
    {
        const int out_n = n, out_y = by * a.TH + sty, out_x = bx * TW + stx;
        __syncthreads();    // the patch is complete (and the tables), the exchange area free
        v16i acc[NPT];
#pragma unroll
        for (int gq = 0; gq < 4; gq++)
        {
            const v4i b4 = *reinterpret_cast<const v4i*>(wave_start + 16 * lh + 4 * gq);
#pragma unroll
            for (int t = 0; t < NPT; t++)
                acc[t][4 * gq] = b4[0], acc[t][4 * gq + 1] = b4[1], acc[t][4 * gq + 2] = b4[2], acc[t][4 * gq + 3] = b4[3];
        }
#pragma unroll
        for (int s = 0; s < KS; s++)
#pragma unroll
            for (int t = 0; t < NPT; t++)
            {
                const v4i fb = *reinterpret_cast<const v4i*>(patch + (pixel_at[t] + (uint32_t)step_at[s]));
                acc[t]       = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[s], fb, acc[t], 0, 0, 0);
            }
#pragma unroll
        for (int t = 0; t < NPT; t++)
#pragma unroll
            for (int gq = 0; gq < 4; gq++)
                *reinterpret_cast<v4i*>(exch + (((t * NW + wave) * 4 + gq) * 64 + lane) * 16) =
                    v4i{ acc[t][4 * gq], acc[t][4 * gq + 1], acc[t][4 * gq + 2], acc[t][4 * gq + 3] };
        // (the stores above have read the matrix instructions' results: no load can land in operands still being read)
        __builtin_amdgcn_sched_barrier(0);
        const bool more = blk + a.n_groups < a.n_blk;
        if (more)
        {
            decode(blk + a.n_groups);
            fetch(0);    // in flight across the barrier
        }
        __syncthreads();    // the partial tiles are there, and every wave has read the patch
        if (more)
        {
            place(0);
            rest();
        }
        if (wave >= 4 * NPT)
            continue;
        const uint8_t* part = exch + ((NPT == 1 ? 0 : (wave >> 2) * NW * 4) + (wave & 3)) * 1024 + lane * 16;
        v4i sum = *reinterpret_cast<const v4i*>(part);
#pragma unroll NW > 8 ? 5 : NW
        for (int w2 = 1; w2 < NW; w2++)
        {
            const v4i o = *reinterpret_cast<const v4i*>(part + w2 * 4096);
            sum.x += o.x, sum.y += o.y, sum.z += o.z, sum.w += o.w;
        }
        const bool store = ch_ok && out_y < a.OH && out_x < a.OW;
        const size_t at  = store ? (size_t)(uint32_t)(((out_n * a.OH + out_y) * a.OW + out_x) * a.OC + oc_lane) : 0;
        split_store(a, sum, c0, at, store, a.rp.enabled ? *form_word : 0, tab_hw, tab_ms, flags);
    }
    raise_flags(a.flag_word, flags);
}

// 1 x 1 layers with few tiles and a long reduction (the classifier of a network, the last projections): a workgroup of eight
// waves per 32 channels x 32 pixels, an eighth of K to a wave.  Both operands come in whole lines, KS loads of each in flight,
// and turn into fragments in the wave's own part of the LDS, which then takes its partial tile: one barrier in all.  What bounds
// it is that chain: arguments, one trip to memory, LDS, the exchange.  The K-split pointwise form (a lane per row, as above) and
// this one, us, graph replays, fused RESCALE: [8,7,7,2048]->512 8.0 / 4.8, [8,1,1,2048]->1000 6.8 / 4.4, [1,1,1,1280]->1000 5.8 /
// 3.8, [64,1,1,2048]->4096 8.0 / 4.8, [8,14,14,2048]->256 (392 tiles) 11.3 / 7.6, [32,7,7,2048]->512 (784) 15.2 / 13.6, [8,7,7,512]->2048
// (832) 7.0 / 6.0; more tiles than that were not measured and stay where weights are kept over several tiles.
struct PointSplitArgs
{
    const uint8_t* in;
    const int8_t* w;
    const int32_t* bias;
    void* out;
    uint32_t* flag_word;
    RescaleParams rp;
    int32_t P, OC;    // pixels, output channels
    int32_t za, bias_len;
    int32_t out_kind;
    FastDiv div_oct;
};

template <int KS, bool ZA>
__global__ __launch_bounds__(512, 2) void point_split_kernel(PointSplitArgs a)
{
    constexpr int NW = 8, IC = NW * KS * 32, kPieces = 2 * KS, kRow = kPieces * 16 + 16;
    constexpr int kOwn = 2 * 32 * kRow > 4096 ? 2 * 32 * kRow : 4096;    // a wave's weights and pixels, later its partial tile
    // [32 x HighWordScale][32 x (m, s)][NW waves x 32 start values][form] and the waves' parts
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    asm volatile("" ::"s"(a.in), "s"(a.w), "s"(a.bias), "s"(a.out), "s"(a.flag_word), "s"(a.rp.multiplier), "s"(a.rp.shift), "s"(a.rp.out_zp),
                 "s"(a.rp.lo), "s"(a.rp.hi), "s"(a.P), "s"(a.OC), "s"(a.za), "s"(a.bias_len), "s"(a.out_kind), "s"(a.div_oct.magic), "s"(a.div_oct.d));
    const int tid  = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 31, lh = lane >> 5;
    const uint32_t g = blockIdx.x;
    const int pt = (int)fdiv(g, a.div_oct), oct = (int)g - pt * (int)a.div_oct.d;
    HighWordScale* tab_hw = reinterpret_cast<HighWordScale*>(lds);
    v2i* tab_ms           = reinterpret_cast<v2i*>(tab_hw + 32);
    int32_t* wave_start   = reinterpret_cast<int32_t*>(tab_ms + 32) + wave * 32;
    int32_t* form_word    = reinterpret_cast<int32_t*>(tab_ms + 32) + NW * 32;
    uint8_t* parts        = reinterpret_cast<uint8_t*>(form_word + 4);
    uint8_t* own          = parts + wave * kOwn;
    const int wr = 4 * (li & 4) + ((li >> 1) & 12) + (li & 3);
    const int ch = oct * 32 + wr;
    int32_t b = 0, m_raw = 0, s_raw = 0;
    if (wave == 0)
    {
        b = a.bias[a.bias_len == 1 ? 0 : (ch < a.OC ? ch : oct * 32)];
        if (a.rp.enabled)
        {
            const int occ = oct * 32 + li < a.OC ? oct * 32 + li : oct * 32;
            m_raw = load_multiplier(a.rp, occ), s_raw = load_shift(a.rp, occ);
        }
    }
    v4i wb[KS], pb[KS];
#pragma unroll
    for (int i = 0; i < KS; i++)
    {
        const int r   = (i * 64 + lane) / kPieces, part = (i * 64 + lane) % kPieces;
        const int row = oct * 32 + r, pix = pt * 32 + r;    // past the end: the last one again, zeroed or never stored
        const uint32_t col = (uint32_t)(wave * KS * 32 + part * 16);
        wb[i] = *reinterpret_cast<const v4i*>(a.w + ((uint32_t)(row < a.OC ? row : a.OC - 1) * (uint32_t)IC + col));
        pb[i] = *reinterpret_cast<const v4i*>(a.in + ((uint32_t)(pix < a.P ? pix : a.P - 1) * (uint32_t)IC + col));
    }
#pragma unroll
    for (int i = 0; i < KS; i++)
    {
        const int at = (i * 64 + lane + (i * 64 + lane) / kPieces) * 16;
        *reinterpret_cast<v4i*>(own + at)             = wb[i];
        *reinterpret_cast<v4i*>(own + 32 * kRow + at) = pb[i];
    }
    __builtin_amdgcn_wave_barrier();    // the wave's own LDS accesses complete in order
    v4i fa[KS], fb[KS];
#pragma unroll
    for (int s = 0; s < KS; s++)
    {
        fa[s] = *reinterpret_cast<const v4i*>(own + wr * kRow + s * 32 + 16 * lh);
        fb[s] = *reinterpret_cast<const v4i*>(own + 32 * kRow + li * kRow + s * 32 + 16 * lh);
    }
    uint32_t flags = 0;
    if (wave == 0 && a.rp.enabled)
        split_tables(a, oct, lane, m_raw, s_raw, tab_hw, tab_ms, form_word, flags);
    if ((oct + 1) * 32 > a.OC)
    {
#pragma unroll
        for (int s = 0; s < KS; s++)
            fa[s] = ch < a.OC ? fa[s] : v4i{ 0, 0, 0, 0 };
    }
    if constexpr (ZA)
    {
        int sum = 0;
#pragma unroll
        for (int s = 0; s < KS; s++)
            sum += dot4_ones(fa[s]);
        sum += __builtin_amdgcn_ds_bpermute((lane ^ 32) * 4, sum);
        b = (int32_t)((uint32_t)b - (uint32_t)a.za * (uint32_t)sum);
    }
    if (lh == 0)
        wave_start[wr] = ch < a.OC ? b : 0;
    __builtin_amdgcn_wave_barrier();
    v16i acc;
#pragma unroll
    for (int gq = 0; gq < 4; gq++)
    {
        const v4i b4 = *reinterpret_cast<const v4i*>(wave_start + 16 * lh + 4 * gq);
        acc[4 * gq] = b4[0], acc[4 * gq + 1] = b4[1], acc[4 * gq + 2] = b4[2], acc[4 * gq + 3] = b4[3];
    }
#pragma unroll
    for (int s = 0; s < KS; s++)
        acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[s], fb[s], acc, 0, 0, 0);
#pragma unroll
    for (int gq = 0; gq < 4; gq++)
        *reinterpret_cast<v4i*>(own + (gq * 64 + lane) * 16) = v4i{ acc[4 * gq], acc[4 * gq + 1], acc[4 * gq + 2], acc[4 * gq + 3] };
    __syncthreads();    // the partial tiles and the tables are there
    if (wave < 4)
    {
        const uint8_t* part = parts + wave * 1024 + lane * 16;
        v4i sum = *reinterpret_cast<const v4i*>(part);
#pragma unroll
        for (int w2 = 1; w2 < NW; w2++)
        {
            const v4i o = *reinterpret_cast<const v4i*>(part + w2 * kOwn);
            sum.x += o.x, sum.y += o.y, sum.z += o.z, sum.w += o.w;
        }
        const int p = pt * 32 + li, c0 = 16 * lh + 4 * wave, oc = oct * 32 + c0;
        const bool store = p < a.P && oc < a.OC;    // OC is a multiple of 8: the four are in or out together
        split_store(a, sum, c0, store ? (size_t)p * a.OC + oc : 0, store, a.rp.enabled ? *form_word : 0, tab_hw, tab_ms, flags);
    }
    raise_flags(a.flag_word, flags);
}

template <int KS>
static bool launch_point_split_ks(hipStream_t st, const PointSplitArgs& a, int grid)
{
    constexpr int own = 2 * 32 * (KS * 32 + 16) > 4096 ? 2 * 32 * (KS * 32 + 16) : 4096;
    constexpr int lds_bytes = 32 * 16 + 32 * 8 + 8 * 128 + 16 + 8 * own;
    auto go = [&](auto kernel) {
        constexpr auto kern = decltype(kernel)::value;
        if (!ensure_dynamic_lds<kern>((size_t)lds_bytes))
            return false;
        hipLaunchKernelGGL(kern, dim3(grid), dim3(512), lds_bytes, st, a);
        last_launch_shape[0] = grid, last_launch_shape[1] = 512, last_launch_shape[2] = lds_bytes;
        return true;
    };
    return a.za != 0 ? go(kernel_constant<point_split_kernel<KS, true>>{}) : go(kernel_constant<point_split_kernel<KS, false>>{});
}

// False where the form does not apply.  (The caller has checked the layer: see launch_conv2d_pointwise.)
bool launch_point_split(hipStream_t st, const ConvGeom& g, const void* in, const void* w, const void* bias, int32_t in_zp,
                        const RescaleParams& rp, int32_t out_kind, void* out, uint32_t* flag_word)
{
    const int64_t P = (int64_t)g.N * g.OH * g.OW, n_oct = (g.OC + 31) / 32, tiles = (P + 31) / 32 * n_oct;
    if (g.IC % 256 != 0 || tiles > 1024 || (int64_t)g.OC * g.IC >= (int64_t(1) << 31))
        return false;
    PointSplitArgs a{};
    a.in = (const uint8_t*)in, a.w = (const int8_t*)w, a.bias = (const int32_t*)bias, a.out = out, a.flag_word = flag_word, a.rp = rp;
    a.P = (int32_t)P, a.OC = g.OC, a.za = in_zp, a.bias_len = g.bias_len, a.out_kind = out_kind;
    a.div_oct = make_fastdiv((uint32_t)n_oct);
    switch (g.IC / 256)
    {
        case 2: return launch_point_split_ks<2>(st, a, (int)tiles);
        case 3: return launch_point_split_ks<3>(st, a, (int)tiles);
        case 4: return launch_point_split_ks<4>(st, a, (int)tiles);
        case 5: return launch_point_split_ks<5>(st, a, (int)tiles);
        case 6: return launch_point_split_ks<6>(st, a, (int)tiles);
        case 7: return launch_point_split_ks<7>(st, a, (int)tiles);
        case 8: return launch_point_split_ks<8>(st, a, (int)tiles);
        default: return false;
    }
}

template <int KS, int NW, bool ZA>
static bool launch_conv_ksplit_za(hipStream_t st, const ConvSplitArgs& a, int grid)
{
    constexpr int lds_bytes = NW * 4096 + 32 * 16 + 32 * 8 + NW * 128 + 16;
    constexpr auto kern = conv_ksplit_i8_kernel<KS, NW, ZA>;
    if (!ensure_dynamic_lds<kern>((size_t)lds_bytes))
        return false;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(NW * 64), lds_bytes, st, a);
    last_launch_shape[0] = grid, last_launch_shape[1] = NW * 64, last_launch_shape[2] = lds_bytes;
    return true;
}

template <int KS, int NW>
static bool launch_conv_ksplit(hipStream_t st, const ConvSplitArgs& a, int grid)
{
    return a.za != 0 ? launch_conv_ksplit_za<KS, NW, true>(st, a, grid) : launch_conv_ksplit_za<KS, NW, false>(st, a, grid);
}

template <int NW, int NPT>
static bool launch_conv_ksplit_patch(hipStream_t st, const ConvPatchSplitArgs& a, int lds_bytes)
{
    auto go = [&](auto kernel) {
        constexpr auto kern = decltype(kernel)::value;
        if (!ensure_dynamic_lds<kern>((size_t)lds_bytes))
            return false;
        const int grid = a.n_groups * (int)a.div_oct.d;
        hipLaunchKernelGGL(kern, dim3(grid), dim3(NW * 64), lds_bytes, st, a);
        last_launch_shape[0] = grid, last_launch_shape[1] = NW * 64, last_launch_shape[2] = lds_bytes;
        return true;
    };
    return a.za != 0 ? go(kernel_constant<conv_ksplit_patch_kernel<NW, NPT, true>>{}) : go(kernel_constant<conv_ksplit_patch_kernel<NW, NPT, false>>{});
}

// Cuts the layer into blocks of up to `slots` output pixels whose patch fits the LDS beside `other` bytes.  False if none does.
static bool cut_patch_blocks(const ConvGeom& g, int slots, int64_t other, ConvPatchSplitArgs& a, int64_t& patch_bytes)
{
    const int across = (g.OW + slots - 1) / slots, TW = (g.OW + across - 1) / across;
    int down = (g.OH + slots / TW - 1) / (slots / TW);
    const int TH = (g.OH + down - 1) / down;
    down         = (g.OH + TH - 1) / TH;
    const int64_t PW = (int64_t)(TW - 1) * g.stride_x + 2 * (int64_t)g.dil_x + 1;
    const int64_t PH = (int64_t)(TH - 1) * g.stride_y + 2 * (int64_t)g.dil_y + 1;
    if (PW > 4096 || PH > 4096)
        return false;
    patch_bytes = PW * PH * (g.IC + 16);
    const int64_t n_blk = (int64_t)g.N * across * down, chunks = PW * PH * (g.IC / 16);
    if (other + patch_bytes > 160 * 1024 || n_blk * a.div_oct.d >= (int64_t(1) << 31))
        return false;
    a.TH = TH, a.n_blk = (int32_t)n_blk, a.chunks = (int32_t)chunks;
    a.div_bx = make_fastdiv((uint32_t)across), a.div_by = make_fastdiv((uint32_t)down), a.div_tw = make_fastdiv((uint32_t)TW);
    a.div_pw = make_fastdiv((uint32_t)PW);
    return fastdiv_exact_up_to((uint64_t)n_blk, (uint32_t)across) && fastdiv_exact_up_to((uint64_t)n_blk / across + 1, (uint32_t)down) &&
           fastdiv_exact_up_to((uint64_t)(PW * PH), (uint32_t)PW);
}

// The form with both operands through the LDS; false where it does not apply.
static bool try_conv_ksplit_patch(hipStream_t st, const ConvGeom& g, const ConvSplitArgs& c)
{
    constexpr int kMaxField = 32767;    // these travel as 16 bits
    if (g.KH != 3 || g.KW != 3 || g.stride_y > kMaxField || g.stride_x > kMaxField || g.dil_y > kMaxField || g.dil_x > kMaxField ||
        g.pad_top > kMaxField || g.pad_left > kMaxField)
        return false;
    ConvPatchSplitArgs a{};
    a.in = c.in, a.w = c.w, a.bias = c.bias, a.pad_page = c.pad_page, a.out = c.out, a.flag_word = c.flag_word, a.rp = c.rp;
    a.OC = c.OC, a.IH = c.IH, a.IW = c.IW, a.OH = c.OH, a.OW = c.OW;
    a.sy = (int16_t)c.sy, a.sx = (int16_t)c.sx, a.dy = (int16_t)c.dy, a.dx = (int16_t)c.dx;
    a.pad_top = (int16_t)c.pad_top, a.pad_left = (int16_t)c.pad_left, a.za = c.za;
    a.bias_len = c.bias_len, a.out_kind = c.out_kind;
    a.div_oct = c.div_oct;
    const int nw         = g.IC / 32;
    const int64_t tables = 32 * 16 + 32 * 8 + nw * 128 + 16;
    int64_t patch_bytes  = 0;
    int npt              = 1;
    if (!cut_patch_blocks(g, 32, tables + nw * 4096, a, patch_bytes))
        return false;
    // Two pixel tiles a block once single ones would be more than a round of workgroups
    if (nw == 8 && (int64_t)a.n_blk * a.div_oct.d > 256)
    {
        ConvPatchSplitArgs b = a;
        int64_t bytes        = 0;
        if (cut_patch_blocks(g, 64, tables + 2 * nw * 4096, b, bytes))
            a = b, patch_bytes = bytes, npt = 2;
    }
    // Images of a few pixels leave most of a block empty; the other form's tiles run across images.
    if ((int64_t)a.n_blk * npt * 2 > 3 * (int64_t)c.n_pt)
        return false;
    const int max_groups  = 256 / (int)a.div_oct.d > 0 ? 256 / (int)a.div_oct.d : 1;
    const int per_group   = (a.n_blk + max_groups - 1) / max_groups;
    a.n_groups            = (a.n_blk + per_group - 1) / per_group;
    const int64_t weights = (int64_t)nw * 32 * (9 * 32 + 16), data = npt * nw * 4096 + patch_bytes;
    const int lds_bytes   = (int)(tables + (data > weights ? data : weights));
    switch (nw)
    {
        case 8: return npt == 2 ? launch_conv_ksplit_patch<8, 2>(st, a, lds_bytes) : launch_conv_ksplit_patch<8, 1>(st, a, lds_bytes);
        case 12: return launch_conv_ksplit_patch<12, 1>(st, a, lds_bytes);
        case 16: return launch_conv_ksplit_patch<16, 1>(st, a, lds_bytes);
        default: return false;
    }
}

// nullptr when the layer is not one these kernels take; `small`: the form without a patch may take it.
const char* launch_conv2d_ksplit(hipStream_t st, int32_t in_dtype, int32_t out_dtype, const ConvGeom& g, const void* in,
                                 const void* w, const void* bias, int32_t in_zp, int32_t w_zp, const RescaleParams& rp,
                                 void* out, const void* pad_page, uint32_t* flag_word, bool small)
{
    if (in_dtype != TMI_INT8 || w_zp != 0 || !flag_word || !pad_page)
        return nullptr;
    const int taps = g.KH * g.KW;
    if (taps < 2 || (g.IC & 31) || g.IC < 32 || (g.OC & 7) || g.OC < 8 || g.OC > 4096)
        return nullptr;
    if (rp.enabled ? (!rp.fast || (out_dtype != TMI_INT8 && out_dtype != TMI_INT16)) : out_dtype != TMI_INT32)
        return nullptr;
    if ((((uintptr_t)in | (uintptr_t)w | (uintptr_t)out | (uintptr_t)pad_page) & 15) || ((uintptr_t)bias & 3))
        return nullptr;
    const int64_t P = (int64_t)g.N * g.OH * g.OW;
    if (P < 1 || (int64_t)g.N * g.IH * g.IW * g.IC >= (int64_t(1) << 31) || P * g.OC >= (int64_t(1) << 31) ||
        (int64_t)g.OC * taps * g.IC >= (int64_t(1) << 31))
        return nullptr;
    // 4, 8 or 16 waves a workgroup: at most 10 K steps a wave (a wave's time is its instruction count)
    const int steps = taps * (g.IC / 32);
    const int nw    = steps > 80 ? 16 : (steps > 40 ? 8 : 4);
    const int ksw   = (steps + nw - 1) / nw;
    if (ksw > 10)
        return nullptr;

    ConvSplitArgs a{};
    a.in = (const uint8_t*)in, a.w = (const int8_t*)w, a.bias = (const int32_t*)bias, a.out = out;
    a.pad_page = (const uint8_t*)pad_page, a.flag_word = flag_word, a.rp = rp;
    a.P = (int32_t)P, a.IC = g.IC, a.OC = g.OC;
    a.IH = g.IH, a.IW = g.IW, a.OH = g.OH, a.OW = g.OW, a.KW = g.KW;
    a.sy = g.stride_y, a.sx = g.stride_x, a.dy = g.dil_y, a.dx = g.dil_x, a.pad_top = g.pad_top, a.pad_left = g.pad_left;
    a.za = in_zp, a.bias_len = g.bias_len;
    a.out_kind = !rp.enabled ? 0 : (out_dtype == TMI_INT8 ? 1 : 2);
    a.n_oct    = (g.OC + 31) / 32;
    a.n_pt     = (int32_t)((P + 31) / 32);
    a.steps = steps, a.spt = g.IC / 32, a.ksw = ksw;
    // At most one workgroup per CU, each walking its pixel tiles with the weight fragments in registers (us for a
    // workgroup per tile / at most 256 workgroups, 3x3, fused RESCALE: [8,14,14,256]->256 10.9 / 9.0, [16,14,14,256]->256
    // 18.5 / 12.8, [4,28,28,256]->256 19.6 / 12.9, [8,14,14,384]->384 24.1 / 15.3; 320 workgroups: 17.0 and 23.0 on the last
    // two, 192: 14.8 and 18.2).
    const int max_groups = 256 / a.n_oct > 0 ? 256 / a.n_oct : 1;
    const int per_group  = (a.n_pt + max_groups - 1) / max_groups;    // pixel tiles a workgroup walks: the same for all
    a.n_groups = (a.n_pt + per_group - 1) / per_group;
    a.div_oct = make_fastdiv((uint32_t)a.n_oct), a.div_spt = make_fastdiv((uint32_t)a.spt);
    a.div_kw = make_fastdiv((uint32_t)g.KW), a.div_ow = make_fastdiv((uint32_t)g.OW), a.div_oh = make_fastdiv((uint32_t)g.OH);
    const int grid = a.n_groups * a.n_oct;
    if (!fastdiv_exact_up_to((uint64_t)grid, (uint32_t)a.n_oct) || !fastdiv_exact_up_to((uint64_t)P, (uint32_t)g.OW) ||
        !fastdiv_exact_up_to((uint64_t)P / g.OW + 1, (uint32_t)g.OH) || !fastdiv_exact_up_to((uint64_t)steps, (uint32_t)a.spt) ||
        !fastdiv_exact_up_to((uint64_t)taps, (uint32_t)g.KW))
        return nullptr;
    if (try_conv_ksplit_patch(st, g, a))
        return rp.enabled ? "conv2d_ksplit_patch_i8_rescale" : "conv2d_ksplit_patch_i8";
    if (!small)
        return nullptr;
    bool ok;
    if (nw == 4)
        ok = ksw <= 4 ? launch_conv_ksplit<4, 4>(st, a, grid) : launch_conv_ksplit<10, 4>(st, a, grid);
    else if (nw == 8)
        ok = launch_conv_ksplit<10, 8>(st, a, grid);
    else
        ok = launch_conv_ksplit<10, 16>(st, a, grid);
    if (!ok)
        return nullptr;
    return rp.enabled ? "conv2d_ksplit_i8_rescale" : "conv2d_ksplit_i8";
}

}    // namespace tmi
