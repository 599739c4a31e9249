// CONV2D whose weights stay in LDS while the pixels stream past them: int8 (fused RESCALE or int32 results), fp16 and bf16 layers
// of any channel count, taps, stride, dilation and padding with weight_zp 0, where a workgroup that stages an input patch for
// one tile of results spends its time on that set-up.
//
//   out[p][oc] = sum_(tap, ic) (in[p, tap][ic] - input_zp) * w[oc][tap][ic] + bias[oc]      (tensor_ops.cpp:843-882)
//
// K is walked in chunks of 16 bytes of one tap's channel vector, (ky, kx, ic) in order, two chunks a matrix instruction (lane
// half h takes chunk 2 s + h).  A workgroup of four waves stages the weights of 32 * OCT channels once, rows side by side
// per chunk, so that a fragment is 512 consecutive bytes; the last chunk of a tap is filled up with zeros, so whatever
// the pixel holds behind its channels counts for nothing (floating point: it is masked away, infinities times zero).  Then
// every wave walks tiles of 32 pixels on its own, without a barrier: a lane loads its 16 bytes straight from the image,
// or from the page of input_zp bytes where the tap lies outside, DEPTH steps ahead.  What a chunk adds to the pixel's offset
// and which of the pixel's row and column bits it needs is read from a table in LDS.
//
// What bounds it: a wave alone on its SIMD issues an instruction every eight clocks, so a step of 27 instructions is 100 ns; three
// waves a SIMD bring it near the memory pipeline's 32 clocks a load.  us patch kernel / this kernel: int8 [36,129,126,20]->101 192 / 43,
// [19,84,89,16]->108 3x3 63 / 22, [5,106,106,16]->232 3x3 stride 2 18.7 / 7.1, fp16 [15,54,65,68]->64 28.2 / 7.6.  Whole groups of
// steps run without a test (a test and a branch a step: 4 ... 7 % slower over 257 layers).
//
// Channel vectors that begin between words (more than 32 bytes of them) are read from the word before and shifted where they are used: int8
// [60,32,32,163]->16 1x1 8.0, with the copies such rows went through before 15.5; K split, [2,11,16,285]->44 5x5 34.4 -> 25.8, bf16 [1,45,9,219]->24 19.7 -> 13.2.
//
// The second kernel, for few tiles and a long reduction, splits K over the waves of a workgroup (see there).
#include <type_traits>

#include "outside_taps.h"

namespace tmi
{

struct TapsArgs
{
    const uint8_t* in;
    const uint8_t* w;
    const void* bias;
    void* out;
    const uint8_t* pad_page;    // 16 bytes of input_zp
    uint32_t* flag_word;
    RescaleParams rp;
    int32_t P, OC, OH, OW, IH, IW;
    int32_t KH, KW, sy, sx, dy, dx, pad_top, pad_left;
    int32_t row_bytes;     // of a pixel's channel vector
    int32_t pieces;        // chunks of a tap
    int32_t chunks;        // taps * pieces
    int32_t steps;         // two chunks each
    int32_t za, bias_len;
    int32_t out_kind;      // 0: int32, 1: int8, 2: int16 through the RESCALE; 3: floating point of the operands' type
    int32_t n_pt;          // tiles of 32 pixels
    int32_t groups;        // workgroups per channel block
    int32_t n_ocb;
    int32_t rows_bytes;    // bytes of 32 pixels' results where they are gathered in LDS, else 0
    int32_t row_skip, chunk_skip;    // a workgroup's lanes of weight chunks: whole rows and chunks
    int32_t last;          // offset of the input's last 16 bytes
    int32_t edge_off;      // the same less the last chunk's offset from its window's first tap
    int32_t w_last;        // offset of the weights' last 16 bytes
    FastDiv div_ow, div_oh, div_chunks, div_pieces, div_kw, div_groups;
};

constexpr int kTapsWaves   = 4;
constexpr int kTapsPartial = 1 << 27;    // table entry: the chunk is filled up behind the pixel's channels
constexpr int kTapsDead    = 1 << 26;    // no chunk at all

template <int OCT>
constexpr int taps_fixed_lds()
{
    return 32 * OCT * (16 + 8 + 4) + 16;
}
template <int OCT>
__host__ __device__ constexpr int taps_lds_bytes(int steps)
{
    return taps_fixed_lds<OCT>() + 2 * steps * (OCT * 512 + 16 + 8);
}

// What the epilogue reads of a tile of 32 channels.
struct TapsTables
{
    const HighWordScale* hw;
    const v2i* ms;           // multiplier and validated shift
    const int32_t* start;    // starting values (floating point: the bias)
    const int32_t* form;     // bit 0: the high-word form for all 32 channels; bit 1: no sign test in it
};

// A lane's V results of pixel p from channel `oc` on, the tile's channel `cb`: RESCALE or bias, and the store.  rows: where the
// results of the tile's 32 pixels are gathered instead, as they lie in memory (channel counts of no whole words).
template <typename T, int V, typename R>
__device__ __forceinline__ void finish_taps(const TapsArgs& a, const TapsTables& tab, const R& v, int oc, int cb, int p, uint32_t& flags,
                                            uint8_t* rows = nullptr)
{
    const int32_t v_lo = a.rp.lo, v_hi = a.rp.hi;
    const int oc_align = (a.OC & 15) == 0 ? 16 : ((a.OC & 7) == 0 ? 8 : ((a.OC & 3) == 0 ? 4 : 1));
    int cnt            = a.OC - oc;
    cnt                = p >= a.P || cnt < 0 ? 0 : (cnt > V ? V : cnt);
    const size_t at    = (size_t)(p < a.P ? p : 0) * a.OC + oc;
    const int row_at   = (p & 31) * a.OC + oc;
    auto store_each = [&](auto* out, const auto& r) {
        auto* o = out + at;
        if (rows)
            o = reinterpret_cast<decltype(o)>(rows) + row_at;
#pragma unroll
        for (int e = 0; e < V; e++)
            if (e < cnt)
                o[e] = (std::remove_reference_t<decltype(*o)>)r[e];
    };
    if constexpr (Mma<T>::is_int)
    {
        if (a.out_kind == 0)
        {
            int32_t* o = reinterpret_cast<int32_t*>(a.out) + at;
            if (oc_align >= 4)
            {
#pragma unroll
                for (int q = 0; q < V / 4; q++)
                    if (4 * q < cnt)
                        *reinterpret_cast<v4i*>(o + 4 * q) = v4i{ v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3] };
            }
            else
#pragma unroll
                for (int e = 0; e < V; e++)
                    if (e < cnt)
                        o[e] = v[e];
            return;
        }
        const int form = __builtin_amdgcn_readfirstlane(*tab.form);
        int first      = cb;
        asm volatile("" : "+v"(first));    // (the constants are read per tile rather than held in registers)
        int32_t r[V];
        if (form & 1)
        {
            auto high = [&](auto DOUBLE) {
#pragma unroll
                for (int e = 0; e < V; e++)
                {
                    r[e] = clamp_med3(high_word_rescale64<decltype(DOUBLE)::value>(v[e], tab.hw[first + e]), v_lo, v_hi);
                    if ((e & 3) == 3)
                        __builtin_amdgcn_sched_barrier(0);
                }
            };
            if (a.rp.double_round && !(form & 2))
                high(std::true_type{});
            else
                high(std::false_type{});
        }
        else
#pragma unroll
            for (int e = 0; e < V; e++)
            {
                // fast_rescale() from multiplier and shift alone; elements that are not stored raise nothing
                const v2i c     = tab.ms[first + e];
                const int32_t s = c.y;
                if (s <= 31 && e < cnt && (v[e] < -(1 << (s - 1)) || v[e] >= (1 << (s - 1))))
                    flags |= TMI_FLAG_SCALE_VALUE;
                int64_t round = int64_t(1) << (s - 1);
                if (a.rp.double_round && s > 31)
                    round += v[e] >= 0 ? (int64_t(1) << 30) : -(int64_t(1) << 30);
                const int64_t pr = (int64_t)v[e] * (int64_t)c.x + round;
                r[e]             = clamp_med3((int32_t)(pr >> s) + a.rp.out_zp, v_lo, v_hi);
            }
        if (a.out_kind == 1)
        {
            int pk[V / 4];
#pragma unroll
            for (int q = 0; q < V / 4; q++)
                pk[q] = __builtin_amdgcn_perm(r[4 * q + 1], r[4 * q], 0x0c0c0400) | __builtin_amdgcn_perm(r[4 * q + 3], r[4 * q + 2], 0x04000c0c);
            int8_t* o = reinterpret_cast<int8_t*>(a.out) + at;
            if constexpr (V == 16)
            {
                if (oc_align == 16)
                {
                    if (cnt > 0)
                        *reinterpret_cast<v4i*>(o) = v4i{ pk[0], pk[1], pk[2], pk[3] };
                    return;
                }
                if (oc_align == 8)
                {
#pragma unroll
                    for (int q = 0; q < 2; q++)
                        if (8 * q < cnt)
                            *reinterpret_cast<v2i*>(o + 8 * q) = v2i{ pk[2 * q], pk[2 * q + 1] };
                    return;
                }
            }
            if (oc_align >= 4)
            {
#pragma unroll
                for (int q = 0; q < V / 4; q++)
                    if (4 * q < cnt)
                        *reinterpret_cast<int*>(o + 4 * q) = pk[q];
            }
            else
                store_each(reinterpret_cast<int8_t*>(a.out), r);
        }
        else if (oc_align >= 4)
        {
            int16_t* o = reinterpret_cast<int16_t*>(a.out) + at;
#pragma unroll
            for (int q = 0; q < V / 4; q++)
                if (4 * q < cnt)
                    *reinterpret_cast<v2i*>(o + 4 * q) = v2i{ (r[4 * q] & 0xffff) | (r[4 * q + 1] << 16), (r[4 * q + 2] & 0xffff) | (r[4 * q + 3] << 16) };
        }
        else
            store_each(reinterpret_cast<int16_t*>(a.out), r);
    }
    else
    {
        float f[V];
#pragma unroll
        for (int q = 0; q < V / 4; q++)
        {
            const v4i b = *reinterpret_cast<const v4i*>(tab.start + cb + 4 * q);
#pragma unroll
            for (int e = 0; e < 4; e++)
                f[4 * q + e] = v[4 * q + e] + __int_as_float(b[e]);
        }
        uint32_t h[V];
#pragma unroll
        for (int e = 0; e < V; e++)
        {
            T x;
            store_from_float(&x, f[e]);
            h[e] = __builtin_bit_cast(uint16_t, x);
        }
        int16_t* o = reinterpret_cast<int16_t*>(a.out) + at;
        if constexpr (V == 16)
            if (oc_align >= 8)
            {
#pragma unroll
                for (int q = 0; q < 2; q++)
                    if (8 * q < cnt)
                        *reinterpret_cast<v4i*>(o + 8 * q) =
                            v4i{ (int)(h[8 * q] | h[8 * q + 1] << 16), (int)(h[8 * q + 2] | h[8 * q + 3] << 16),
                                 (int)(h[8 * q + 4] | h[8 * q + 5] << 16), (int)(h[8 * q + 6] | h[8 * q + 7] << 16) };
                return;
            }
        if (oc_align >= 4)
        {
#pragma unroll
            for (int q = 0; q < V / 4; q++)
                if (4 * q < cnt)
                    *reinterpret_cast<v2i*>(o + 4 * q) = v2i{ (int)(h[4 * q] | h[4 * q + 1] << 16), (int)(h[4 * q + 2] | h[4 * q + 3] << 16) };
        }
        else
            store_each(reinterpret_cast<int16_t*>(a.out), h);
    }
}

// Results that are NaN because of a tap outside the image (see outside_taps.h): a wave that met a NaN looks at its channels' weights behind its loop, and goes
// over its tiles once more where one is infinite or NaN.
template <int N, typename R>
__device__ __forceinline__ bool any_nan(const R& v)
{
    bool nan = false;
#pragma unroll
    for (int e = 0; e < N; e += 2)
        nan |= __builtin_isunordered(v[e], v[e + 1]);
    return __any(nan);
}
// `channels` of the weights from channel oc on, by all lanes of the wave
template <typename T>
__device__ __forceinline__ bool odd_weights(const TapsArgs& a, int oc, int channels)
{
    const int64_t row = (int64_t)a.KH * a.KW * a.row_bytes;
    channels          = a.OC - oc < channels ? a.OC - oc : channels;
    return channels > 0 && __any(weights_not_finite<T>(a.w + oc * row, channels * row, lane_counted(), 64));
}
// the lane's pixel p, `tiles` tiles of 32 channels of which it holds `each` from channel oc on
template <typename T>
__device__ __forceinline__ void sum_again(const TapsArgs& a, int p, int oc, int tiles, int each)
{
    const int r = (int)fdiv((uint32_t)p, a.div_ow), n = (int)fdiv((uint32_t)r, a.div_oh);
    without_outside_taps<T>(OutsideTaps{ a.in, a.w, a.bias, a.out, a.row_bytes, a.IH, a.IW, a.OC, a.OH, a.OW, a.KH, a.KW, a.sy, a.sx, a.dy, a.dx, a.pad_top, a.pad_left, a.bias_len },
                            p < a.P, n, r - n * a.OH, p - r * a.OW, oc, tiles, each);
}

// How channel vectors lie: whole chunks from 16 bytes on; anywhere, beginning with words; anywhere.
enum TapsRows
{
    kTapsWhole,
    kTapsWords,
    kTapsOdd
};

template <typename T, int OCT, int ROWS>
__global__ __launch_bounds__(kTapsWaves * 64, 2) void conv_taps_kernel(TapsArgs a)
{
    constexpr bool RAGGED = ROWS != kTapsWhole;
    using M             = Mma<T>;
    using acc_t         = typename M::acc_t;
    constexpr int NT    = kTapsWaves * 64;
    constexpr int OCB   = 32 * OCT;
    constexpr int PITCH = OCT * 512 + 16;
    constexpr int DEPTH = OCT <= 2 ? 8 : 4;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    HighWordScale* tab_hw = reinterpret_cast<HighWordScale*>(lds);
    v2i* tab_ms           = reinterpret_cast<v2i*>(lds + OCB * 16);
    int32_t* tab_start    = reinterpret_cast<int32_t*>(lds + OCB * 24);
    int32_t* tab_form     = reinterpret_cast<int32_t*>(lds + OCB * 28);
    v2i* tab_chunk        = reinterpret_cast<v2i*>(lds + taps_fixed_lds<OCT>());
    uint8_t* wl           = lds + taps_fixed_lds<OCT>() + 2 * a.steps * 8;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 31, lh = lane >> 5;
    const int ocb = (int)fdiv(blockIdx.x, a.div_groups), grp = (int)blockIdx.x - ocb * a.groups;
    const int oc0 = ocb * OCB;

    // ---- weights into registers (on their way while the tables are written), then LDS ----------------------------------
    // (consecutive lanes take consecutive chunks of a row; all of a batch's loads are in flight at once)
    const int partial = a.row_bytes & 15;    // bytes of a tap's last chunk, 0: whole
    constexpr int WB  = RAGGED ? 8 : 12;
    v4i wv[WB];
    int wdst[WB];
    int w_oc = (int)fdiv((uint32_t)tid, a.div_chunks), w_c = tid - w_oc * a.chunks;    // the lane's next chunk
    auto load_weights = [&]() {
#pragma unroll
        for (int u = 0; u < WB; u++)
        {
            const bool ok = w_oc < OCB && oc0 + w_oc < a.OC;
            const int row = ok ? oc0 + w_oc : 0, c = ok ? w_c : 0;
            wdst[u] = w_oc < OCB ? w_c * PITCH + (w_oc >> 5) * 512 + (((w_oc >> 2) & 3) * 8 + ((w_oc >> 4) & 1) * 4 + (w_oc & 3)) * 16 : -1;
            if constexpr (!RAGGED)
                wv[u] = *reinterpret_cast<const v4i*>(a.w + (uint32_t)((row * a.chunks + c) * 16));
            else
            {
                const int tap = (int)fdiv((uint32_t)c, a.div_pieces), piece = c - tap * a.pieces;
                const int off = (row * (a.KH * a.KW) + tap) * a.row_bytes + piece * 16;
                const int n   = piece == a.pieces - 1 && partial ? partial : 16;
                const int at  = off <= a.w_last ? off : a.w_last;
                wv[u]         = load16(a.w + (uint32_t)at);
                if (__any(off > a.w_last))
                    wv[u] = drop_bytes(wv[u], off - at);
                wv[u] = keep_bytes(wv[u], n);
            }
            if (!ok)
                wv[u] = v4i{ 0, 0, 0, 0 };
            w_oc += a.row_skip, w_c += a.chunk_skip;    // NT chunks on
            const bool wrap = w_c >= a.chunks;
            w_oc += wrap ? 1 : 0, w_c -= wrap ? a.chunks : 0;
        }
    };
    auto store_weights = [&]() {
#pragma unroll
        for (int u = 0; u < WB; u++)
            if (wdst[u] >= 0)
                *reinterpret_cast<v4i*>(wl + wdst[u]) = wv[u];
    };
    load_weights();

    for (int c = tid; c < 2 * a.steps; c += NT)
    {
        v2i e = { 0, kTapsDead };
        if (c < a.chunks)
        {
            const int tap = (int)fdiv((uint32_t)c, a.div_pieces), piece = c - tap * a.pieces;
            const int ky = (int)fdiv((uint32_t)tap, a.div_kw), kx = tap - ky * a.KW;
            e.x = (ky * a.dy * a.IW + kx * a.dx) * a.row_bytes + piece * 16;
            e.y = (1 << ky) | (1 << (13 + kx)) | (piece == a.pieces - 1 && partial ? kTapsPartial : 0);
        }
        tab_chunk[c] = e;
    }
    if (a.chunks & 1)    // the dead half of the last step
        for (int r = tid; r < OCB; r += NT)
            *reinterpret_cast<v4i*>(wl + a.chunks * PITCH + r * 16) = v4i{ 0, 0, 0, 0 };
    uint32_t flags = 0;
    if (wave < OCT)
    {
        // wave t works out the constants of channel tile t, both halves alike
        const int oc  = oc0 + wave * 32 + li;
        const bool ok = oc < a.OC;
        const int occ = ok ? oc : oc0;
        if constexpr (M::is_int)
        {
            const int32_t b = reinterpret_cast<const int32_t*>(a.bias)[a.bias_len == 1 ? 0 : occ];
            if (a.rp.enabled)
            {
                const int32_t m_raw   = load_multiplier(a.rp, occ);
                const int32_t s_raw   = load_shift(a.rp, occ);
                const int32_t s_first = __builtin_amdgcn_readfirstlane(s_raw);
                const ChannelScale cs = make_channel_scale(ok ? m_raw : 0, ok ? s_raw : s_first, a.rp.double_round != 0, flags);
                const int s_min       = a.rp.double_round ? 33 : 32;
                // bit 0: the high-word form for all 32 channels; bit 1: no sign test in it (a negative value is clamped away
                // with either rounding term)
                const int form = (__all(cs.s >= s_min && cs.s <= zp_fold_max_shift(a.rp.out_zp)) ? 1 : 0) |
                                 (a.rp.lo >= a.rp.out_zp && __all(cs.m >= 0) ? 2 : 0);
                if (lh == 0)
                {
                    tab_ms[wave * 32 + li] = v2i{ cs.m, cs.s };
                    tab_hw[wave * 32 + li] = make_high_word_scale(cs, a.rp.out_zp);
                }
                if (lane == 0)
                    tab_form[wave] = form;
            }
            if (lh == 0)
                tab_start[wave * 32 + li] = ok ? b : 0;
        }
        else if (lh == 0)
            tab_start[wave * 32 + li] = ok ? __float_as_int(load_as_float<T>(a.bias, a.bias_len == 1 ? 0 : occ)) : 0;
    }
    __syncthreads();    // the tables

    // ---- pixels ---------------------------------------------------------------------------------------------------------
    const int first_pt = grp * kTapsWaves + wave, pt_step = a.groups * kTapsWaves;
    int32_t pix_off = 0, pix_miss = -1;    // offset of the window's first tap; a zero bit per tap row and column inside the image
    bool edge = false;                     // RAGGED: the tensor may end inside the 16 bytes of a lane of this tile
    auto enter_tile = [&](int pt) {
        int p = pt * 32 + li;
        p     = p < a.P ? p : a.P - 1;
        const int r  = (int)fdiv((uint32_t)p, a.div_ow), ox = p - r * a.OW;
        const int n  = (int)fdiv((uint32_t)r, a.div_oh), oy = r - n * a.OH;
        const int y0 = oy * a.sy - a.pad_top, x0 = ox * a.sx - a.pad_left;
        pix_off      = ((n * a.IH + y0) * a.IW + x0) * a.row_bytes;
        int in_bits  = 0;
        for (int k = 0; k < a.KH; k++)
            in_bits |= ((unsigned)(y0 + k * a.dy) < (unsigned)a.IH ? 1 : 0) << k;
        for (int k = 0; k < a.KW; k++)
            in_bits |= ((unsigned)(x0 + k * a.dx) < (unsigned)a.IW ? 1 : 0) << (13 + k);
        pix_miss = ~(in_bits | kTapsPartial);
        if constexpr (RAGGED)
            edge = __any(pix_off > a.edge_off);
    };
    // A 16-byte load from between words takes the memory pipeline more than twice as long as one from a word on: such chunks are read from the word
    // before, with the word behind, and shifted where they are used.  So are they cut there to their channels: here a lane would wait for
    // its load.
    constexpr bool ODD = ROWS == kTapsOdd, CUT = RAGGED && !M::is_int;
    v4i fb[DEPTH];
    int behind[ODD ? DEPTH : 1] = {};
    uint32_t places = 0;    // where in a word each load's chunk begins, two bits each; from bit 16 on: whether it is a tap's last
    auto note        = [&](int d, uint32_t place, int bits) {
        if constexpr (ODD)
            places = (places & ~(3u << (2 * d))) | place << (2 * d);
        if constexpr (CUT)
            places = (places & ~(65536u << d)) | (bits & kTapsPartial ? 65536u << d : 0u);
    };
    auto load_pixels = [&](int d, v2i e, bool careful) {
        const bool inside  = (e.y & pix_miss) == 0;
        const int off      = pix_off + e.x;
        const uint8_t* src = inside ? a.in + (uint32_t)off : a.pad_page;
        if constexpr (!RAGGED)
            fb[d] = *reinterpret_cast<const v4i*>(src);
        else if (careful)
        {
            const int past = inside && off > a.last ? off - a.last : 0;
            if (__any(past))
                fb[d] = drop_bytes(load16(src - past), past);
            else
                fb[d] = load16(src);
            note(d, 0, e.y);
        }
        else if constexpr (ODD)
        {
            const uint8_t* word = reinterpret_cast<const uint8_t*>((uintptr_t)src & ~(uintptr_t)3);
            __builtin_memcpy(&fb[d], __builtin_assume_aligned(word, 4), 16);
            behind[d] = *reinterpret_cast<const int*>(word + 16);
            note(d, (uint32_t)(uintptr_t)src & 3u, e.y);
        }
        else
        {
            fb[d] = load16(src);
            note(d, 0, e.y);
        }
    };
    auto pixels = [&](int d) {
        v4i v = fb[d];
        if constexpr (ODD)
        {
            const uint32_t by = places >> (2 * d) & 3u;
#pragma unroll
            for (int k = 0; k < 4; k++)
                v[k] = (int)__builtin_amdgcn_alignbyte((uint32_t)(k < 3 ? fb[d][k < 3 ? k + 1 : 3] : behind[d]), (uint32_t)fb[d][k], by);
        }
        if constexpr (CUT)
            if (__any(places & (65536u << d)))
            {
                const int n = places & (65536u << d) ? partial : 16;
#pragma unroll
                for (int k = 0; k < 4; k++)
                {
                    // (channels are 16 bits: whole words, half of one, none)
                    const int m = n - 4 * k;
                    v[k]        = m >= 4 ? v[k] : (m == 2 ? v[k] & 0xffff : 0);
                }
            }
        return v;
    };
    auto load_group = [&](bool careful) {
#pragma unroll
        for (int d = 0; d < DEPTH; d++)
            if (d < a.steps)
                load_pixels(d, tab_chunk[2 * d + lh], careful);
    };
    if (first_pt < a.n_pt)
    {
        enter_tile(first_pt);
        if (edge)
            load_group(true);
        else
            load_group(false);
    }
    store_weights();
    for (int first = WB * NT; first < OCB * a.chunks; first += WB * NT)
    {
        load_weights();
        store_weights();
    }
    __syncthreads();
    if constexpr (M::is_int)
        if (a.za != 0)
        {
            // -input_zp * sum(w) joins a channel's starting value: the rows' sums from LDS, NT / OCB lanes a row
            constexpr int LPR = NT / OCB > 0 ? NT / OCB : 1;
            const int row = tid % OCB, r32 = row & 31;
            int sum       = 0;
            for (int c = tid / OCB; c < a.chunks; c += LPR)
                sum += dot4_ones(*reinterpret_cast<const v4i*>(wl + c * PITCH + row * 16));
            if (tid < LPR * OCB)
                atomicAdd(&tab_start[(row & ~31) + 16 * ((r32 >> 2) & 1) + 4 * (r32 >> 3) + (r32 & 3)], -a.za * sum);
            __syncthreads();
        }

    const uint8_t* wfrag = wl + lh * PITCH + li * 16;
    uint8_t* rows        = wl + 2 * a.steps * PITCH + wave * a.rows_bytes;
    bool met_nan         = false;
    int pt               = first_pt;
    for (; pt < a.n_pt; pt += pt_step)
    {
        acc_t acc[OCT];
#pragma unroll
        for (int t = 0; t < OCT; t++)
        {
#pragma unroll
            for (int e = 0; e < 16; e++)
                acc[t][e] = 0;
            if constexpr (M::is_int)
#pragma unroll
                for (int q = 0; q < 4; q++)
                {
                    const v4i b = *reinterpret_cast<const v4i*>(tab_start + t * 32 + 16 * lh + 4 * q);
                    acc[t][4 * q] = b[0], acc[t][4 * q + 1] = b[1], acc[t][4 * q + 2] = b[2], acc[t][4 * q + 3] = b[3];
                }
        }
        v4i fa[2][OCT];
        auto load_weight_fragments = [&](int s, v4i (&f)[OCT]) {
            const uint8_t* wf = wfrag + (s < a.steps ? s : 0) * 2 * PITCH;
#pragma unroll
            for (int t = 0; t < OCT; t++)
                f[t] = *reinterpret_cast<const v4i*>(wf + t * 512);
        };
        load_weight_fragments(0, fa[0]);
        // whole groups whose successor is whole, without a test; then what is left, step by step
        int s0 = 0;
#pragma unroll 1
        for (; !edge && s0 + 2 * DEPTH <= a.steps; s0 += DEPTH)
        {
            v2i next[DEPTH];
#pragma unroll
            for (int d = 0; d < DEPTH; d++)
                next[d] = tab_chunk[2 * (s0 + DEPTH + d) + lh];
            const uint8_t* wf = wfrag + s0 * 2 * PITCH;
#pragma unroll
            for (int d = 0; d < DEPTH; d++)
            {
#pragma unroll
                for (int t = 0; t < OCT; t++)
                    fa[(d + 1) & 1][t] = *reinterpret_cast<const v4i*>(wf + (d + 1) * 2 * PITCH + t * 512);
                const v4i px = pixels(d);
#pragma unroll
                for (int t = 0; t < OCT; t++)
                    acc[t] = M::mma(fa[d & 1][t], px, acc[t]);
                load_pixels(d, next[d], false);
            }
        }
#pragma unroll 1
        for (; s0 < a.steps; s0 += DEPTH)
        {
            v2i next[DEPTH];
#pragma unroll
            for (int d = 0; d < DEPTH; d++)
                next[d] = tab_chunk[2 * (s0 + DEPTH + d < a.steps ? s0 + DEPTH + d : 0) + lh];
#pragma unroll
            for (int d = 0; d < DEPTH; d++)
            {
                if (s0 + d >= a.steps)
                    break;
                load_weight_fragments(s0 + d + 1, fa[(d + 1) & 1]);
                const v4i px = pixels(d);
#pragma unroll
                for (int t = 0; t < OCT; t++)
                    acc[t] = M::mma(fa[d & 1][t], px, acc[t]);
                if (s0 + DEPTH + d < a.steps)
                    load_pixels(d, next[d], edge);
            }
        }
        const int p = pt * 32 + li;
        if (pt + pt_step < a.n_pt)
        {
            enter_tile(pt + pt_step);    // on its way while this tile is finished
            if (edge)
                load_group(true);
            else
                load_group(false);
        }
#pragma unroll
        for (int t = 0; t < OCT; t++)
        {
            if constexpr (!M::is_int)
                met_nan |= any_nan<16>(acc[t]);
            finish_taps<T, 16>(a, TapsTables{ tab_hw + 32 * t, tab_ms + 32 * t, tab_start + 32 * t, tab_form + t }, acc[t],
                               oc0 + 32 * t + 16 * lh, 16 * lh, p, flags, a.rows_bytes ? rows : nullptr);
            __builtin_amdgcn_sched_barrier(0);    // (one channel tile's values at a time)
        }
        if (a.rows_bytes)
        {
            // (one channel block: the tile's results are consecutive in memory)
            __builtin_amdgcn_wave_barrier();    // the wave's own LDS accesses complete in order
            const int px    = a.P - pt * 32 < 32 ? a.P - pt * 32 : 32;
            const int bytes = px * (a.rows_bytes / 32);
            uint8_t* dst    = reinterpret_cast<uint8_t*>(a.out) + (size_t)pt * a.rows_bytes;
            for (int i = 16 * lane; i + 16 <= bytes; i += 16 * 64)
                *reinterpret_cast<v4i*>(dst + i) = *reinterpret_cast<const v4i*>(rows + i);
            const int i = (bytes & ~15) + lane;
            if (i < bytes)
                dst[i] = rows[i];
            __builtin_amdgcn_wave_barrier();
        }
    }
    if constexpr (M::is_int)
        raise_flags(a.flag_word, flags);
    else if (met_nan)
    {
        const TapsArgs b = args_read_anew<TapsArgs>();
        // (its channels' weights as they lie in LDS)
        const uint8_t* w_lds = lds + taps_fixed_lds<OCT>() + 2 * b.steps * 8;
        bool odd             = false;
        for (int i = lane_counted(); i < OCB * b.chunks; i += 64)
            odd |= not_finite<T>(*reinterpret_cast<const v4i*>(w_lds + i / OCB * PITCH + i % OCB * 16));
        if (__any(odd))
        {
            __threadfence();    // (gathered rows were stored by other lanes)
            while ((pt -= pt_step) >= 0)
                sum_again<T>(b, pt * 32 + li, oc0 + 16 * lh, OCT, 16);
        }
    }
}

// Few tiles and a long reduction: a workgroup of NW waves shares a tile of 32 channels x 32 pixels (or several of pixels, one
// after the other) and splits K, both operands straight from global memory into the registers of the matrix instruction, eight
// steps at a time; the partial sums meet in LDS and the first four waves finish 4 of a lane's 16 channels each.  Where a wave's
// share is eight steps at most, its weights stay in registers from one tile of pixels to the next.  What bounds it is the CU's
// memory pipeline, two loads a step with a line per lane: 23 ns a step of the workgroup, whatever NW is.  us patch kernel / this
// kernel: int8 [1,49,49,616]->59 3x3 stride 2 77 / 11.8, [2,13,18,200]->40 5x5 stride 2 47 / 11.2, [5,24,29,8]->48 3x3 stride 2 7.4 / 4.2, fp16
// [9,31,41,240]->32 3x3 stride 2 28.9 / 8.2; with the weights staged in LDS first, as above, [2,79,7,88]->23 bf16 3x3 6.3 / 4.6.
// (Rows between words, with the words behind them: six.)
constexpr int kTapsShare = 8, kTapsOddShare = 6;

template <typename T, int NW, int ROWS>
__global__ __launch_bounds__(NW * 64, NW == 16 ? 4 : 2) void conv_taps_split_kernel(TapsArgs a)
{
    constexpr bool RAGGED = ROWS != kTapsWhole, ODD = ROWS == kTapsOdd;
    using M           = Mma<T>;
    using acc_t       = typename M::acc_t;
    using v4          = std::conditional_t<M::is_int, v4i, v4f>;
    constexpr int KSW = ODD ? kTapsOddShare : kTapsShare;    // (what the registers of two workgroups hold)
    __shared__ __attribute__((aligned(16))) v4 red[NW][4][64];
    __shared__ __attribute__((aligned(16))) HighWordScale tab_hw[32];
    __shared__ __attribute__((aligned(16))) v2i tab_ms[32];
    __shared__ __attribute__((aligned(16))) int32_t tab_start[NW + 1][32];    // per wave: its share of the starting values; the bias
    __shared__ int32_t tab_form;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 31, lh = lane >> 5;
    const int ocb = (int)fdiv(blockIdx.x, a.div_groups), grp = (int)blockIdx.x - ocb * a.groups;
    const int oc0 = ocb * 32;
    const int partial = a.row_bytes & 15;
    const int share   = (a.steps + NW - 1) / NW;
    const int s_begin = wave * share < a.steps ? wave * share : a.steps;
    const int s_end   = s_begin + share < a.steps ? s_begin + share : a.steps;

    // the lane's chunk: its offset from the window's first tap, its bit of the window's rows and columns, its place in the
    // channel vector and in the weight row
    struct Chunk
    {
        int32_t off, w_off, piece, kx, bits, index;
    };
    const int next_tap = a.dx * a.row_bytes - a.pieces * 16, next_row = (a.dy * a.IW - a.KW * a.dx) * a.row_bytes;
    auto chunk_at = [&](int c) {
        const int tap = (int)fdiv((uint32_t)c, a.div_pieces), ky = (int)fdiv((uint32_t)tap, a.div_kw);
        Chunk q;
        q.piece = c - tap * a.pieces, q.kx = tap - ky * a.KW, q.index = c;
        q.off   = (ky * a.dy * a.IW + q.kx * a.dx) * a.row_bytes + q.piece * 16;
        q.w_off = tap * a.row_bytes + q.piece * 16;
        q.bits  = (1 << ky) | (1 << (13 + q.kx));
        return q;
    };
    auto advance = [&](Chunk& q) {    // two chunks on
        q.off += 32, q.w_off += 32, q.piece += 2, q.index += 2;
        auto wrap = [&]() {
            if (q.piece >= a.pieces)
            {
                q.piece -= a.pieces, q.kx++;
                q.off += next_tap, q.w_off += a.row_bytes - a.pieces * 16;
                const int y = q.bits & 0x1fff, x = q.bits & ~0x1fff;
                const bool row_end = q.kx == a.KW;
                q.bits = row_end ? (y << 1) | (1 << 13) : y | (x << 1);
                q.off += row_end ? next_row : 0;
                q.kx = row_end ? 0 : q.kx;
            }
        };
        wrap();
        if (a.pieces == 1)
            wrap();
    };
    Chunk first_chunk = chunk_at(2 * s_begin + lh < a.chunks ? 2 * s_begin + lh : 0);
    first_chunk.index = 2 * s_begin + lh;    // (the dead half of the last step: at or behind a.chunks)

    // ---- pixels -----------------------------------------------------------------------------------------------------------
    int32_t pix_off = 0, pix_miss = -1;
    bool edge       = false;    // RAGGED: the tensor may end inside the 16 bytes of a lane of this tile
    auto enter_tile = [&](int pt) {
        int p = pt * 32 + li;
        p     = p < a.P ? p : a.P - 1;
        const int r  = (int)fdiv((uint32_t)p, a.div_ow), ox = p - r * a.OW;
        const int n  = (int)fdiv((uint32_t)r, a.div_oh), oy = r - n * a.OH;
        const int y0 = oy * a.sy - a.pad_top, x0 = ox * a.sx - a.pad_left;
        pix_off      = ((n * a.IH + y0) * a.IW + x0) * a.row_bytes;
        int in_bits  = 0;
        for (int k = 0; k < a.KH; k++)
            in_bits |= ((unsigned)(y0 + k * a.dy) < (unsigned)a.IH ? 1 : 0) << k;
        for (int k = 0; k < a.KW; k++)
            in_bits |= ((unsigned)(x0 + k * a.dx) < (unsigned)a.IW ? 1 : 0) << (13 + k);
        pix_miss = ~in_bits;
        if constexpr (RAGGED)
            edge = __any(pix_off > a.edge_off);
    };
    const int wr  = 4 * (li & 4) + ((li >> 1) & 12) + (li & 3);    // the channel of operand row li
    const int w_row = (oc0 + wr < a.OC ? oc0 + wr : a.OC - 1) * (a.KH * a.KW) * a.row_bytes;    // (rows past the end are never stored)
    v4i fa[KSW], fb[KSW];
    int fa_behind[ODD ? KSW : 1] = {}, fb_behind[ODD ? KSW : 1] = {};    // the words behind chunks that begin between words (see above)
    uint32_t fa_places = 0, fb_places = 0;
    auto load_words = [&](int d, const uint8_t* src, v4i& v, int& behind, uint32_t& places) {
        const uint32_t place = (uint32_t)(uintptr_t)src & 3u;
        const uint8_t* word  = reinterpret_cast<const uint8_t*>((uintptr_t)src & ~(uintptr_t)3);
        __builtin_memcpy(&v, __builtin_assume_aligned(word, 4), 16);
        behind = *reinterpret_cast<const int*>(word + (place ? 16 : 12));    // (never a word past the tensor)
        places |= place << (2 * d);
    };
    auto shifted = [&](int d, v4i v, int behind, uint32_t places) {
        const uint32_t by = places >> (2 * d) & 3u;
#pragma unroll
        for (int k = 0; k < 4; k++)
            v[k] = (int)__builtin_amdgcn_alignbyte((uint32_t)(k < 3 ? v[k < 3 ? k + 1 : 3] : behind), (uint32_t)v[k], by);
        return v;
    };
    auto load_pixels = [&](int d, const Chunk& q) {
        const bool inside  = q.index < a.chunks && (q.bits & pix_miss) == 0;
        const int off      = pix_off + q.off;
        const uint8_t* src = inside ? a.in + (uint32_t)off : a.pad_page;
        if constexpr (!RAGGED)
            fb[d] = *reinterpret_cast<const v4i*>(src);
        else
        {
            if (edge)
            {
                const int past = inside && off > a.last ? off - a.last : 0;
                if (__any(past))
                    fb[d] = drop_bytes(load16(src - past), past);
                else
                    fb[d] = load16(src);
            }
            else if constexpr (ODD)
                load_words(d, src, fb[d], fb_behind[d], fb_places);
            else
                fb[d] = load16(src);
        }
    };
    auto load_weights = [&](int d, const Chunk& q) {
        const int off = w_row + (q.index < a.chunks ? q.w_off : 0);
        if constexpr (!RAGGED)
            fa[d] = *reinterpret_cast<const v4i*>(a.w + (uint32_t)off);
        else
        {
            const int at = off <= a.w_last ? off : a.w_last;
            if (ODD && !__any(off > a.w_last))
                load_words(d, a.w + (uint32_t)at, fa[d], fa_behind[ODD ? d : 0], fa_places);
            else
            {
                fa[d] = load16(a.w + (uint32_t)at);
                if (__any(off > a.w_last))
                    fa[d] = drop_bytes(fa[d], off - at);
            }
        }
    };
    // what lies behind a channel vector counts for nothing, nor does the dead half of an odd count's last step
    auto trim = [&](int d, const Chunk& q, bool weights) {
        if constexpr (ODD)
        {
            fb[d] = shifted(d, fb[d], fb_behind[d], fb_places);
            if (weights)
                fa[d] = shifted(d, fa[d], fa_behind[d], fa_places);
        }
        if (RAGGED && partial && q.piece == a.pieces - 1)
        {
            if (weights)
                fa[d] = keep_bytes(fa[d], partial);
            if constexpr (!M::is_int)
                fb[d] = keep_bytes(fb[d], partial);
        }
        if (weights && q.index >= a.chunks)
            fa[d] = v4i{ 0, 0, 0, 0 };
    };

    uint32_t flags = 0;
    if (wave == NW - 1)    // (the wave whose share may be the shortest)
    {
        const int oc  = oc0 + li;
        const bool ok = oc < a.OC;
        const int occ = ok ? oc : oc0;
        if constexpr (M::is_int)
        {
            const int32_t b = reinterpret_cast<const int32_t*>(a.bias)[a.bias_len == 1 ? 0 : occ];
            if (a.rp.enabled)
            {
                const int32_t m_raw   = load_multiplier(a.rp, occ);
                const int32_t s_raw   = load_shift(a.rp, occ);
                const int32_t s_first = __builtin_amdgcn_readfirstlane(s_raw);
                const ChannelScale cs = make_channel_scale(ok ? m_raw : 0, ok ? s_raw : s_first, a.rp.double_round != 0, flags);
                const int s_min       = a.rp.double_round ? 33 : 32;
                const int form = (__all(cs.s >= s_min && cs.s <= zp_fold_max_shift(a.rp.out_zp)) ? 1 : 0) |
                                 (a.rp.lo >= a.rp.out_zp && __all(cs.m >= 0) ? 2 : 0);
                if (lh == 0)
                {
                    tab_ms[li] = v2i{ cs.m, cs.s };
                    tab_hw[li] = make_high_word_scale(cs, a.rp.out_zp);
                }
                if (lane == 0)
                    tab_form = form;
            }
            if (lh == 0)
                tab_start[NW][li] = ok ? b : 0;
        }
        else if (lh == 0)
            tab_start[NW][li] = ok ? __float_as_int(load_as_float<T>(a.bias, a.bias_len == 1 ? 0 : occ)) : 0;
    }

    const bool keep = share <= KSW;
    bool have_start = false, met_nan = false;
    int pt = grp;
    for (; pt < a.n_pt; pt += a.groups)
    {
        enter_tile(pt);
        acc_t acc;
#pragma unroll
        for (int e = 0; e < 16; e++)
            acc[e] = 0;
        int sum = 0;    // of the lane's weights
        Chunk q = first_chunk;
        const bool weights = !keep || !have_start;
        for (int s0 = s_begin; s0 < s_end; s0 += KSW)
        {
            Chunk qd  = q;
            fb_places = 0;
            if (weights)
                fa_places = 0;
#pragma unroll
            for (int d = 0; d < KSW; d++)
                if (s0 + d < s_end)
                {
                    load_pixels(d, qd);
                    if (weights)
                        load_weights(d, qd);
                    advance(qd);
                }
            if (RAGGED || s0 + KSW >= s_end)
            {
                Chunk qt = q;
#pragma unroll
                for (int d = 0; d < KSW; d++)
                    if (s0 + d < s_end)
                    {
                        trim(d, qt, weights);
                        advance(qt);
                    }
            }
            q = qd;
#pragma unroll
            for (int d = 0; d < KSW; d++)
                if (s0 + d < s_end)
                {
                    if constexpr (M::is_int)
                        if (!have_start && a.za != 0)
                            sum += dot4_ones(fa[d]);
                    acc = M::mma(fa[d], fb[d], acc);
                }
        }
        if constexpr (M::is_int)
            if (a.za != 0)
            {
                // the wave's share of -input_zp * sum(w), for the 16 channels of the lane's results
                if (!have_start)
                {
                    sum += __builtin_amdgcn_ds_bpermute((lane ^ 32) * 4, sum);
                    if (lh == 0)
                        tab_start[wave][wr] = (int32_t)(0u - (uint32_t)a.za * (uint32_t)sum);
                    __builtin_amdgcn_wave_barrier();    // the wave's own LDS accesses complete in order
                }
#pragma unroll
                for (int g = 0; g < 4; g++)
                {
                    const v4i b = *reinterpret_cast<const v4i*>(&tab_start[wave][16 * lh + 4 * g]);
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        acc[4 * g + e] += b[e];
                }
            }
        have_start = true;
#pragma unroll
        for (int g = 0; g < 4; g++)
            red[wave][g][lane] = v4{ acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3] };
        __syncthreads();    // (also publishes the tables)
        if (wave < 4)
        {
            v4 total = red[0][wave][lane];
#pragma unroll NW == 16 ? 5 : NW
            for (int w2 = 1; w2 < NW; w2++)
                total += red[w2][wave][lane];
            const int cb = 16 * lh + 4 * wave;
            if constexpr (M::is_int)
                total += *reinterpret_cast<const v4i*>(&tab_start[NW][cb]);
            if constexpr (!M::is_int)
                met_nan |= any_nan<4>(total);
            finish_taps<T, 4>(a, TapsTables{ tab_hw, tab_ms, tab_start[NW], &tab_form }, total, oc0 + cb, cb, pt * 32 + li, flags);
        }
        if (pt + a.groups < a.n_pt)
            __syncthreads();    // (the same for every wave)
    }
    if constexpr (M::is_int)
        raise_flags(a.flag_word, flags);
    else if (met_nan)
    {
        const TapsArgs b = args_read_anew<TapsArgs>();
        if (odd_weights<T>(b, oc0 + 4 * wave, 4) || odd_weights<T>(b, oc0 + 16 + 4 * wave, 4))
            while ((pt -= b.groups) >= 0)
                sum_again<T>(b, pt * 32 + li, oc0 + 16 * lh + 4 * wave, 1, 4);
    }
}

// Workgroups: as many as the CUs hold at once.  (Neighbours walk one tile more or less, and neighbours lie on different CUs; fewer
// workgroups with the same number of tiles each leave CUs with two of them beside CUs with three.)
static bool taps_grid(TapsArgs& a, int oct, int64_t wanted, int resident, unsigned& grid)
{
    a.n_ocb            = (a.OC + 32 * oct - 1) / (32 * oct);
    const int64_t most = 256 * resident / a.n_ocb > 0 ? 256 * resident / a.n_ocb : 1;
    a.groups           = (int32_t)(wanted < most ? wanted : most);
    a.div_groups       = make_fastdiv((uint32_t)a.groups);
    const int64_t all  = (int64_t)a.groups * a.n_ocb;
    grid               = (unsigned)all;
    return all <= (1 << 24) && fastdiv_exact_up_to((uint64_t)all, (uint32_t)a.groups);
}

template <typename T, int OCT, int ROWS>
static bool launch_taps(hipStream_t st, TapsArgs& a)
{
    // results whose rows are no whole words and all of one workgroup
    a.rows_bytes           = (a.OC & 3) && a.OC <= 32 * OCT && a.out_kind != 0 ? 32 * a.OC * (a.out_kind == 1 ? 1 : 2) : 0;
    const size_t lds_bytes = (size_t)taps_lds_bytes<OCT>(a.steps) + kTapsWaves * a.rows_bytes;
    constexpr auto kern    = conv_taps_kernel<T, OCT, ROWS>;
    unsigned grid;
    if (!ensure_dynamic_lds<kern>(lds_bytes) ||
        !taps_grid(a, OCT, (a.n_pt + kTapsWaves - 1) / kTapsWaves, lds_bytes > 80 * 1024 ? 1 : (lds_bytes > 53 * 1024 ? 2 : 3), grid))
        return false;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(kTapsWaves * 64), lds_bytes, st, a);
    return true;
}

template <typename T, int NW, int ROWS>
static bool launch_taps_split(hipStream_t st, TapsArgs& a)
{
    unsigned grid;
    if (!taps_grid(a, 1, a.n_pt, NW == 4 ? 3 : (NW == 8 ? 2 : 1), grid))
        return false;
    hipLaunchKernelGGL((conv_taps_split_kernel<T, NW, ROWS>), dim3(grid), dim3(NW * 64), 0, st, a);
    return true;
}

// How a layer is run: waves that share a tile's reduction (split), or channel tiles a wave owns (oct).  us is what the form takes, from
// a fit to 280 layers (int8, fp16, bf16; rms 12 % split, 15 % not).  A workgroup of the split form spends 3.4 us on launch, first
// loads and the exchange and 23 ns a step, whatever its waves (two loads a step on the CU's one memory pipeline; 100 ns where
// channel vectors start on odd addresses); the other form 4.2 us on its weights and first pixels and, a wave alone
// on its SIMD, 100 ns a step of each tile it walks, less when others fill in.
struct TapsForm
{
    int32_t oct, split;    // split 0: the form with resident weights
    double us;
};
// rows: 0 whole chunks, 1 whole words, 2 any, 3 any and read from the word before, of which a wave holds kTapsOddShare steps
static int taps_rows(int64_t row)
{
    return row % 16 == 0 ? 0 : (row % 4 == 0 ? 1 : (row <= 32 ? 2 : 3));
}
static TapsForm taps_form(int64_t n_pt, int64_t oc, int64_t steps, int rows)
{
    const int odd = rows < 3 ? rows : 2;
    static const double split_base[3] = { 3.3, 3.8, 3.5 }, split_step[3] = { 0.0235, 0.038, 0.1 }, split_all[3] = { 0.035, 0.037, 0.053 };
    static const double base[3] = { 4.5, 4.6, 4.9 }, weights[3] = { 0.018, 0.078, 0.08 }, chain[3] = { 0.0, 0.06, 0.05 }, step[3] = { 0.047, 0.045, 0.085 },
                        tile[3] = { 0.028, 0.008, 0.008 };
    const int64_t tiles_oc = (oc + 31) / 32, tiles = n_pt * tiles_oc;
    TapsForm best{ 0, 0, 1e9 };
    for (int nw = 4; nw <= 16; nw *= 2)
    {
        const int64_t most = 256 * (nw == 4 ? 3 : (nw == 8 ? 2 : 1));
        const int64_t each = (tiles + most - 1) / most;
        double us          = split_base[odd] + (nw == 4 ? (steps > 32 ? 0.4 : 0.0) : (nw == 8 ? 0.1 : 0.3)) + split_step[odd] * (double)steps +
                          split_all[odd] * (double)(tiles * steps) / 256 * (nw == 16 ? 0.9 : 1.0) + 1.4 * (double)(each - 1);
        // A share of seven or eight steps of rows read from the word before is fetched and shifted again for every tile.  us so / with weights in LDS: 1x1
        // int8 [5,32,33,939]->200 19.8 / 16.5, [9,31,32,823]->99 18.7 / 17.5, [9,31,30,945]->128 17.9 / 16.3; up to two tiles of channels, where many workgroups
        // would lay the same weights out, it stays: [35,32,32,930]->24 18.3 / 23.7, fp16 [35,32,32,491]->9 16.0 / 22.5, bf16 [35,32,32,455]->14 16.1 / 20.9.
        const int64_t share = (steps + nw - 1) / nw;
        if (rows == 3 && each > 1 && tiles_oc > 2 && share > kTapsOddShare && share <= kTapsShare)
            us += 2.0;
        if (us < best.us)
            best = TapsForm{ 1, nw, us };
    }
    for (int oct = 1; oct <= 4; oct++)
    {
        const int64_t lds = oct == 1 ? taps_lds_bytes<1>((int)steps) : (oct == 2 ? taps_lds_bytes<2>((int)steps) : (oct == 3 ? taps_lds_bytes<3>((int)steps) : taps_lds_bytes<4>((int)steps)));
        if (lds > 128 * 1024 || (oct > 1 && 32 * (oct - 1) >= oc))
            break;
        const int64_t blocks = (tiles_oc + oct - 1) / oct, wanted = (n_pt + 3) / 4 * blocks;    // channel blocks, rounds of four tiles
        const int64_t held   = lds > 80 * 1024 ? 1 : (lds > 53 * 1024 ? 2 : 3), busy = (wanted + 255) / 256 < held ? (wanted + 255) / 256 : held;
        const double rounds  = (double)((wanted + 255) / 256);    // per CU
        const double us      = base[odd] + weights[odd] * (double)(steps * oct) + rounds * (double)steps * (chain[odd] / (double)busy + step[odd] + tile[odd] * oct) +
                          0.43 * rounds * oct;
        if (us < best.us)
            best = TapsForm{ oct, 0, us };
    }
    return best;
}

static int64_t taps_steps(int64_t taps, int64_t row)
{
    return (taps * ((row + 15) / 16) + 1) / 2;
}

double conv2d_taps_us(int32_t in_dtype, const ConvGeom& g)
{
    const int64_t row = (int64_t)g.IC * (in_dtype == TMI_INT8 ? 1 : 2), steps = taps_steps((int64_t)g.KH * g.KW, row);
    return taps_form(((int64_t)g.N * g.OH * g.OW + 31) / 32, g.OC, steps, taps_rows(row)).us;
}

template <typename T>
static bool launch_taps_t(hipStream_t st, TapsArgs& a, bool ragged)
{
    const TapsForm form = taps_form(a.n_pt, a.OC, a.steps, !ragged ? 0 : (a.row_bytes % 4 == 0 ? 1 : taps_rows(a.row_bytes)));
    // (up to 32 bytes a pixel, neighbouring pixels share lines and the other loads are no slower: [20,136,133,13]->488 3x3 stride 2 52.0 / 38.3,
    // [5,14,14,30]->16 5x5 6.6 / 6.0)
    const bool odd = a.row_bytes > 32 && (a.row_bytes % 4 != 0 || (((uintptr_t)a.in | (uintptr_t)a.w) & 3));
    if (odd)
        a.edge_off -= 4;    // (the word behind)
#define TMI_TAPS(O)                                                                                                   \
    if (!form.split && form.oct == O)                                                                                 \
        return !ragged ? launch_taps<T, O, kTapsWhole>(st, a) : (odd ? launch_taps<T, O, kTapsOdd>(st, a) : launch_taps<T, O, kTapsWords>(st, a));
    TMI_TAPS(1)
    TMI_TAPS(2)
    TMI_TAPS(3)
    TMI_TAPS(4)
#undef TMI_TAPS
#define TMI_TAPS(NW)                                                                                                  \
    if (form.split == NW)                                                                                             \
        return !ragged ? launch_taps_split<T, NW, kTapsWhole>(st, a) : (odd ? launch_taps_split<T, NW, kTapsOdd>(st, a) : launch_taps_split<T, NW, kTapsWords>(st, a));
    TMI_TAPS(4)
    TMI_TAPS(8)
    TMI_TAPS(16)
#undef TMI_TAPS
    return false;
}

// the results by out_kind, -1: none of this kernel's
static int taps_kind(int32_t in_dtype, int32_t out_dtype, const RescaleParams& rp)
{
    if (in_dtype == TMI_INT8)
        return !rp.enabled ? (out_dtype == TMI_INT32 ? 0 : -1) : (!rp.fast ? -1 : (out_dtype == TMI_INT8 ? 1 : (out_dtype == TMI_INT16 ? 2 : -1)));
    return (in_dtype == TMI_FP16 || in_dtype == TMI_BF16) && !rp.enabled && out_dtype == in_dtype ? 3 : -1;
}
static int64_t taps_window(const ConvGeom& g, int64_t row)    // the last chunk's offset from its window's first tap
{
    return ((int64_t)(g.KH - 1) * g.dil_y * g.IW + (int64_t)(g.KW - 1) * g.dil_x) * row + (row - 1) / 16 * 16;
}
bool conv2d_taps_takes(int32_t in_dtype, int32_t out_dtype, const ConvGeom& g, int32_t w_zp, const RescaleParams& rp, const void* out)
{
    if (w_zp != 0 || g.KH > 13 || g.KW > 13 || taps_kind(in_dtype, out_dtype, rp) < 0 || ((uintptr_t)out & 15))
        return false;
    const int64_t P        = (int64_t)g.N * g.OH * g.OW, row = (int64_t)g.IC * (in_dtype == TMI_INT8 ? 1 : 2), taps = (int64_t)g.KH * g.KW;
    const int64_t in_bytes = (int64_t)g.N * g.IH * g.IW * row, w_bytes = (int64_t)g.OC * taps * row, chunks = taps * ((row + 15) / 16);
    // 32-bit offsets (a window's first tap may lie before the tensor)
    if (P < 1 || g.OC < 1 || P > (1 << 30) || in_bytes < 16 || w_bytes < 16 || in_bytes >= (int64_t(1) << 30) || w_bytes >= (int64_t(1) << 30) ||
        (int64_t)(g.pad_top + 1) * g.IW * row >= (int64_t(1) << 30) || (int64_t)g.pad_left * row >= (int64_t(1) << 29) ||
        taps_window(g, row) >= (int64_t(1) << 30) || taps_steps(taps, row) > 1024)
        return false;
    return fastdiv_exact_up_to((uint64_t)P, (uint32_t)g.OW) && fastdiv_exact_up_to((uint64_t)P / g.OW + 1, (uint32_t)g.OH) &&
           fastdiv_exact_up_to((uint64_t)128 * chunks, (uint32_t)chunks);
}

const char* launch_conv2d_taps(hipStream_t st, int32_t in_dtype, int32_t out_dtype, const ConvGeom& g, const void* in, const void* w,
                               const void* bias, int32_t in_zp, int32_t w_zp, const RescaleParams& rp, void* out, const void* pad_page,
                               uint32_t* flag_word)
{
    if (!flag_word || !pad_page || !conv2d_taps_takes(in_dtype, out_dtype, g, w_zp, rp, out))
        return nullptr;
    const bool i8          = in_dtype == TMI_INT8;
    const int kind         = taps_kind(in_dtype, out_dtype, rp);
    const int64_t P        = (int64_t)g.N * g.OH * g.OW, row = (int64_t)g.IC * (i8 ? 1 : 2), taps = (int64_t)g.KH * g.KW;
    const int64_t in_bytes = (int64_t)g.N * g.IH * g.IW * row, w_bytes = (int64_t)g.OC * taps * row, window = taps_window(g, row);
    const int64_t pieces = (row + 15) / 16, chunks = taps * pieces;
    TapsArgs a{};
    a.steps = (int32_t)taps_steps(taps, row);
    a.in = (const uint8_t*)in, a.w = (const uint8_t*)w, a.bias = bias, a.out = out, a.pad_page = (const uint8_t*)pad_page;
    a.flag_word = flag_word, a.rp = rp;
    a.P = (int32_t)P, a.OC = g.OC, a.OH = g.OH, a.OW = g.OW, a.IH = g.IH, a.IW = g.IW, a.KH = g.KH, a.KW = g.KW;
    a.sy = g.stride_y, a.sx = g.stride_x, a.dy = g.dil_y, a.dx = g.dil_x, a.pad_top = g.pad_top, a.pad_left = g.pad_left;
    a.row_bytes = (int32_t)row, a.pieces = (int32_t)pieces, a.chunks = (int32_t)chunks;
    a.za = in_zp, a.bias_len = g.bias_len, a.out_kind = kind;
    a.n_pt = (int32_t)((P + 31) / 32);
    a.last = (int32_t)(in_bytes - 16), a.edge_off = (int32_t)(in_bytes - 16 - window), a.w_last = (int32_t)(w_bytes - 16);
    a.div_ow = make_fastdiv((uint32_t)g.OW), a.div_oh = make_fastdiv((uint32_t)g.OH), a.div_chunks = make_fastdiv((uint32_t)chunks);
    a.row_skip = (int32_t)(kTapsWaves * 64 / chunks), a.chunk_skip = (int32_t)(kTapsWaves * 64 % chunks);
    a.div_pieces = make_fastdiv((uint32_t)pieces), a.div_kw = make_fastdiv((uint32_t)g.KW);
    const bool ragged = row % 16 != 0 || (((uintptr_t)in | (uintptr_t)w) & 15);
    const bool ok     = i8 ? launch_taps_t<int8_t>(st, a, ragged)
                           : (in_dtype == TMI_FP16 ? launch_taps_t<_Float16>(st, a, ragged) : launch_taps_t<bf16_t>(st, a, ragged));
    return !ok ? nullptr : (i8 ? (rp.enabled ? "conv2d_taps_i8_rescale" : "conv2d_taps_i8") : (in_dtype == TMI_FP16 ? "conv2d_taps_f16" : "conv2d_taps_bf16"));
}

}    // namespace tmi
