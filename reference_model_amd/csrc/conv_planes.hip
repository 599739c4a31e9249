// CONV2D with taps on 16-bit floats, or on int8 with the fused RESCALE, whose input patch streams through LDS, 128 bytes of channels at a time.
//
// A workgroup of 8 waves owns 64 output channels x IT * 128 pixels, whole output rows of one image.  K is walked in stages of one tap and 128 bytes of
// channels, all taps of a slice of channels before the next slice: the slice's patch (with its halo) lies in one of two buffers, loaded
// under the taps of the slice before, and a stage's 64 weight rows, whole lines, pass through a ring of eight.  Both go straight into LDS, one barrier a
// stage.  Two groups of four waves take half of a stage's channels each, so that a wave owns 64 channels x IT * 32 pixels and reads four (IT 1: three)
// fragments for four (two) matrix instructions; after the loop a wave hands half of its sums to its partner.
//
// What bounds it: on few tiles the instructions of a stage (0.21 us, of which its matrix instructions are 0.11; with 256 pixels 0.41 and 0.21), on all CUs the clock under the
// matrix instructions: [16,28,28,256]->256 3x3 14.9 us without any operand in the loop, 18.8 with its fragment reads.  A wave's loads straight into LDS go
// one after the other, 0.3 us each, so the second group fetches the patch through registers (all loads straight into LDS: 26.2, so 21.5), in a loop of its own,
// or the compiler has the first group wait for them too (28.9).
// us before / here: [16,14,14,512]->512 40.0 / 23.9, [16,28,28,256]->64 20.7 / 13.0, 5x5 [2,20,20,480]->592 129 / 51, stride 2 [14,36,28,328]->240 46.6 / 22.2.
#include <type_traits>

#include "outside_taps.h"

namespace tmi
{

struct PlanesArgs
{
    const uint8_t *x, *w, *pad_page, *zeros;    // pad_page: 16 bytes of the input's zero point; 16 zero bytes
    const void* bias;
    void* out;
    int32_t N;                   // output channels, a multiple of 8
    int32_t kb, icb;             // bytes of a weight row, of a channel vector (multiples of 16)
    int32_t slices, taps, KW;    // of 128 bytes
    int32_t IH, IW, OH, OW;
    int32_t sy, sx, dy, dx, pad_top, pad_left;
    int32_t bias_len;
    int32_t rows;                      // output rows of a tile
    int32_t patch_w, patch_pixels;
    int32_t buffer_bytes;              // of a slice's patch in LDS
    int32_t tiles, per_xcd;
    FastDiv tiles_n, tiles_image, div_pw, div_ow;
    int32_t padded;         // a tap can fall outside the image
    int32_t za;             // int8: the input's zero point; the weights' is 0
    RescaleParams rp;
    uint32_t* flag_word;    // where its REQUIRE conditions are latched
};

static constexpr int kPlanesRing = 8, kPlanesLoads = 12;    // stages of weights; KB of a slice's patch a wave fetches at most
static constexpr int kPlanesPatches = 160 * 1024 - kPlanesRing * 8192 - 256 - 64 * 32;    // LDS for the two patches, beside the tables

// 16-byte chunk c of a 128-byte row lies at c ^ key(row): the lanes the LDS serves in one cycle read one chunk of rows whose (row / 2) % 8 differ
// or that lie in the two halves of the banks (no conflict for any 32 consecutive rows, nor for the weights' order).  A patch pixel's key is that of
// its row * OW + column: consecutive outputs read consecutive ones, past the halo between two rows too.
__device__ __forceinline__ int planes_key(int row)
{
    return (row >> 1) & 7;
}

template <typename T, int IT>
__global__ __launch_bounds__(512) void conv_planes_kernel(PlanesArgs a)
{
    constexpr int D = kPlanesRing, STAGE = 64 * 128;
    constexpr bool I8 = Mma<T>::is_int;
    using word_t      = std::conditional_t<I8, int, float>;
    using word4_t     = std::conditional_t<I8, v4i, v4f>;
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const int lane = threadIdx.x & 63, rho = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int kg = wave >> 2, wq = wave & 3;    // half of a stage's channels, pixel tiles

    // a contiguous range of tiles for each of the eight L2s; those of the same pixels are neighbours
    const int L = (blockIdx.x & 7) * a.per_xcd + (blockIdx.x >> 3);
    if (L >= a.tiles)
        return;
    const uint32_t tm = fdiv((uint32_t)L, a.tiles_n), tn = (uint32_t)L - tm * a.tiles_n.d;
    const uint32_t image = fdiv(tm, a.tiles_image);
    const int oy0 = (int)(tm - image * a.tiles_image.d) * a.rows, oc0 = (int)tn * 64;
    const int rows_here = a.OH - oy0 < a.rows ? a.OH - oy0 : a.rows, pixels = rows_here * a.OW;
    const uint8_t* x = a.x + (size_t)image * a.IH * a.IW * a.icb;

    // ---- loads: 64 lanes move eight rows of 128 bytes ---------------------------------------------------------
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
    // the first group of waves: weights, two of a stage's eight loads each
    uint32_t w_off[2];
    int w_at[2];    // of the lane's chunk
#pragma unroll
    for (int q = 0; q < 2; q++)
    {
        const int row = (2 * wq + q) * 8 + (lane >> 3), oc = oc0 + row < a.N ? oc0 + row : a.N - 1;    // (rows past the last are not stored)
        w_at[q]  = ((lane & 7) ^ planes_key(row)) * 16;
        w_off[q] = (uint32_t)oc * (uint32_t)a.kb + (uint32_t)w_at[q];
    }
    const int whole = a.icb >> 7;    // slices of 128 bytes
    int l_tap = 0, l_slice = 0;      // the next stage whose weights are requested; past the end the last slice again, which nobody reads
    const uint8_t* l_base = a.w;
    const uint32_t w_dst = lds0 + wq * 2048;
    auto load_weights = [&](int slot_at) {
        const uint32_t dst = w_dst + slot_at;
        if (l_slice < whole)
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %3\n\ts_add_u32 m0, %2, 1024\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %3"
                         :
                         : "v"(w_off[0]), "v"(w_off[1]), "s"(dst), "s"(l_base)
                         : "memory", "scc");
        else    // (a slice of fewer than 128 bytes: zeros for the others)
        {
#pragma unroll
            for (int q = 0; q < 2; q++)
            {
                const uint8_t* src = l_slice * 128 + w_at[q] < a.icb ? l_base + w_off[q] : a.zeros;
                asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(src), "s"(dst + 1024 * q) : "memory");
            }
        }
        l_base += a.icb;
        if (++l_tap == a.taps)
        {
            l_tap   = 0;
            l_slice = l_slice + 1 < a.slices ? l_slice + 1 : l_slice;
            l_base  = a.w + l_slice * 128;
        }
    };
    // the second group: the patch, through registers (a wave's loads straight into LDS go one after the other, these are in flight together)
    const int iy0 = oy0 * a.sy - a.pad_top;
    v4i held[kPlanesLoads];
    auto fetch_patch = [&](int slice) {
#pragma unroll
        for (int j = 0; j < kPlanesLoads; j++)
        {
            const int u = (j * 4 + wq) * 8;    // the wave's first pixel
            if (u >= a.patch_pixels)
                break;
            const int pix = u + (lane >> 3), r = (int)fdiv((uint32_t)pix, a.div_pw), c = pix - r * a.patch_w;
            const int iy = iy0 + r, ix = c - a.pad_left, at = slice * 128 + (((lane & 7) ^ planes_key(r * a.OW + c)) * 16);
            const bool there   = (uint32_t)iy < (uint32_t)a.IH && (uint32_t)ix < (uint32_t)a.IW && at < a.icb && pix < a.patch_pixels;
            const uint8_t* src = there ? x + (uint32_t)((iy * a.IW + ix) * a.icb + at) : a.pad_page;
            held[j]            = *reinterpret_cast<const v4i*>(src);
        }
    };
    auto store_patch = [&](int slice) {
        uint8_t* to = lds + D * STAGE + (slice & 1) * a.buffer_bytes + wq * 1024 + lane * 16;
#pragma unroll
        for (int j = 0; j < kPlanesLoads; j++)
        {
            if ((j * 4 + wq) * 8 >= a.patch_pixels)
                break;
            *reinterpret_cast<v4i*>(to + j * 4096) = held[j];
        }
    };
    word_t* tab_bias     = reinterpret_cast<word_t*>(lds + D * STAGE + 2 * a.buffer_bytes);
    ChannelScale* tab_cs = reinterpret_cast<ChannelScale*>(tab_bias + 64);
    uint32_t flags       = 0;
    if (threadIdx.x < 64)
    {
        const bool ok = oc0 + (int)threadIdx.x < a.N;
        const int oc  = ok ? oc0 + (int)threadIdx.x : a.N - 1;
        if constexpr (I8)
        {
            tab_bias[threadIdx.x] = reinterpret_cast<const int32_t*>(a.bias)[a.bias_len == 1 ? 0 : oc];
            const int32_t m = load_multiplier(a.rp, oc), sh = load_shift(a.rp, oc);    // (channels past the end: neutral constants, nothing raised)
            tab_cs[threadIdx.x] = make_channel_scale(ok ? m : 0, ok ? sh : 32, a.rp.double_round != 0, flags);
        }
        else
            tab_bias[threadIdx.x] = load_as_float<T>(a.bias, a.bias_len == 1 ? 0 : oc);
    }
    if (kg)
    {
        fetch_patch(0);
        store_patch(0);
    }
    else
    {
#pragma unroll
        for (int s = 0; s < D - 1; s++)
            load_weights(s * STAGE);
    }

    // ---- fragments --------------------------------------------------------------------------------------------
    // Tile i of the wave is the workgroup's pixel tile wq * IT + (i ^ kg): the one it stores (IT 2) first.
    const int w_frag = channel_of_row(rho);
    const uint32_t aw0 = (uint32_t)(w_frag * 128 + (((4 * kg + h) ^ planes_key(w_frag)) * 16));
    uint32_t pbase[IT];    // byte of the patch under the first tap, and its position for the key
    int pkey[IT];
#pragma unroll
    for (int i = 0; i < IT; i++)
    {
        int p = (wq * IT + (IT == 2 ? i ^ kg : 0)) * 32 + rho;
        p     = p < pixels ? p : 0;    // (not stored)
        const int py = (int)fdiv((uint32_t)p, a.div_ow);
        pbase[i]     = (uint32_t)(py * a.sy * a.patch_w + (p - py * a.OW) * a.sx) * 128u;
        pkey[i]      = py * a.sy * a.OW + (p - py * a.OW) * a.sx;
    }
    // Where the stage read next lies: its weights, its tap in the slice's patch (byte and position).  Scalars that go on by additions: a stage of few tiles is
    // as long as its instructions.
    const int dx_at = a.dx * 128, row_at = (a.dy * a.patch_w - a.KW * a.dx) * 128, row_key = a.dy * a.OW - a.KW * a.dx;
    uint32_t aw = aw0, ap[IT], w_at_stage = 0, patch_at = D * STAGE, tap_at = patch_at;
    int taps_left = a.taps, kx_left = a.KW, tap_key = 0;
    auto address = [&](int i) {    // of pixel tile i; of the weights
        if (i == IT)
            aw = aw0 + w_at_stage;
        else
            ap[i] = pbase[i] + tap_at + (uint32_t)(((4 * kg + h) ^ planes_key(pkey[i] + tap_key)) << 4);
    };
    auto next_stage = [&]() {
        w_at_stage = (w_at_stage + STAGE) & (D * STAGE - 1);
        tap_at += dx_at, tap_key += a.dx;
        if (--kx_left == 0)
            kx_left = a.KW, tap_at += row_at, tap_key += row_key;
        if (--taps_left == 0)
        {
            patch_at  = 2 * D * STAGE + (uint32_t)a.buffer_bytes - patch_at;    // the other buffer
            taps_left = a.taps, tap_at = patch_at, tap_key = 0;
        }
    };
    using acc_t = typename Mma<T>::acc_t;
    acc_t acc[IT][2];
#pragma unroll
    for (int i = 0; i < IT; i++)
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int e = 0; e < 16; e++)
                acc[i][t][e] = 0;
    v4i fa[2][2], fb[2][IT];
    auto read_one = [&](int s, int j) {    // j: pixel tile 0, channel tile 0, the others
        if (j == 0 || (IT == 2 && j == 2))
            fb[s][j >> 1] = *reinterpret_cast<const v4i*>(lds + (ap[j >> 1] ^ (32 * s)));
        else
            fa[s][j == 1 ? 0 : 1] = *reinterpret_cast<const v4i*>(lds + (aw ^ (32 * s)) + (j == 1 ? 0 : 4096));
    };
    constexpr int NM = 2 * IT, NR = 2 + IT;
    // int8, sum((x - za) w) = sum(x w) - za sum(w): of the four waves that read the same weights each adds up one channel tile of one step
    int wsum            = 0;
    const int sums_step = I8 && a.za != 0 ? wq >> 1 : -1;
    // Step S; behind its instructions the requests for the next step's fragments and what `behind` does there.
    auto multiply = [&](auto S_tag, auto&& behind) {
        constexpr int S = decltype(S_tag)::value;
        if constexpr (I8)
            if (sums_step == S)
            {
                if (wq & 1)
                    wsum += dot4_ones(fa[S][1]);
                else
                    wsum += dot4_ones(fa[S][0]);
            }
#pragma unroll
        for (int k = 0; k < NM; k++)
        {
            const int t = k / IT, i = t & 1 ? IT - 1 - k % IT : k % IT;
            acc[i][t]   = Mma<T>::mma(fa[S][t], fb[S][i], acc[i][t]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < NR; j++)
                if (j * (NM - 1) / NR == k)
                    read_one(1 - S, j);
            behind(k);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // the patch and the first stage
    if (kg)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    else
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(2 * (D - 2)) : "memory");
    asm volatile("s_barrier" ::: "memory");
#pragma unroll
    for (int i = 0; i <= IT; i++)
        address(i);
#pragma unroll
    for (int j = 0; j < NR; j++)
        read_one(0, j);

    // One stage: its first step, the barrier behind which the next stage is there and every wave is past the one before this, its second.
    auto stage = [&](auto&& wait, auto&& loads) {
        multiply(std::integral_constant<int, 0>{}, [&](int k) {
            if (k == NM - 1)
            {
                // (every request of this step's fragments is out)
                next_stage();
#pragma unroll
                for (int i = 0; i <= IT; i++)
                    address(i);
            }
        });
        wait();
        asm volatile("s_barrier" ::: "memory");
        multiply(std::integral_constant<int, 1>{}, [&](int k) {
            if (k == 0)
                loads();
        });
    };
    auto none = []() {};
    // (a loop for each group: the compiler would have the one with loads to wait for also wait in the other's place)
    if (!kg)
    {
        // the next stage's weights, with those of D - 3 later ones on their way
        int free_slot = (D - 1) * STAGE;
#pragma unroll 1
        for (int s = a.slices * a.taps; s > 0; s--)
            stage([]() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * (D - 3)) : "memory"); },
                  [&]() {
                      load_weights(free_slot);
                      free_slot = (free_slot + STAGE) & (D * STAGE - 1);
                  });
    }
    else
    {
        // the next slice's patch: fetched in the first stage of a slice, stored in the last but one
#pragma unroll 1
        for (int next = 1; next < a.slices; next++)
        {
            stage(none, [&]() { fetch_patch(next); });
#pragma unroll 1
            for (int t = a.taps - 3; t > 0; t--)
                stage(none, none);
            stage(none, [&]() { store_patch(next); });
            stage([]() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }, none);
        }
#pragma unroll 1
        for (int t = a.taps; t > 0; t--)
            stage(none, none);
    }

    // ---- the other half of the channels: a wave's second pixel tile (IT 1: its channel tile 1 - kg) is its partner's ---------
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    constexpr int HT = IT == 2 ? 2 : 1;    // channel tiles a wave stores
    int* tab_wsum       = reinterpret_cast<int*>(lds + D * STAGE);    // a row of 64 words for each part
    if constexpr (I8)
    {
        const int both = wsum + __shfl_xor(wsum, 32);
        if (h == 0)
            tab_wsum[(2 * kg + (wq >> 1)) * 64 + (wq & 1) * 32 + channel_of_row(rho)] = both;
    }
    uint8_t* give       = lds + wave * (HT * 4096) + lane * 16;
    const uint8_t* take = lds + (wave ^ 4) * (HT * 4096) + lane * 16;
#pragma unroll
    for (int t = 0; t < HT; t++)
#pragma unroll
        for (int q = 0; q < 4; q++)
        {
            word4_t v;
#pragma unroll
            for (int e = 0; e < 4; e++)
                v[e] = IT == 2 ? acc[IT - 1][t][4 * q + e] : (kg ? acc[0][0][4 * q + e] : acc[0][1][4 * q + e]);
            *reinterpret_cast<word4_t*>(give + (t * 4 + q) * 1024) = v;
        }
    __syncthreads();
    word_t sum[HT][16];
#pragma unroll
    for (int t = 0; t < HT; t++)
#pragma unroll
        for (int q = 0; q < 4; q++)
        {
            const word4_t v = *reinterpret_cast<const word4_t*>(take + (t * 4 + q) * 1024);
#pragma unroll
            for (int e = 0; e < 4; e++)
                sum[t][4 * q + e] = v[e] + (IT == 2 ? acc[0][t][4 * q + e] : (kg ? acc[0][1][4 * q + e] : acc[0][0][4 * q + e]));
        }
    float largest = 0.0f;    // (see outside_taps.h)
    if constexpr (!I8)
        if (a.padded)
#pragma unroll
            for (int t = 0; t < HT; t++)
                largest = largest_or_nan<16>(largest, sum[t]);
    __syncthreads();

    // ---- results: gathered by pixel, so that whole lines leave ----------------------------------------------------
    constexpr int EB = (int)sizeof(T), ROW = HT * 32 * EB, PITCH = ROW + 16;
    uint8_t* tbuf = lds + wave * (32 * PITCH);
    const int oc_w = oc0 + (IT == 2 ? 0 : 32 * kg), p_w = (IT == 2 ? wq * 2 + kg : wq) * 32;
#pragma unroll
    for (int t = 0; t < HT; t++)
    {
        const int at = oc_w - oc0 + 32 * t + 16 * h;    // the lane's channels
        alignas(16) T packed[16];
        if constexpr (I8)
        {
            if (p_w + rho < pixels && oc0 + at < a.N)
            {
                v4i out;
#pragma unroll
                for (int q = 0; q < 4; q++)
                {
                    v4i b = *reinterpret_cast<const v4i*>(tab_bias + at + 4 * q);
                    if (a.za != 0)
                    {
                        v4i ws = *reinterpret_cast<const v4i*>(tab_wsum + at + 4 * q);
#pragma unroll
                        for (int part = 1; part < 4; part++)
                            ws += *reinterpret_cast<const v4i*>(tab_wsum + part * 64 + at + 4 * q);
                        b -= a.za * ws;
                    }
                    int word = 0;
#pragma unroll
                    for (int e = 0; e < 4; e++)
                    {
                        const ChannelScale cs = tab_cs[at + 4 * q + e];
                        word |= (fast_rescale(sum[t][4 * q + e] + b[e], cs, a.rp.out_zp, a.rp.lo, a.rp.hi, flags) & 0xff) << (8 * e);
                    }
                    out[q] = word;
                }
                *reinterpret_cast<v4i*>(tbuf + rho * PITCH + t * 32 + h * 16) = out;
            }
        }
        else
        {
#pragma unroll
            for (int q = 0; q < 4; q++)
            {
                const v4f b = *reinterpret_cast<const v4f*>(tab_bias + at + 4 * q);
#pragma unroll
                for (int e = 0; e < 4; e++)
                    store_from_float(packed + 4 * q + e, sum[t][4 * q + e] + b[e]);
            }
            uint8_t* d = tbuf + rho * PITCH + t * 64 + h * 32;
            reinterpret_cast<v4i*>(d)[0] = reinterpret_cast<const v4i*>(packed)[0];
            reinterpret_cast<v4i*>(d)[1] = reinterpret_cast<const v4i*>(packed)[1];
        }
    }
    // (pieces of eight channels)
    using piece_t        = std::conditional_t<I8, v2i, v4i>;
    constexpr int PIECES = ROW / (8 * EB), RPI = 64 / PIECES;
    uint8_t* to = reinterpret_cast<uint8_t*>(a.out) + (((size_t)(image * a.OH + oy0) * a.OW + p_w) * a.N + oc_w) * EB;
#pragma unroll
    for (int j = 0; j < 32 / RPI; j++)
    {
        const int row   = lane / PIECES + RPI * j, piece = lane % PIECES;
        const piece_t d = *reinterpret_cast<const piece_t*>(tbuf + row * PITCH + piece * 8 * EB);
        if (p_w + row < pixels && oc_w + piece * 8 < a.N)
            *reinterpret_cast<piece_t*>(to + ((size_t)row * a.N + piece * 8) * EB) = d;
    }
    if constexpr (I8)
        raise_flags(a.flag_word, flags);
    else if (a.padded)
    {
        auto weights = [&](auto&& look) {
            const PlanesArgs g = args_read_anew<PlanesArgs>();
            look(g.w + (size_t)oc0 * g.kb, (int64_t)(g.N - oc0 < 64 ? g.N - oc0 : 64) * g.kb);
        };
        if (__builtin_expect(met_odd_weights<T, 8>(largest, wave, tab_wsum, weights), 0))
        {
            __threadfence();    // (results were stored by other lanes)
            const PlanesArgs g = args_read_anew<PlanesArgs>();
            const int p = p_w + rho, py = p / g.OW;
            without_outside_taps<T>(OutsideTaps{ g.x, g.w, g.bias, g.out, g.icb, g.IH, g.IW, g.N, g.OH, g.OW, g.taps / g.KW, g.KW, g.sy, g.sx, g.dy, g.dx, g.pad_top, g.pad_left, g.bias_len },
                                    p < pixels, (int)image, oy0 + py, p - py * g.OW, oc_w + 16 * h, HT, 16);
        }
    }
}

struct PlanesPlan
{
    int32_t rows = 0;    // of a tile; 0: none
    int64_t patch_pixels, slices, tiles_image, tiles;
    double us;           // a prediction: 230 layers of 0.3 to 30 GFLOP, half of them within 5 %, nine in ten within 13 %
    bool wide;           // more than 128 pixels a tile
};

// The tile of whole output rows that takes the chip the shortest time
static PlanesPlan plan_planes(const ConvGeom& g, int eb)
{
    PlanesPlan best;
    const int64_t slices = ((int64_t)g.IC * eb + 127) / 128, taps = (int64_t)g.KH * g.KW, tn = (g.OC + 63) / 64;
    const int64_t patch_w = (int64_t)(g.OW - 1) * g.stride_x + (int64_t)(g.KW - 1) * g.dil_x + 1;
    for (int rows = 1; rows <= g.OH && (int64_t)rows * g.OW <= 256; rows++)
    {
        PlanesPlan p;
        p.rows         = rows;
        p.patch_pixels = ((int64_t)(rows - 1) * g.stride_y + (int64_t)(g.KH - 1) * g.dil_y + 1) * patch_w;
        if (p.patch_pixels > 8 * 4 * kPlanesLoads || 2 * ((p.patch_pixels + 7) / 8 * 1024) > kPlanesPatches)
            break;
        p.slices      = slices;
        p.tiles_image = (g.OH + rows - 1) / rows;
        p.tiles       = (int64_t)g.N * p.tiles_image * tn;
        p.wide        = (int64_t)rows * g.OW > 128;
        p.us          = 1.6 + (double)((p.tiles + 255) / 256) * (3.2 + (double)(slices * taps) * (p.wide ? 0.416 : 0.215) + 0.0029 * (double)(p.patch_pixels * slices));
        if (best.rows == 0 || p.us < best.us * 0.999)
            best = p;
    }
    return best;
}

static bool planes_take(int32_t in_dtype, const ConvGeom& g)
{
    const int64_t taps = (int64_t)g.KH * g.KW, icb = (int64_t)g.IC * (in_dtype == TMI_INT8 ? 1 : 2);
    return (in_dtype == TMI_FP16 || in_dtype == TMI_BF16 || in_dtype == TMI_INT8) && taps >= 3 && taps <= 64 && icb % 16 == 0 && g.OC % 8 == 0 && g.OW <= 256 && icb * taps * g.OC < INT32_MAX &&
           (int64_t)g.IH * g.IW * icb < INT32_MAX;
}

// Whether a layer runs here: one round of workgroups and 18 stages or more.  us the kernel it would go to / here, 3x3 unless noted:
//   the patch kernel (conv2d_mfma.hip): [16,28,28,256]->64 20.7 / 13.4, [26,10,22,376]->160 32.8 / 20.8, 5x5 [2,20,20,480]->592 129 / 53,
//     [11,58,21,96]->96 30.9 / 19.3, stride 2 [14,36,28,328]->240 46.9 / 22.7; over 34 of them 0.41 ... 0.96.  Two rounds: [4,29,109,136]->136 19.7 / 26.9,
//     [22,75,13,288]->144 stride 2 27.6 / 34.6; 9 stages: [20,50,50,64]->72 stride 2 11.5 / 13.3, [11,28,28,32]->104 5.9 / 7.6.
//   split reductions (conv_taps.hip), from 106 TFLOP/s predicted on: [2,18,18,384]->448 (115) 26.4 / 17.9, [2,54,54,512]->48 (107) 33.9 / 23.2, [7,14,21,200]->288 19.9 / 14.7, the least
//     gain [1,85,85,88]->96 (108) 11.5 / 11.6; below [4,14,14,448]->320 (103) 17.1 / 19.8, [3,25,25,600]->128 (98) 23.2 / 28.1, [3,14,14,512]->160 (39) 18.6 / 21.1.
//     Where the last slice is cut off (its stages choose every source) and four fifths of their last round of tiles are filled, they keep theirs: over 49 drawn layers here 1.07 of their time,
//     [9,14,61,136]->328 stride 2 (682 tiles) 11.1 / 14.5, 5x5 [11,23,8,88]->216 (448) 14.2 / 18.4, [4,47,8,144]->320 (470) 9.9 / 12.1; the most given up [6,26,42,120]->384 stride 2 (624) 14.3 / 11.7.
//     Less filled 0.88 over 55, [12,96,21,176]->96 stride 2 (594) 21.0 / 13.5; the most lost [7,16,16,208]->216 (392) 12.1 / 15.1.
//   the GEMM kernel, only with tiles of up to 128 pixels and whole slices: [14,22,22,384]->176 31.8 / 18.8, [16,14,14,512]->512 40.1 / 24.2, 5x5 [24,52,10,64]->128 15.2 / 10.6, [10,22,22,128]->296 20.7 / 17.7; else
//     [16,28,28,256]->256 (196 pixels) 20.2 / 21.5, [16,40,15,160]->136 (two and a half slices) 12.6 / 13.0.
//   int8 with RESCALE, where the patch kernel has the layer, at most a third of the slices cut off: [8,29,29,208]->248 19.8 / 13.1, [14,30,30,592]->96 30.9 / 23.1, [4,31,36,480]->240 25.7 / 19.6, 5x5
//     [18,20,20,624]->64 85 / 48; over 36 of them 0.56 ... 0.94; beyond a third [3,61,61,160]->176 19.0 / 17.8, [10,25,94,176]->64 12.7 / 13.4.  The kernels with resident weights
//     or split reductions keep theirs: of 83 layers 9 gained, [11,7,8,416]->616 10.4 / 17.8, [8,30,86,160]->128 14.4 / 18.0.
//   Up to 32 channels on tiles of more than 128 pixels, half of whose matrix instructions have no channel: the patch kernel keeps int8 and rows of less than 600 bytes.  Over 69
//     and 40 drawn layers of these here 1.07 and 1.10 of its time: int8 [21,48,48,192]->32 11.6 / 16.2, [13,34,89,192]->8 12.4 / 16.4, bf16 [16,55,55,96]->32 10.9 / 15.1, fp16
//     [9,71,71,80]->32 10.4 / 13.7; the most given up bf16 5x5 [23,35,35,128]->32 25.1 / 22.9, int8 [14,46,46,624]->16 30.3 / 28.1.  Longer rows 0.92 over 30: [31,52,22,512]->16 39.9 / 32.8.
bool conv_planes_leads(int32_t in_dtype, const ConvGeom& g, PlanesRival rival)
{
    if (!planes_take(in_dtype, g))
        return false;
    const int eb       = in_dtype == TMI_INT8 ? 1 : 2;
    const PlanesPlan p = plan_planes(g, eb);
    if (p.rows == 0 || p.tiles > 256 || p.slices * g.KH * g.KW < 18)
        return false;
    if (p.wide && g.OC <= 32 && (in_dtype == TMI_INT8 || g.IC * eb < 600))
        return false;
    if (in_dtype == TMI_INT8)
        return p.slices * 128 * 3 <= (int64_t)g.IC * 4;
    if (rival == PLANES_GEMM)
        return !p.wide && g.IC * eb % 128 == 0;
    if (p.slices == 1 && g.IC * eb < 128)    // (a slice cut short and no other under which a patch is fetched: 5x5 [5,47,47,48]->48 10.2 / 11.9)
        return false;
    if (rival == PLANES_SPLIT && !p.wide && g.IC * eb % 128 != 0)
    {
        const int64_t tiles = (((int64_t)g.N * g.OH * g.OW + 31) / 32) * ((g.OC + 31) / 32);    // of 32 x 32 results, a workgroup each
        if (tiles * 5 >= (tiles + 255) / 256 * 256 * 4)
            return false;
    }
    return 2e-6 * (double)g.N * g.OH * g.OW * g.OC * g.IC * g.KH * g.KW >= 106 * p.us;
}

bool launch_conv_planes(hipStream_t st, int32_t in_dtype, const ConvGeom& g, const void* in, const void* w, const void* bias, const void* pad_page,
                        const void* zeros, int32_t in_zp, const RescaleParams& rp, uint32_t* flag_word, void* out)
{
    if (!planes_take(in_dtype, g) || (in_dtype == TMI_INT8) != (rp.enabled != 0) || (rp.enabled && !rp.fast) || (((uintptr_t)in | (uintptr_t)w | (uintptr_t)out | (uintptr_t)pad_page) & 15) != 0)
        return false;
    const int eb       = in_dtype == TMI_INT8 ? 1 : 2;
    const PlanesPlan p = plan_planes(g, eb);
    if (p.rows == 0)
        return false;
    const int64_t icb = (int64_t)g.IC * eb, taps = (int64_t)g.KH * g.KW, kb = icb * taps, tn = (g.OC + 63) / 64, tiles_m = (int64_t)g.N * p.tiles_image;
    PlanesArgs a{};
    a.patch_w = (int32_t)((int64_t)(g.OW - 1) * g.stride_x + (int64_t)(g.KW - 1) * g.dil_x + 1);
    if (p.tiles > (1 << 22) || !fastdiv_exact_up_to((uint64_t)p.tiles, (uint32_t)tn) || !fastdiv_exact_up_to((uint64_t)tiles_m, (uint32_t)p.tiles_image) ||
        !fastdiv_exact_up_to((uint64_t)p.patch_pixels + 8, (uint32_t)a.patch_w) || !fastdiv_exact_up_to(256, (uint32_t)g.OW))
        return false;
    a.x = (const uint8_t*)in, a.w = (const uint8_t*)w, a.pad_page = (const uint8_t*)pad_page, a.zeros = (const uint8_t*)zeros, a.bias = bias, a.out = out;
    a.N = g.OC, a.kb = (int32_t)kb, a.icb = (int32_t)icb, a.slices = (int32_t)p.slices, a.taps = (int32_t)taps, a.KW = g.KW;
    a.IH = g.IH, a.IW = g.IW, a.OH = g.OH, a.OW = g.OW;
    a.sy = g.stride_y, a.sx = g.stride_x, a.dy = g.dil_y, a.dx = g.dil_x, a.pad_top = g.pad_top, a.pad_left = g.pad_left;
    a.bias_len = g.bias_len, a.rows = p.rows, a.patch_pixels = (int32_t)p.patch_pixels;
    a.buffer_bytes = (int32_t)((p.patch_pixels + 7) / 8 * 1024);
    a.tiles = (int32_t)p.tiles, a.per_xcd = (int32_t)((p.tiles + 7) / 8);
    a.tiles_n = make_fastdiv((uint32_t)tn), a.tiles_image = make_fastdiv((uint32_t)p.tiles_image);
    a.div_pw = make_fastdiv((uint32_t)a.patch_w), a.div_ow = make_fastdiv((uint32_t)g.OW);
    a.padded = g.pad_top > 0 || g.pad_left > 0 || (int64_t)(g.OH - 1) * g.stride_y - g.pad_top + (int64_t)(g.KH - 1) * g.dil_y >= g.IH ||
               (int64_t)(g.OW - 1) * g.stride_x - g.pad_left + (int64_t)(g.KW - 1) * g.dil_x >= g.IW;
    a.za = in_zp, a.rp = rp, a.flag_word = flag_word;
    const size_t lds = (size_t)kPlanesRing * 8192 + 2 * (size_t)a.buffer_bytes + 256 + 64 * 32;    // and the tables
    auto run = [&](auto kernel) {
        if (!ensure_dynamic_lds<kernel.value>(lds))
            return false;
        hipLaunchKernelGGL(kernel.value, dim3((unsigned)(a.per_xcd * 8)), dim3(512), lds, st, a);
        return true;
    };
    if (in_dtype == TMI_INT8)
        return p.wide ? run(kernel_constant<conv_planes_kernel<int8_t, 2>>{}) : run(kernel_constant<conv_planes_kernel<int8_t, 1>>{});
    if (in_dtype == TMI_FP16)
        return p.wide ? run(kernel_constant<conv_planes_kernel<_Float16, 2>>{}) : run(kernel_constant<conv_planes_kernel<_Float16, 1>>{});
    return p.wide ? run(kernel_constant<conv_planes_kernel<bf16_t, 2>>{}) : run(kernel_constant<conv_planes_kernel<bf16_t, 1>>{});
}

}    // namespace tmi
