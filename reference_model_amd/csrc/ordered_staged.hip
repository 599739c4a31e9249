// The sums of ordered_gemm.hip for CONV2D (the fp64 precise-mode and bounds-mode passes, and the fp32 operator on few tiles) on
// operands whose channel vectors are whole units of eight elements, read where they lie and widened once on their way into LDS.
//
// What bounds it: the fp64 and fp32 matrix instructions run on the vector units - a v_mfma_f64_16x16x4 takes 27.4 ns of its SIMD, and every
// vector instruction of any wave on that SIMD comes on top (8 additions 17 ns, 8 conversions to fp64 29 ns, whether from the same wave or
// another).  So the loop has as few as it can: a lane stages one unit of eight k a stage (8 conversions to fp64, and 8 to fp32 for 16-bit
// operands, or none for the fp32 sums), which two rows or columns of waves share; taps are entered by a scalar walk where the channel
// vectors are whole stages; and a tap or a row that does not exist is a load past the end of the buffer, which returns zeros.  LDS holds
// what lane 16 e + row multiplies, the operands of two instructions side by side: fragments are 16-byte reads in lane order, a pair ahead of
// the instructions, no bank conflict.  Loads are three stages ahead in registers; a stage costs one barrier, which is for the stage after the
// present one.  The ring is three stages, 48 KB, so that three workgroups fit a CU (with four: 129 to 192 tiles in two rounds, 15.3 / 11.6 us).
//
// us before (ordered_gemm.hip or ordered_copies.hip) / here, 3x3, fp64: [9,50,66,224]->16 stride 2 67.3 / 32.9, [1,7,7,512]->512 67.4 / 49.2
// (31.6 of it the matrix instructions of one chain), [4,14,14,1024]->256 1x1 21.4 / 14.0, [8,56,56,64]->64 43.4 / 38.8, [16,28,28,256]->256 232 / 229
// (190 of matrix instructions); fp32 sums: [9,50,66,224]->16 stride 2 52.5 / 36.9.
#include <type_traits>

#include "outside_taps.h"

namespace tmi
{

typedef double v2d __attribute__((ext_vector_type(2)));
typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v2f __attribute__((ext_vector_type(2)));

struct StagedArgs
{
    const void *a, *b, *bias;    // input, weights [OC][K], bias
    void* out;
    uint32_t a_bytes, b_bytes;
    int32_t M, OC;
    int32_t units, gp;              // of a reduction, of a channel vector
    uint32_t tap_skip, row_skip;    // bytes from a tap's end to the next, and what is added at a row's end
    int32_t IC, IH, IW, KH, KW;
    int32_t pad_top, pad_left, stride_y, stride_x, dil_y, dil_x;
    int32_t tiles, n_big;           // of 64 x 64; those not cut into quarters (a multiple of eight)
    int32_t quarters_per_xcd;
    int32_t bias_len;
    int32_t padded;                 // a tap can fall outside the image, and adds nothing there
    FastDiv ow, oh, tiles_n;
};

template <typename T>
__device__ __forceinline__ float widened(T v)
{
    if constexpr (std::is_same_v<T, bf16_t>)
        return bf16_to_float(v);
    else
        return (float)v;
}

// One workgroup of four waves, 2 x 2 of WT x WT results from (m0, n0) on.  A stage is 256 units of eight k, one a lane: WT 16 32 rows of
// either operand and 32 k, WT 32 64 rows and 16 k.
template <typename T, bool F64, bool ABS, bool WHOLE, int WT>
__device__ __forceinline__ void staged_tile(const StagedArgs& p, int m0, int n0, uint8_t* lds)
{
    using acc_t  = std::conditional_t<F64, double, float>;
    using pair_t = std::conditional_t<F64, v2d, v2f>;    // a lane's operands of two consecutive instructions
    constexpr int CH = WT == 16 ? 4 : 2, UB = 8 * sizeof(T), NR = UB / 16;
    constexpr int PAIR = sizeof(pair_t), BLOCK = 64 * PAIR, OPERAND = 8 * BLOCK, STAGE = 2 * OPERAND, RING = 3, AHEAD = 3;
    constexpr int TW = WT / 16;    // tiles of 16 of a wave's side
    constexpr uint32_t OUTSIDE = 0x80000000u;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // What this lane stages: unit `chunk` of a stage of row `row`, of the first operand (waves 0 and 1) or the second, a row of which is
    // one tap of all its units.
    const bool second = wave >= 2;
    const int row     = WT == 16 ? 16 * (wave & 1) + (lane & 15) : 32 * (wave & 1) + (lane & 31);
    const int chunk   = WT == 16 ? lane >> 4 : lane >> 5;
    uint8_t* stage_to = lds + (second ? OPERAND : 0) + ((row >> 4) * CH + chunk) * BLOCK + (row & 15) * PAIR;
    const auto rsrc   = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(second ? p.b : p.a), 0, (int)(second ? p.b_bytes : p.a_bytes), 0x00020000);
    const int gp = second ? p.units : p.gp, KW = second ? 1 : p.KW, KH = second ? 1 : p.KH, IH = second ? 1 : p.IH, IW = second ? 1 : p.IW;
    int kx = 0, ky = 0, x0 = 0, x = 0, y = 0, image = n0 + row;
    bool row_there = n0 + row < p.OC;
    if (!second)
    {
        const int m = m0 + row;
        row_there   = m < p.M;
        const uint32_t pix = row_there ? (uint32_t)m : 0u, t = fdiv(pix, p.ow), n = fdiv(t, p.oh);
        y     = (int32_t)(t - n * p.oh.d) * p.stride_y - p.pad_top;
        x     = x0 = (int32_t)(pix - t * p.ow.d) * p.stride_x - p.pad_left;
        image = (int32_t)n * IH * IW;
    }
    // Where the lane's next unit lies, and whether it does (loads from OUTSIDE on return zeros).  The position goes on modulo 2^32 where the
    // tap is outside.
    uint32_t at = (uint32_t)((image + y * IW + x) * gp + chunk) * (uint32_t)UB, from = OUTSIDE;
    const uint32_t tap_skip = second ? 0u : p.tap_skip, row_skip = second ? 0u : p.row_skip;    // behind a tap's units
    auto enter = [&]() {
        from = (row_there & (ky < KH) & ((uint32_t)y < (uint32_t)IH) & ((uint32_t)x < (uint32_t)IW)) ? at : OUTSIDE;
    };
    auto next_tap = [&]() {
        x += p.dil_x, at += tap_skip;
        if (++kx == KW)
            kx = 0, x = x0, y += p.dil_y, at += row_skip, ky++;
    };
    // Units up to the end of the tap.  WHOLE: the channel vectors are whole stages, so that all lanes enter a tap together and the walk
    // inside it is scalar.
    int left        = WHOLE ? gp : gp - chunk;
    uint32_t walked = 0;
    auto settle     = [&]() {
        while (left <= 0 && ky < KH)
        {
            next_tap();
            left += gp;
        }
    };
    if constexpr (!WHOLE)
        settle();
    enter();
    v4i raw[AHEAD][NR];
    auto load = [&](int set) {
#pragma unroll
        for (int i = 0; i < NR; i++)
            raw[set][i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)(from + 16 * i), __builtin_amdgcn_readfirstlane((int)walked), 0));
        left -= CH;
        if constexpr (WHOLE)
        {
            walked += CH * UB;
            left = __builtin_amdgcn_readfirstlane(left);
            if (left == 0)
            {
                at += walked, left = gp, walked = 0;
                next_tap();
                enter();
            }
        }
        else
        {
            at += CH * UB;
            settle();
            enter();
        }
    };
    // k % 4 = e of the unit side by side: what lane 16 e + row % 16 multiplies in the unit's two instructions
    auto stage = [&](int set, int slot) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; i++)
        {
            if constexpr (sizeof(T) == 4)
                v[i] = __int_as_float(raw[set][i >> 2][i & 3]);
            else
            {
                const uint32_t u = (uint32_t)raw[set][0][i >> 1];
                if constexpr (std::is_same_v<T, bf16_t>)
                    v[i] = __uint_as_float(i & 1 ? u & 0xffff0000u : u << 16);
                else
                    v[i] = (float)__builtin_bit_cast(_Float16, (uint16_t)(i & 1 ? u >> 16 : u));
            }
            if constexpr (ABS)
                v[i] = __builtin_fabsf(v[i]);
        }
#pragma unroll
        for (int e = 0; e < 4; e++)
        {
            acc_t* to = reinterpret_cast<acc_t*>(stage_to + slot * STAGE + e * 16 * PAIR);
            to[0] = (acc_t)v[e], to[1] = (acc_t)v[e + 4];
        }
    };
    const int wm = (wave >> 1) * WT, wn = (wave & 1) * WT, l16 = lane & 15, q = lane >> 4;
    v4d acc64[TW * TW];
    v4f acc4 = { 0, 0, 0, 0 };
    if constexpr (F64)
    {
#pragma unroll
        for (int t = 0; t < TW * TW; t++)
            acc64[t] = v4d{ 0, 0, 0, 0 };
    }
    const uint8_t* fa_from = lds + (wm >> 4) * CH * BLOCK + lane * PAIR;
    const uint8_t* fb_from = lds + OPERAND + (wn >> 4) * CH * BLOCK + lane * PAIR;
    pair_t fa[2][TW], fb[2][TW];
    auto fetch = [&](int set, int slot, int pair) {
#pragma unroll
        for (int t = 0; t < TW; t++)
        {
            fa[set][t] = *reinterpret_cast<const pair_t*>(fa_from + slot * STAGE + (t * CH + pair) * BLOCK);
            fb[set][t] = *reinterpret_cast<const pair_t*>(fb_from + slot * STAGE + (t * CH + pair) * BLOCK);
        }
    };
    v16f prod;
    auto product = [&](int set, int i) {
        const v16f zero = { 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0 };
        float u         = (float)fa[set][0][i];
        asm volatile("" : "+v"(u), "+v"(acc4));    // (one product ahead, no more)
        return __builtin_amdgcn_mfma_f32_16x16x1f32(u, (float)fb[set][0][i], zero, 0, 0, 0);
    };
    auto multiply = [&](int set) {
#pragma unroll
        for (int i = 0; i < 2; i++)
        {
            if constexpr (F64)
            {
#pragma unroll
                for (int t = 0; t < TW * TW; t++)
                    acc64[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[set][t / TW][i], fb[set][t % TW][i], acc64[t], 0, 0, 0);
            }
            else
            {
                const v16f ahead = i == 0 ? product(set, 1) : product(set ^ 1, 0);
#pragma unroll
                for (int t = 0; t < 16; t++)
                    acc4[t & 3] = acc4[t & 3] + prod[t];    // the four blocks of an instruction are four k
                prod = ahead;
            }
        }
    };

    const int S = (p.units + CH - 1) / CH;
#pragma unroll
    for (int s = 0; s < AHEAD; s++)
        load(s);
    stage(0, 0), load(0);
    stage(1, 1), load(1);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    fetch(0, 0, 0);
    if constexpr (!F64)
        prod = product(0, 0);
    auto walk = [&](auto multiplies) {
        for (int s0 = 0; s0 < S; s0 += AHEAD)
        {
#pragma unroll
            for (int r = 0; r < AHEAD; r++)
            {
                if (s0 + r >= S)
                    break;
                // every wave has written its part of the next stage and is past the one before this
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
                for (int pair = 0; pair < CH; pair++)
                {
                    if constexpr (multiplies.value)
                    {
                        if (pair + 1 < CH)
                            fetch((pair + 1) & 1, r % RING, pair + 1);
                        else
                            fetch(0, (r + 1) % RING, 0);
                        __builtin_amdgcn_sched_barrier(0);    // (a pair ahead)
                        multiply(pair & 1);
                    }
                    if (pair == 0)
                    {
                        // (past the end too: a load that is sometimes left out would have the compiler wait for all loads in flight)
                        stage((r + 2) % AHEAD, (r + 2) % RING);
                        load((r + 2) % AHEAD);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
    };
    // A tap outside the image adds nothing in the reference (but in its bounds pass); here it adds 0 * weight, which is not nothing when the weight is
    // infinite or NaN (see outside_taps.h): results that are NaN under a window that leaves the image, in channels with such a weight, are summed again.
    // us a call on a NaN image, every NaN summed again / so (on finite values): [4,14,14,256]->64 3x3 fp64 1050 / 33 (29), fp32 1062 / 48 (43).
    auto met_odd = [&](bool nan) {
        if (ABS || !p.padded)
            return false;
        const int64_t row_bytes = (int64_t)p.KH * p.KW * p.IC * (int)sizeof(T);
        const int channels      = p.OC - n0 < 2 * WT ? p.OC - n0 : 2 * WT;
        return met_odd_weights<T, 4>(nan ? __builtin_nanf("") : 0.0f, wave, reinterpret_cast<int32_t*>(lds + RING * STAGE),
                                     [&](auto&& look) { look(reinterpret_cast<const uint8_t*>(p.b) + n0 * row_bytes, channels * row_bytes); });
    };
    if (m0 + wm >= p.M || n0 + wn >= p.OC)
    {
        walk(std::false_type{});    // a wave without results: only its part of the stages
        met_odd(false);
        return;
    }
    walk(std::true_type{});

    // A lane's results: fp64 rows lane / 16 + 4 r, column lane % 16 (16 lanes store 128 bytes of one pixel), fp32 rows 4 (lane / 16) + r.
    constexpr int RESULTS = F64 ? 4 * TW * TW : 4;
    auto place = [&](int i, int& m, int& oc) {
        const int t = i >> 2, r = i & 3;
        m           = m0 + wm + 16 * (t / TW) + (F64 ? q + 4 * r : 4 * q + r), oc = n0 + wn + 16 * (t % TW) + l16;
        return m < p.M && oc < p.OC;
    };
    auto store_result = [&](int m, int oc, acc_t v) {
        const float b = widened<T>(reinterpret_cast<const T*>(p.bias)[p.bias_len == 1 ? 0 : oc]);
        reinterpret_cast<acc_t*>(p.out)[(size_t)m * p.OC + oc] = v + (acc_t)(ABS ? __builtin_fabsf(b) : b);
    };
    bool nan = false;
#pragma unroll
    for (int i = 0; i < RESULTS; i++)
    {
        acc_t v;
        if constexpr (F64)
            v = acc64[i >> 2][i & 3];
        else
            v = acc4[i];
        int m, oc;
        nan |= v != v;
        if (place(i, m, oc))
            store_result(m, oc, v);
    }
    if (!met_odd(nan))
        return;
    const int64_t row_bytes = (int64_t)p.KH * p.KW * p.IC * (int)sizeof(T);
    uint32_t odd = 0;    // a bit for each column of the lane
    for (int t = 0; t < TW; t++)
    {
        const int oc        = n0 + wn + 16 * t + l16;
        const uint64_t part = __ballot(weights_not_finite<T>(reinterpret_cast<const uint8_t*>(p.b) + (oc < p.OC ? oc : n0) * row_bytes, row_bytes, q, 4));
        odd |= (part >> l16 & 0x0001000100010001u) != 0 ? 1u << t : 0u;
    }
    for (int i = 0; i < RESULTS; i++)
    {
        int m, oc;
        if (!place(i, m, oc) || (odd >> ((i >> 2) % TW) & 1) == 0)
            continue;
        const uint32_t t = fdiv((uint32_t)m, p.ow), n = fdiv(t, p.oh);
        const int yb = (int32_t)(t - n * p.oh.d) * p.stride_y - p.pad_top, xb = (int32_t)((uint32_t)m - t * p.ow.d) * p.stride_x - p.pad_left;
        const acc_t stored = reinterpret_cast<const acc_t*>(p.out)[(size_t)m * p.OC + oc];
        if (stored == stored || (yb >= 0 && xb >= 0 && yb + (p.KH - 1) * p.dil_y < p.IH && xb + (p.KW - 1) * p.dil_x < p.IW))
            continue;
        const T* img = reinterpret_cast<const T*>(p.a) + (int64_t)n * p.IH * p.IW * p.IC;
        const T* w   = reinterpret_cast<const T*>(p.b) + (int64_t)oc * p.KH * p.KW * p.IC;
        acc_t sum    = 0;
        for (int ky = 0; ky < p.KH; ky++)
            for (int kx = 0; kx < p.KW; kx++, w += p.IC)
            {
                const int iy = yb + ky * p.dil_y, ix = xb + kx * p.dil_x;
                if ((uint32_t)iy < (uint32_t)p.IH && (uint32_t)ix < (uint32_t)p.IW)
                    for (int c = 0; c < p.IC; c++)
                        sum = sum + (acc_t)widened<T>(img[(iy * p.IW + ix) * p.IC + c]) * (acc_t)widened<T>(w[c]);
            }
        store_result(m, oc, sum);
    }
}

// The first n_big tiles of 64 x 64 results whole, each of the others as four workgroups of 32 x 32.
template <typename T, bool F64, bool ABS, bool WHOLE>
__global__ __launch_bounds__(256, 2) void ordered_staged_kernel(StagedArgs p)
{
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const uint32_t n_big = (uint32_t)p.n_big;
    // neighbouring tiles share operand rows: a contiguous run of them for each of the eight L2s
    if constexpr (F64)
        if (blockIdx.x < n_big)
        {
            const uint32_t tile = (blockIdx.x & 7) * (n_big >> 3) + (blockIdx.x >> 3);
            const uint32_t tm = fdiv(tile, p.tiles_n), tn = tile - tm * p.tiles_n.d;
            staged_tile<T, F64, ABS, WHOLE, 32>(p, (int)tm * 64, (int)tn * 64, lds);
            return;
        }
    const uint32_t at = blockIdx.x - n_big, quarter = (at & 7) * (uint32_t)p.quarters_per_xcd + (at >> 3), tile = n_big + (quarter >> 2);
    if (tile >= (uint32_t)p.tiles)
        return;
    const uint32_t tm = fdiv(tile, p.tiles_n), tn = tile - tm * p.tiles_n.d;
    const int m0 = (int)tm * 64 + 32 * (int)((quarter >> 1) & 1), n0 = (int)tn * 64 + 32 * (int)(quarter & 1);
    if (m0 < p.M && n0 < p.OC)
        staged_tile<T, F64, ABS, WHOLE, 16>(p, m0, n0, lds);
}

template <typename T, bool F64>
static bool launch_staged(hipStream_t st, const StagedArgs& p, bool abs_mode)
{
    constexpr int kLds  = 3 * 64 * 2 * 8 * (F64 ? 16 : 8) + 64;    // the ring, and the words of met_odd_weights()
    const unsigned grid = (unsigned)(p.n_big + 8 * p.quarters_per_xcd);
    auto run = [&](auto kernel) {
        if (!ensure_dynamic_lds<kernel.value>(kLds))
            return false;
        hipLaunchKernelGGL(kernel.value, dim3(grid), dim3(256), kLds, st, p);
        return true;
    };
    if (F64 && abs_mode)
        return p.gp % 4 == 0 ? run(kernel_constant<ordered_staged_kernel<T, F64, F64, true>>{}) : run(kernel_constant<ordered_staged_kernel<T, F64, F64, false>>{});
    return p.gp % 4 == 0 ? run(kernel_constant<ordered_staged_kernel<T, F64, false, true>>{}) : run(kernel_constant<ordered_staged_kernel<T, F64, false, false>>{});
}

// Whether a layer runs here.  us by the other ordered kernels / here over layers of 5 to 3750 tiles of 64 x 64, fp64 unless noted:
//   K 144 6.5 / 5.9, 21.7 / 18.5, 101 / 92; 504 14.5 / 10.2, 52.9 / 44.1, 289 / 255; 2376 39.1 / 30.8, 195 / 177.  K 64: 5.3 / 5.5, 15.5 / 17.5; 24 4.3 / 5.0.
//   fp32 operands of whole 32 channels, which ordered_gemm.hip reads without decodes: K 160 7.1 / 7.5, 27.2 / 28.7, 288 30.7 / 28.1.
//   16-bit operands, two conversions an element, on many tiles with long reductions: [16,28,28,256]->256 3x3 232 on copies / 243; K 1152, 564 tiles
//     90.5 / 90.0.
//   Few channels on many tiles, where half the waves have no results: 938 tiles of 16 channels K 144 19.3 / 32.4, 1152 94 / 112; 407 tiles none slower.
//   fp32 sums, up to 192 tiles: K 504 15.5 / 13.0, 1152 25.0 / 21.8, 2376 49.4 / 44.4; 288 8.8 / 8.2 and 13.3 / 14.1; 160 8.6 / 10.0.
//   The same on images of a few pixels: 1 to 15 of them, [1,4,3,128]->65 3x3 17.9 / 14.3, [1,1,1,1024]->256 1x1 20.6 / 12.4, fp32 sums [1,2,2,512]->512 3x3 87.4 / 74.8;
//     over 15 layers of seven shapes 0.55 ... 0.89 of the time.
bool ordered_staged_leads(int32_t in_dtype, bool f64, const ConvGeom& g, const void* in, const void* w)
{
    const int64_t pixels = (int64_t)g.N * g.OH * g.OW, K = (int64_t)g.KH * g.KW * g.IC, eb = in_dtype == TMI_FP32 ? 4 : 2;
    const int64_t tiles = ((pixels + 63) / 64) * ((g.OC + 63) / 64), tn = (g.OC + 63) / 64;
    if (g.IC % 8 != 0 || (((uintptr_t)in | (uintptr_t)w) & 15) != 0 || K < 1 || K > INT32_MAX / 8 || (int64_t)g.N * g.IH * g.IW * g.IC * eb >= INT32_MAX ||
        (int64_t)g.OC * K * eb >= INT32_MAX || pixels > INT32_MAX - 64 || tiles > INT32_MAX / 8 || !fastdiv_exact_up_to((uint64_t)tiles, (uint32_t)tn) ||
        !fastdiv_exact_up_to((uint64_t)pixels, (uint32_t)g.OW) || !fastdiv_exact_up_to((uint64_t)pixels / g.OW, (uint32_t)g.OH))
        return false;
    if (!f64)
        return tiles <= 192 && K >= 400;
    if (g.OC <= 32 && tiles > 600)
        return false;
    if (eb == 2 && tiles > 512 && K > 900)
        return false;
    return K >= (eb == 4 && g.IC % 32 == 0 ? 224 : 96);
}

bool launch_ordered_conv_staged(hipStream_t st, int32_t in_dtype, bool f64, const ConvGeom& g, const void* in, const void* w, const void* bias, bool abs_mode,
                                void* out)
{
    const int64_t pixels = (int64_t)g.N * g.OH * g.OW, K = (int64_t)g.KH * g.KW * g.IC, eb = in_dtype == TMI_FP32 ? 4 : 2;
    const int64_t tn = (g.OC + 63) / 64, tiles = ((pixels + 63) / 64) * tn, over = tiles % 256;
    StagedArgs p{};
    p.a = in, p.b = w, p.bias = bias, p.out = out;
    p.a_bytes = (uint32_t)((int64_t)g.N * g.IH * g.IW * g.IC * eb), p.b_bytes = (uint32_t)(g.OC * K * eb);
    p.M = (int32_t)pixels, p.OC = g.OC, p.units = (int32_t)(K / 8), p.gp = g.IC / 8;
    p.IC = g.IC, p.IH = g.IH, p.IW = g.IW, p.KH = g.KH, p.KW = g.KW;
    p.pad_top = g.pad_top, p.pad_left = g.pad_left, p.stride_y = g.stride_y, p.stride_x = g.stride_x, p.dil_y = g.dil_y, p.dil_x = g.dil_x;
    p.bias_len = g.bias_len;
    p.tap_skip = (uint32_t)((g.dil_x - 1) * g.IC * eb), p.row_skip = (uint32_t)(((int64_t)g.dil_y * g.IW - (int64_t)g.KW * g.dil_x) * g.IC * eb);
    p.ow = make_fastdiv((uint32_t)g.OW), p.oh = make_fastdiv((uint32_t)g.OH), p.tiles_n = make_fastdiv((uint32_t)tn);
    // (the bounds pass multiplies the padding out, tensor_ops.cpp:845-852: an infinite weight there makes NaN, as zeros in the operand do)
    p.padded = !abs_mode &&
               (g.pad_top > 0 || g.pad_left > 0 || (int64_t)(g.OH - 1) * g.stride_y - g.pad_top + (int64_t)(g.KH - 1) * g.dil_y >= g.IH ||
                (int64_t)(g.OW - 1) * g.stride_x - g.pad_left + (int64_t)(g.KW - 1) * g.dil_x >= g.IW);
    // Whole tiles by rounds of one per CU, what is left over as quarters (see ordered_gemm.hip)
    p.tiles            = (int32_t)tiles;
    p.n_big            = tiles <= 192 || g.OC <= 32 || !f64 ? 0 : (int32_t)(over <= 192 ? tiles - over : tiles / 8 * 8);
    p.quarters_per_xcd = (int32_t)((4 * (tiles - p.n_big) + 7) / 8);
    if (!f64)
        return in_dtype == TMI_FP32 && launch_staged<float, false>(st, p, abs_mode);
    switch (in_dtype)
    {
        case TMI_FP16: return launch_staged<_Float16, true>(st, p, abs_mode);
        case TMI_BF16: return launch_staged<bf16_t, true>(st, p, abs_mode);
        case TMI_FP32: return launch_staged<float, true>(st, p, abs_mode);
        default: return false;
    }
}

}    // namespace tmi
