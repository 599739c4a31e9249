// CONV2D and MATMUL whose sums keep the reference's order, on the matrix cores: the FP32 operators (fp32 products and sums,
// each rounded, ky -> kx -> ic) and the fp64 precise-mode / bounds-mode passes.  A reduction that may not be reordered
// still tiles over its results, and both forms have a matrix instruction that rounds as the loop nest does:
//
//  * fp64: v_mfma_f64_16x16x4 adds its four products to the accumulator one after the other with fused multiply-adds
//    (bit for bit against fma() in k order on 512 000 random results).  The operands are fp16, bf16 or fp32 values, whose
//    products fit 53 bits, so a fused multiply-add is the multiply and the add of the reference.
//  * fp32: v_mfma_f32_16x16x1 (four blocks) with a zero addend is the outer product of 32 x 32 operands, every product
//    rounded as v_mul_f32 rounds it (8 M products, subnormal ones among them); the additions stay on the vector ALU in
//    k order, 16 per lane and k, and the multiplications run beside them on the matrix cores.
//
// A workgroup of WM x WN waves owns 32 WM pixels (rows of the first operand) x 32 WN channels, a wave 32 x 32 of them; K is
// flattened over (ky, kx, ic) and staged through registers into two LDS buffers of BK elements a row, as fp32 (fp16 and
// bf16 widen exactly).  Rows are BK + 4 words long: the 16-byte reads of the fp32 form and the 4-byte reads of the fp64 form
// (row lane % 16, k lane / 16) then touch every bank once.
//
// What bounds it: a k of 32 x 32 results costs a SIMD 33.6 ns in fp32 (the instruction's 13.6 ns and the additions' 15.7 do not
// overlap: the two share the fp32 units) and four k 108 ns in fp64, where the matrix pipe is the limit.  us one result per
// lane -> these tiles, [16,28,28,256]x[256,3,3,256] of fp32: the operator 27 100 -> 299 (49 TFLOP/s), precise pass 7 300 ->
// 257, bounds pass 7 300 -> 255 (58 TFLOP/s); the distance to the 190 us of the fp64 pipe is the conversions to fp64, the
// stages' barriers and the tiles left over by whole rounds (see launch_ordered).
#include "tmi_mfma.h"

namespace tmi
{

typedef double v4d __attribute__((ext_vector_type(4)));

struct OrderedArgs
{
    const void* a;       // CONV2D input / MATMUL first operand
    const void* b;       // CONV2D weights [OC][K] / MATMUL second operand [K][OC]
    const void* bias;    // nullptr: none
    void* out;
    const double* input_abs_max;    // bounds pass without local_bound: what replaces every input element (nullptr: nothing does)
    int32_t M, OC, K;               // pixels (per batch), channels, reduction length
    int32_t IH, IW, IC, KW;
    int32_t pad_top, pad_left, stride_y, stride_x, dil_y, dil_x;
    FastDiv ow, oh, ic, kw;         // divisors of the pixel decode (OW, OH) and of the k decode (IC, KW)
    FastDiv tiles_n;
    int32_t tiles;                  // per batch
    int32_t n_big;                  // of these, tiles that are not cut into quarters
    int32_t bias_len;
    uint32_t abs_mask;              // 0x7fffffff in the bounds pass, else all ones
    int32_t vec_a, vec_b;           // operand rows are whole, aligned groups of four elements
    int32_t padded;                 // a tap can fall outside the image, and adds nothing there
};

template <typename T>
__device__ __forceinline__ float widen32(T v);
template <>
__device__ __forceinline__ float widen32<float>(float v)
{
    return v;
}
template <>
__device__ __forceinline__ float widen32<_Float16>(_Float16 v)
{
    return (float)v;
}
template <>
__device__ __forceinline__ float widen32<bf16_t>(bf16_t v)
{
    return bf16_to_float(v);
}

template <typename T>
__device__ __forceinline__ v4f load4(const T* p)
{
    struct alignas(4 * sizeof(T)) Four
    {
        T e[4];
    };
    const Four q = *reinterpret_cast<const Four*>(p);
    return v4f{ widen32<T>(q.e[0]), widen32<T>(q.e[1]), widen32<T>(q.e[2]), widen32<T>(q.e[3]) };
}

__device__ __forceinline__ float masked(float v, uint32_t mask)
{
    return __uint_as_float(__float_as_uint(v) & mask);
}

template <bool F64>
struct OrderedAcc;
template <>
struct OrderedAcc<false>
{
    using scalar = float;
};
template <>
struct OrderedAcc<true>
{
    using scalar = double;
};

// How the first operand is read: CONV2D whose stages lie inside one tap (IC a multiple of BK, 32-bit byte offsets), any
// CONV2D, MATMUL.
enum OrderedMode
{
    kTapStages,
    kAnyConv,
    kMatmul
};

// One workgroup's tile of results from (m0, n0) on; a wave has WT x WT of them.
template <typename T, bool F64, int MODE, int WM, int WN, int BK, int WT>
__device__ __forceinline__ void ordered_tile(const OrderedArgs& p, int m0, int n0, float* lds)
{
    using acc_t            = typename OrderedAcc<F64>::scalar;
    constexpr bool MATMUL  = MODE == kMatmul;
    constexpr int kThreads = 64 * WM * WN, BM = WT * WM, BN = WT * WN, LD = BK + 4;
    constexpr int KC  = BK / 4;          // groups of four k in a stage
    constexpr int RPP = kThreads / KC;   // rows a pass of the workgroup stages
    constexpr int NA = BM / RPP, NB = BN / RPP;
    static_assert(NA * RPP == BM && NB * RPP == BN && NB * kThreads == KC * BN, "staging");
    float (*sa)[BM * LD] = reinterpret_cast<float (*)[BM * LD]>(lds);
    float (*sb)[BN * LD] = reinterpret_cast<float (*)[BN * LD]>(lds + 2 * BM * LD);
    int& met_infinite    = *reinterpret_cast<int*>(lds + 2 * (BM + BN) * LD);

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t batch = blockIdx.y;
    const T* __restrict__ a_base = reinterpret_cast<const T*>(p.a) + (MATMUL ? batch * p.M * p.K : 0);
    const T* __restrict__ b_base = reinterpret_cast<const T*>(p.b) + (MATMUL ? batch * p.K * p.OC : 0);
    const bool flat  = F64 && p.input_abs_max != nullptr;
    const float gmax = flat ? (float)*p.input_abs_max : 0.0f;    // a value of the storage type: exact

    // rows of the first operand this lane stages: row RPP * i + tid / KC, k group tid % KC
    const int kq = tid & (KC - 1), r0 = tid / KC;
    int32_t y0[NA], x0[NA];
    const T* row[NA];
    bool row_ok[NA];
#pragma unroll
    for (int i = 0; i < NA; i++)
    {
        const int m = m0 + r0 + RPP * i;
        row_ok[i]   = m < p.M;
        y0[i] = x0[i] = 0;
        if constexpr (MATMUL)
            row[i] = a_base + (int64_t)(row_ok[i] ? m : p.M - 1) * p.K;
        else
        {
            const uint32_t pix = row_ok[i] ? (uint32_t)m : 0u, t = fdiv(pix, p.ow), n = fdiv(t, p.oh);
            y0[i]  = (int32_t)(t - n * p.oh.d) * p.stride_y - p.pad_top;
            x0[i]  = (int32_t)(pix - t * p.ow.d) * p.stride_x - p.pad_left;
            row[i] = a_base + (int64_t)n * p.IH * p.IW * p.IC;
        }
    }

    // kTapStages, kMatmul: byte offsets of the rows (under the present tap) and of the second operand's rows or columns, both
    // against scalar bases that walk along K.  Rows and columns past the end read the last one, whose results are not stored;
    // a row whose tap lies outside the image loads anything and is masked on its way to LDS.
    uint32_t off_a[NA], off_b[NB], mask_a[NA];
    int tap_ic = 0, tap_y = 0, tap_x = 0, tap_kx = 0;
    auto enter_tap = [&]() {
#pragma unroll
        for (int i = 0; i < NA; i++)
        {
            const int y = y0[i] + tap_y, x = x0[i] + tap_x;
            const bool ok = row_ok[i] && (uint32_t)y < (uint32_t)p.IH && (uint32_t)x < (uint32_t)p.IW;
            mask_a[i]     = ok ? p.abs_mask : 0u;
            off_a[i]      = ok ? (uint32_t)((row[i] - a_base) + (y * p.IW + x) * p.IC + 4 * kq) * (uint32_t)sizeof(T) : 0u;
        }
    };
    if constexpr (MODE == kTapStages)
    {
#pragma unroll
        for (int i = 0; i < NB; i++)
        {
            const int n = n0 + r0 + RPP * i;
            off_b[i]    = (uint32_t)((n < p.OC ? n : p.OC - 1) * p.K + 4 * kq) * (uint32_t)sizeof(T);
        }
        enter_tap();
    }
    const uint32_t k_pitch = (uint32_t)p.OC * (uint32_t)sizeof(T);    // MATMUL: a row of the second operand
    if constexpr (MATMUL)
    {
        const int n = n0 + (tid & (BN - 1));
#pragma unroll
        for (int i = 0; i < NA; i++)
            off_a[i] = (uint32_t)((row[i] - a_base) + 4 * kq) * (uint32_t)sizeof(T);
#pragma unroll
        for (int i = 0; i < NB; i++)
            off_b[i] = 4u * (uint32_t)(tid / BN + i * (kThreads / BN)) * k_pitch + (uint32_t)(n < p.OC ? n : p.OC - 1) * (uint32_t)sizeof(T);
    }
    const uint8_t* walk_b = reinterpret_cast<const uint8_t*>(b_base);
    v4f ra[NA], rb[NB];
    float finite = 0.0f;    // stays zero while every weight is finite

    auto load_stage = [&](int k0) {
        const int k = k0 + 4 * kq;
        if constexpr (MODE == kTapStages)
        {
            if (k0 && (tap_ic += BK) == p.IC)
            {
                tap_ic = 0, tap_x += p.dil_x;
                if (++tap_kx == p.KW)
                    tap_kx = 0, tap_x = 0, tap_y += p.dil_y;
                enter_tap();
            }
            const uint8_t* walk_a = reinterpret_cast<const uint8_t*>(a_base + tap_ic);
#pragma unroll
            for (int i = 0; i < NA; i++)
                ra[i] = flat ? v4f{ gmax, gmax, gmax, gmax } : load4<T>(reinterpret_cast<const T*>(walk_a + off_a[i]));
#pragma unroll
            for (int i = 0; i < NB; i++)
                rb[i] = load4<T>(reinterpret_cast<const T*>(walk_b + off_b[i]));
            walk_b += BK * sizeof(T);
            return;
        }
        if constexpr (MATMUL)
        {
            const uint8_t* walk_a = reinterpret_cast<const uint8_t*>(a_base + k0);
            if (p.vec_a && k0 + BK <= p.K)
            {
#pragma unroll
                for (int i = 0; i < NA; i++)
                    ra[i] = load4<T>(reinterpret_cast<const T*>(walk_a + off_a[i]));
            }
            else
            {
#pragma unroll
                for (int i = 0; i < NA; i++)
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        ra[i][e] = k + e < p.K ? widen32<T>(reinterpret_cast<const T*>(walk_a + off_a[i])[e]) : 0.0f;
            }
        }
        else if (p.vec_a)
        {
            const uint32_t kk = k < p.K ? (uint32_t)k : 0u, tap = fdiv(kk, p.ic), ky = fdiv(tap, p.kw);
            const int ic = (int)(kk - tap * p.ic.d), dy = (int)ky * p.dil_y, dx = (int)(tap - ky * p.kw.d) * p.dil_x;
#pragma unroll
            for (int i = 0; i < NA; i++)
            {
                const int y = y0[i] + dy, x = x0[i] + dx;
                ra[i] = v4f{ 0, 0, 0, 0 };
                if (row_ok[i] && k < p.K && (uint32_t)y < (uint32_t)p.IH && (uint32_t)x < (uint32_t)p.IW)
                    ra[i] = flat ? v4f{ gmax, gmax, gmax, gmax } : load4<T>(row[i] + (y * p.IW + x) * p.IC + ic);
            }
        }
        else
        {
#pragma unroll
            for (int i = 0; i < NA; i++)
                ra[i] = v4f{ 0, 0, 0, 0 };
            for (int e = 0; e < 4; e++)
                if (k + e < p.K)
                {
                    const uint32_t kk = (uint32_t)(k + e), tap = fdiv(kk, p.ic), ky = fdiv(tap, p.kw);
                    const int ic = (int)(kk - tap * p.ic.d), dy = (int)ky * p.dil_y, dx = (int)(tap - ky * p.kw.d) * p.dil_x;
#pragma unroll
                    for (int i = 0; i < NA; i++)
                    {
                        const int y = y0[i] + dy, x = x0[i] + dx;
                        if (row_ok[i] && (uint32_t)y < (uint32_t)p.IH && (uint32_t)x < (uint32_t)p.IW)
                        {
                            const float v = flat ? gmax : widen32<T>(row[i][(y * p.IW + x) * p.IC + ic]);
                            // (a constant index per copy: a register array under a run-time index would live in scratch)
                            ra[i] = v4f{ e == 0 ? v : ra[i].x, e == 1 ? v : ra[i].y, e == 2 ? v : ra[i].z, e == 3 ? v : ra[i].w };
                        }
                    }
                }
        }
        if constexpr (MATMUL)
        {
            // [K][OC]: a lane takes four k of one column, neighbouring lanes neighbouring columns
            if (k0 + BK <= p.K)
            {
#pragma unroll
                for (int i = 0; i < NB; i++)
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        rb[i][e] = widen32<T>(*reinterpret_cast<const T*>(walk_b + off_b[i] + e * k_pitch));
            }
            else
            {
#pragma unroll
                for (int i = 0; i < NB; i++)
                {
                    const int kb = k0 + 4 * (tid / BN + i * (kThreads / BN));
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        rb[i][e] = kb + e < p.K ? widen32<T>(*reinterpret_cast<const T*>(walk_b + off_b[i] + e * k_pitch)) : 0.0f;
                }
            }
            walk_b += (int64_t)BK * k_pitch;
        }
        else
        {
#pragma unroll
            for (int i = 0; i < NB; i++)
            {
                const int n = n0 + r0 + RPP * i;
                rb[i]       = v4f{ 0, 0, 0, 0 };
                if (n < p.OC)
                {
                    const T* w = b_base + (int64_t)n * p.K + k;
                    if (p.vec_b)
                    {
                        if (k < p.K)
                            rb[i] = load4<T>(w);
                    }
                    else
                    {
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            if (k + e < p.K)
                                rb[i][e] = widen32<T>(w[e]);
                    }
                }
            }
        }
    };
    auto store_stage = [&](int buf) {
#pragma unroll
        for (int i = 0; i < NA; i++)
        {
            v4f v = ra[i];
            if constexpr (MODE == kTapStages)
                v = v4f{ masked(v.x, mask_a[i]), masked(v.y, mask_a[i]), masked(v.z, mask_a[i]), masked(v.w, mask_a[i]) };
            else if constexpr (F64)
                v = v4f{ masked(v.x, p.abs_mask), masked(v.y, p.abs_mask), masked(v.z, p.abs_mask), masked(v.w, p.abs_mask) };
            *reinterpret_cast<v4f*>(&sa[buf][(r0 + RPP * i) * LD + 4 * kq]) = v;
        }
#pragma unroll
        for (int i = 0; i < NB; i++)
        {
            v4f v = rb[i];
            if (!MATMUL && p.padded)
            {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    finite = __builtin_fmaf(v[e], 0.0f, finite);
            }
            if constexpr (F64)
                v = v4f{ masked(v.x, p.abs_mask), masked(v.y, p.abs_mask), masked(v.z, p.abs_mask), masked(v.w, p.abs_mask) };
            const int at = MATMUL ? (tid & (BN - 1)) * LD + 4 * (tid / BN + i * (kThreads / BN)) : (r0 + RPP * i) * LD + 4 * kq;
            *reinterpret_cast<v4f*>(&sb[buf][at]) = v;
        }
    };

    // 32 x 32 results of a wave.  fp32: one instruction of four blocks, block q = lane / 16 of the operands = (row half q / 2,
    // column half q % 2), results in registers 4 q + r.  fp64: four instructions.
    // 16 x 16 results of a wave.  fp32: the four blocks are four k, whose products are added one after the other.  fp64: one
    // instruction.
    const int wm = (wave / WN) * WT, wn = (wave % WN) * WT, l16 = lane & 15, q = lane >> 4;
    v16f acc32;
    v4f acc4 = { 0, 0, 0, 0 };
    v4d acc64[4];
    if constexpr (F64)
    {
#pragma unroll
        for (int t = 0; t < 4; t++)
            acc64[t] = v4d{ 0, 0, 0, 0 };
    }
    else
    {
#pragma unroll
        for (int t = 0; t < 16; t++)
            acc32[t] = 0.0f;
    }
    auto compute = [&](int buf) {
        if constexpr (WT == 16)
        {
            const float* pa = &sa[buf][(wm + l16) * LD + q];
            const float* pb = &sb[buf][(wn + l16) * LD + q];
            float fa[BK / 4], fb[BK / 4];
#pragma unroll
            for (int k = 0; k < BK / 4; k++)
                fa[k] = pa[4 * k], fb[k] = pb[4 * k];
            if constexpr (F64)
            {
#pragma unroll
                for (int k = 0; k < BK / 4; k++)
                    acc64[0] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)fa[k], (double)fb[k], acc64[0], 0, 0, 0);
            }
            else
            {
                const v16f zero = { 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0 };
                v16f prod       = __builtin_amdgcn_mfma_f32_16x16x1f32(fa[0], fb[0], zero, 0, 0, 0);
#pragma unroll
                for (int k = 0; k < BK / 4; k++)
                {
                    v16f next = prod;
                    if (k + 1 < BK / 4)
                    {
                        float x = fa[k + 1];
                        asm volatile("" : "+v"(x), "+v"(acc4));    // (as below: one product ahead, no more)
                        next = __builtin_amdgcn_mfma_f32_16x16x1f32(x, fb[k + 1], zero, 0, 0, 0);
                    }
#pragma unroll
                    for (int t = 0; t < 16; t++)
                        acc4[t & 3] = acc4[t & 3] + prod[t];
                    prod = next;
                }
            }
        }
        else if constexpr (F64)
        {
            const float* pa = &sa[buf][(wm + l16) * LD + q];
            const float* pb = &sb[buf][(wn + l16) * LD + q];
            float fa[2][2], fb[2][2];    // this step's and the next one's fragments
            fa[0][0] = pa[0], fa[0][1] = pa[16 * LD], fb[0][0] = pb[0], fb[0][1] = pb[16 * LD];
#pragma unroll
            for (int k = 0; k < BK; k += 4)
            {
                const int c = (k >> 2) & 1;
                if (k + 4 < BK)
                    fa[c ^ 1][0] = pa[k + 4], fa[c ^ 1][1] = pa[16 * LD + k + 4], fb[c ^ 1][0] = pb[k + 4], fb[c ^ 1][1] = pb[16 * LD + k + 4];
                const double a0 = fa[c][0], a1 = fa[c][1], b0 = fb[c][0], b1 = fb[c][1];
                acc64[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc64[0], 0, 0, 0);
                acc64[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc64[1], 0, 0, 0);
                acc64[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc64[2], 0, 0, 0);
                acc64[3] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc64[3], 0, 0, 0);
            }
        }
        else
        {
            const float* pa = &sa[buf][(wm + 16 * (q >> 1) + l16) * LD];
            const float* pb = &sb[buf][(wn + 16 * (q & 1) + l16) * LD];
            const v16f zero = { 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0 };
            // The products of the next k are under way while those of this one are added.  The empty asm ties each instruction's
            // operand to the sums of the step before: without it the compiler issues a stage's 32 instructions at once and keeps
            // all their results.
            v4f a = *reinterpret_cast<const v4f*>(pa), b = *reinterpret_cast<const v4f*>(pb);
            v16f prod = __builtin_amdgcn_mfma_f32_16x16x1f32(a[0], b[0], zero, 0, 0, 0);
#pragma unroll
            for (int k = 0; k < BK; k += 4)
            {
                v4f an = a, bn = b;
                if (k + 4 < BK)
                    an = *reinterpret_cast<const v4f*>(pa + k + 4), bn = *reinterpret_cast<const v4f*>(pb + k + 4);
#pragma unroll
                for (int e = 0; e < 4; e++)
                {
                    v16f next = prod;
                    if (k + e + 1 < BK)
                    {
                        float x = e < 3 ? a[(e + 1) & 3] : an[0];
                        asm volatile("" : "+v"(x), "+v"(acc32));
                        next = __builtin_amdgcn_mfma_f32_16x16x1f32(x, e < 3 ? b[(e + 1) & 3] : bn[0], zero, 0, 0, 0);
                    }
#pragma unroll
                    for (int t = 0; t < 16; t++)
                        acc32[t] = acc32[t] + prod[t];
                    prod = next;
                }
                a = an, b = bn;
            }
        }
    };

    const int stages = (p.K + BK - 1) / BK;
    if (tid == 0)
        met_infinite = 0;
    load_stage(0);
    store_stage(0);
    __syncthreads();
    for (int s = 0; s < stages; s++)
    {
        if (s + 1 < stages)
            load_stage((s + 1) * BK);
        compute(s & 1);
        if (s + 1 < stages)
            store_stage((s + 1) & 1);    // the buffer every wave left behind at the last barrier
        __syncthreads();
    }

    auto store_result = [&](int m, int oc, acc_t v) {
        if (p.bias)
        {
            const float b = masked(widen32<T>(reinterpret_cast<const T*>(p.bias)[p.bias_len == 1 ? 0 : oc]), F64 ? p.abs_mask : ~0u);
            v             = v + (acc_t)b;
        }
        reinterpret_cast<acc_t*>(p.out)[(batch * p.M + m) * p.OC + oc] = v;
    };
    // A tap outside the image adds nothing in the reference (but in its bounds pass); here it adds 0 * weight, which is not nothing
    // when the weight is infinite or NaN.  A tile that met such a weight is summed again one result at a time.
    if (!MATMUL && p.padded)
    {
        // (not __syncthreads_or: it brings 256 bytes of hidden arguments into every launch)
        if (finite != 0.0f)
            met_infinite = 1;
        __syncthreads();
    }
    if (!MATMUL && p.padded && met_infinite)
    {
        for (int t = tid; t < BM * BN; t += kThreads)
        {
            const int m = m0 + t / BN, oc = n0 + t % BN;
            if (m >= p.M || oc >= p.OC)
                continue;
            const uint32_t tt = fdiv((uint32_t)m, p.ow), n = fdiv(tt, p.oh);
            const int yb = (int32_t)(tt - n * p.oh.d) * p.stride_y - p.pad_top, xb = (int32_t)((uint32_t)m - tt * p.ow.d) * p.stride_x - p.pad_left;
            const T* img = a_base + (int64_t)n * p.IH * p.IW * p.IC;
            const T* w   = b_base + (int64_t)oc * p.K;
            acc_t sum    = 0;
            int y = yb, x = xb, kx = 0;
            for (int k = 0; k < p.K; k += p.IC)
            {
                if ((uint32_t)y < (uint32_t)p.IH && (uint32_t)x < (uint32_t)p.IW)
                    for (int ic = 0; ic < p.IC; ic++)
                    {
                        const float u = flat ? gmax : masked(widen32<T>(img[(y * p.IW + x) * p.IC + ic]), F64 ? p.abs_mask : ~0u);
                        const float v = masked(widen32<T>(w[k + ic]), F64 ? p.abs_mask : ~0u);
                        sum           = sum + (acc_t)u * (acc_t)v;
                    }
                x += p.dil_x;
                if (++kx == p.KW)
                    kx = 0, x = xb, y += p.dil_y;
            }
            store_result(m, oc, sum);
        }
        return;
    }
    if constexpr (F64)
    {
        // row lane / 16 + 4 r, column lane % 16: 16 lanes store 128 bytes of one pixel
#pragma unroll
        for (int t = 0; t < (WT == 16 ? 1 : 4); t++)
#pragma unroll
            for (int r = 0; r < 4; r++)
            {
                const int m = m0 + wm + 16 * (t >> 1) + q + 4 * r, oc = n0 + wn + 16 * (t & 1) + l16;
                if (m < p.M && oc < p.OC)
                    store_result(m, oc, acc64[t][r]);
            }
    }
    else
    {
#pragma unroll
        for (int t = 0; t < (WT == 16 ? 4 : 16); t++)
        {
            const int m = m0 + wm + 16 * (t >> 3) + 4 * q + (t & 3), oc = n0 + wn + 16 * ((t >> 2) & 1) + l16;
            if (m < p.M && oc < p.OC)
                store_result(m, oc, WT == 16 ? acc4[t & 3] : acc32[t]);
        }
    }
}

template <int BM, int BN, int BK>
constexpr int ordered_lds_floats()
{
    return 2 * (BM + BN) * (BK + 4) + 1;
}

template <typename T, bool F64, int MODE, int WM, int WN, int BK>
__global__ __launch_bounds__(64 * WM * WN, 4) void ordered_gemm_kernel(OrderedArgs p)
{
    constexpr int BM = 32 * WM, BN = 32 * WN;
    __shared__ __attribute__((aligned(16))) float lds[ordered_lds_floats<BM, BN, BK>()];
    // neighbouring tiles share operand rows: a contiguous run of tiles for each of the eight L2s
    const uint32_t per_xcd = ((uint32_t)p.tiles + 7) >> 3;
    const uint32_t tile    = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (tile >= (uint32_t)p.tiles)
        return;
    const uint32_t tm = fdiv(tile, p.tiles_n), tn = tile - tm * p.tiles_n.d;
    ordered_tile<T, F64, MODE, WM, WN, BK, 32>(p, (int)tm * BM, (int)tn * BN, lds);
}

// The first p.n_big tiles of 64 x 64 (a multiple of eight) as above, each of the others as four workgroups of 32 x 32 results.
template <typename T, bool F64, int MODE>
__global__ __launch_bounds__(256, 4) void ordered_gemm_tail_kernel(OrderedArgs p)
{
    __shared__ __attribute__((aligned(16))) float lds[ordered_lds_floats<64, 64, 32>()];
    const uint32_t n_big = (uint32_t)p.n_big;
    if (blockIdx.x < n_big)
    {
        const uint32_t tile = (blockIdx.x & 7) * (n_big >> 3) + (blockIdx.x >> 3);
        const uint32_t tm = fdiv(tile, p.tiles_n), tn = tile - tm * p.tiles_n.d;
        ordered_tile<T, F64, MODE, 2, 2, 32, 32>(p, (int)tm * 64, (int)tn * 64, lds);
        return;
    }
    const uint32_t quarter = blockIdx.x - n_big, tile = n_big + (quarter >> 2);
    const uint32_t tm = fdiv(tile, p.tiles_n), tn = tile - tm * p.tiles_n.d;
    const int m0 = (int)tm * 64 + 32 * (int)((quarter >> 1) & 1), n0 = (int)tn * 64 + 32 * (int)(quarter & 1);
    if (m0 < p.M && n0 < p.OC)
        ordered_tile<T, F64, MODE, 2, 2, 32, 16>(p, m0, n0, lds);
}

template <typename T, bool F64, int MODE>
static OrderedForm launch_ordered(hipStream_t st, OrderedArgs p, int64_t batches)
{
    // Workgroups of four waves and 64 x 64 results, in stages of 32 (of 16 where a reduction of at most 96 would leave half a
    // stage empty); of two waves and 64 x 32 or 32 x 64 where a ragged side would leave more than a quarter of those empty.  A
    // wave has 32 x 32 results in every such shape, so a smaller workgroup only shares fewer operand rows (us 64 x 64 / 32 x 64,
    // fp64 [16,28,28,256]->256 332 / 389).
    auto padded_area = [&](int bm, int bn) { return (int64_t)((p.M + bm - 1) / bm) * bm * ((p.OC + bn - 1) / bn) * bn; };
    const int64_t area = padded_area(64, 64);
    int bm = 64, bn = 64;
    if (4 * padded_area(64, 32) < 3 * area)
        bn = 32;
    else if (4 * padded_area(32, 64) < 3 * area)
        bm = 32;
    const bool short_stages = MODE != kTapStages && p.K <= 96 && (p.K & 31) != 0 && (p.K & 31) <= 16;
    // Quarters: a round of tiles is one per CU, a wave on each SIMD, and takes as long for one tile as for 256.  Up to 192 tiles
    // (together, or left over by whole rounds) are cut into four workgroups of 32 x 32 results, 16 x 16 a wave, which take a
    // quarter of the time each and spread over four times the SIMDs; beyond, four quarters a CU are a round again.  us whole
    // tiles / quarters, fp32 operator and fp64 pass: [16,28,28,256]->256 3x3 (784 tiles: 16 left over) 330 and 314 / 299 and 257,
    // [1,14,14,256]->256 (16) 130 and 102 / 45 and 45, [4,28,28,128]->128 (98) 71 and 56 / 33 and 34, [3,28,28,256]->256 (148) 137
    // and 104 / 85 and 85, [9,28,28,256]->256 (444: 188 left over) fp64 188 / 161, MATMUL 333 x 500 x 300 (30) 34 and 26 / 14 and 12.
    const int64_t tiles64 = area / 4096, tn64 = (p.OC + 63) / 64;
    const int64_t over       = tiles64 % 256;    // left over by whole rounds
    const bool all_quarters  = tiles64 * batches <= 192;
    const bool some_quarters = batches == 1 && bm == 64 && bn == 64 && !short_stages && over > 0 && over <= 192;
    if ((all_quarters || some_quarters) && tiles64 <= INT32_MAX / 4 && fastdiv_exact_up_to((uint64_t)tiles64, (uint32_t)tn64))
    {
        p.n_big   = (int32_t)(all_quarters ? 0 : tiles64 - over);
        p.tiles_n = make_fastdiv((uint32_t)tn64), p.tiles = (int32_t)tiles64;
        const dim3 grid((unsigned)(p.n_big + 4 * (tiles64 - p.n_big)), (unsigned)batches);
        hipLaunchKernelGGL((ordered_gemm_tail_kernel<T, F64, MODE>), grid, dim3(256), 0, st, p);
        return OrderedForm::quarters;
    }
    const int64_t tiles = padded_area(bm, bn) / (bm * bn);
    const int64_t tn = (p.OC + bn - 1) / bn;
    if (!fastdiv_exact_up_to((uint64_t)tiles + 8, (uint32_t)tn) || tiles > INT32_MAX - 8 || batches > 65535)
        return OrderedForm::none;
    p.tiles_n = make_fastdiv((uint32_t)tn), p.tiles = (int32_t)tiles;
    const dim3 grid((unsigned)((tiles + 7) / 8 * 8), (unsigned)batches);
    if (bn == 32)
        hipLaunchKernelGGL((ordered_gemm_kernel<T, F64, MODE, 2, 1, 16>), grid, dim3(128), 0, st, p);
    else if (bm == 32)
        hipLaunchKernelGGL((ordered_gemm_kernel<T, F64, MODE, 1, 2, 16>), grid, dim3(128), 0, st, p);
    else if (short_stages)
        hipLaunchKernelGGL((ordered_gemm_kernel<T, F64, MODE, 2, 2, MODE == kTapStages ? 32 : 16>), grid, dim3(256), 0, st, p);
    else
        hipLaunchKernelGGL((ordered_gemm_kernel<T, F64, MODE, 2, 2, 32>), grid, dim3(256), 0, st, p);
    return OrderedForm::tiles;
}

static bool aligned16(const void* p)
{
    return ((uintptr_t)p & 15) == 0;
}

OrderedForm launch_ordered_conv(hipStream_t st, int32_t in_dtype, bool f64, const ConvGeom& g, const void* in, const void* w,
                         const void* bias, bool abs_mode, const double* input_abs_max, void* out)
{
    const int64_t pixels = (int64_t)g.N * g.OH * g.OW, K = (int64_t)g.KH * g.KW * g.IC;
    // 32-bit offsets inside an image and exact divisions of the decodes
    if (K < 1 || K > INT32_MAX - 64 || pixels > INT32_MAX - 64 || (int64_t)g.IH * g.IW * g.IC > INT32_MAX ||
        !fastdiv_exact_up_to((uint64_t)pixels, (uint32_t)g.OW) || !fastdiv_exact_up_to((uint64_t)pixels / g.OW, (uint32_t)g.OH) ||
        !fastdiv_exact_up_to((uint64_t)K, (uint32_t)g.IC) || !fastdiv_exact_up_to((uint64_t)g.KH * g.KW, (uint32_t)g.KW))
        return OrderedForm::none;
    OrderedArgs p{};
    p.a = in, p.b = w, p.bias = bias, p.out = out, p.input_abs_max = input_abs_max;
    p.M = (int32_t)pixels, p.OC = g.OC, p.K = (int32_t)K, p.IH = g.IH, p.IW = g.IW, p.IC = g.IC, p.KW = g.KW;
    p.pad_top = g.pad_top, p.pad_left = g.pad_left, p.stride_y = g.stride_y, p.stride_x = g.stride_x, p.dil_y = g.dil_y, p.dil_x = g.dil_x;
    p.ow = make_fastdiv((uint32_t)g.OW), p.oh = make_fastdiv((uint32_t)g.OH), p.ic = make_fastdiv((uint32_t)g.IC), p.kw = make_fastdiv((uint32_t)g.KW);
    p.bias_len = g.bias_len, p.abs_mask = abs_mode ? 0x7fffffffu : ~0u;
    p.vec_a = p.vec_b = g.IC % 4 == 0 && aligned16(in) && aligned16(w);
    // (the bounds pass multiplies the padding out, tensor_ops.cpp:845-852: an infinite weight there makes NaN, as zeros in the operand do)
    p.padded = !abs_mode &&
               (g.pad_top > 0 || g.pad_left > 0 || (int64_t)(g.OH - 1) * g.stride_y - g.pad_top + (int64_t)(g.KH - 1) * g.dil_y >= g.IH ||
                (int64_t)(g.OW - 1) * g.stride_x - g.pad_left + (int64_t)(g.KW - 1) * g.dil_x >= g.IW);
    const int64_t eb = in_dtype == TMI_FP32 ? 4 : 2;
    const bool taps  = p.vec_a && g.IC % 32 == 0 && (int64_t)g.N * g.IH * g.IW * g.IC * eb < INT32_MAX && (int64_t)g.OC * K * eb < INT32_MAX;
    if (!f64)
        return in_dtype != TMI_FP32 ? OrderedForm::none
                                    : (taps ? launch_ordered<float, false, kTapStages>(st, p, 1) : launch_ordered<float, false, kAnyConv>(st, p, 1));
    switch (in_dtype)
    {
        case TMI_FP16: return taps ? launch_ordered<_Float16, true, kTapStages>(st, p, 1) : launch_ordered<_Float16, true, kAnyConv>(st, p, 1);
        case TMI_BF16: return taps ? launch_ordered<bf16_t, true, kTapStages>(st, p, 1) : launch_ordered<bf16_t, true, kAnyConv>(st, p, 1);
        case TMI_FP32: return taps ? launch_ordered<float, true, kTapStages>(st, p, 1) : launch_ordered<float, true, kAnyConv>(st, p, 1);
        default: return OrderedForm::none;
    }
}

OrderedForm launch_ordered_matmul(hipStream_t st, int32_t in_dtype, bool f64, int32_t N, int32_t H, int32_t C, int32_t W, const void* a,
                           const void* b, bool abs_mode, void* out)
{
    // 32-bit byte offsets inside a batch
    if (C < 1 || H > INT32_MAX - 64 || W > INT32_MAX - 64 || (int64_t)H * C > INT32_MAX / 4 || (int64_t)C * W > INT32_MAX / 4)
        return OrderedForm::none;
    OrderedArgs p{};
    p.a = a, p.b = b, p.out = out, p.M = H, p.OC = W, p.K = C;
    p.bias_len = 1, p.abs_mask = abs_mode ? 0x7fffffffu : ~0u;
    p.vec_a = C % 4 == 0 && aligned16(a);
    if (!f64)
        return in_dtype != TMI_FP32 ? OrderedForm::none : launch_ordered<float, false, kMatmul>(st, p, N);
    switch (in_dtype)
    {
        case TMI_FP16: return launch_ordered<_Float16, true, kMatmul>(st, p, N);
        case TMI_BF16: return launch_ordered<bf16_t, true, kMatmul>(st, p, N);
        case TMI_FP32: return launch_ordered<float, true, kMatmul>(st, p, N);
        default: return OrderedForm::none;
    }
}

}    // namespace tmi
