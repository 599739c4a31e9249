// The two extra passes of the reference's floating-point compliance flow, on the device:
//
//  * precise mode (--precise_mode: every floating-point tensor is evaluated in fp64) of CONV2D,
//    DEPTHWISE_CONV2D and MATMUL: operands in their storage type (fp16 / bf16 / fp32), products and sums in
//    fp64 in the reference's loop order - taps (ky, kx, ic), bias added last - so the result is the same
//    fp64 number the reference's loop nest produces (tensor_ops.cpp:843-882, 1291-1334, 1463-1500);
//  * bounds mode (bounds_mode: the same sums over absolute values, tensor_ops.cpp:757-765);
//  * the DOT_PRODUCT check of the verifier library (reference_model/src/verify/verify_dot_product.cpp:30-139)
//    as a reduction: per element the error in units of the bound, then sum, sum of squares, largest
//    magnitude and the number of elements that fail on their own.
//
// These are checkers for the fast kernels at shapes where a scalar CPU pass takes seconds to minutes.  CONV2D and MATMUL run
// on the ordered tiles of ordered_gemm.hip; the kernels here, one output element per lane, take DEPTHWISE_CONV2D and the
// shapes those decline (offsets or divisions beyond 32 bits).
#include "tmi_kernels.h"

namespace tmi
{

typedef int pr_v4i __attribute__((ext_vector_type(4)));

template <typename T>
__device__ __forceinline__ double widen(const void* p, size_t i);
template <>
__device__ __forceinline__ double widen<_Float16>(const void* p, size_t i)
{
    return (double)reinterpret_cast<const _Float16*>(p)[i];
}
template <>
__device__ __forceinline__ double widen<bf16_t>(const void* p, size_t i)
{
    return (double)bf16_to_float(reinterpret_cast<const bf16_t*>(p)[i]);
}
template <>
__device__ __forceinline__ double widen<float>(const void* p, size_t i)
{
    return (double)reinterpret_cast<const float*>(p)[i];
}

struct PreciseConvArgs
{
    ConvGeom g;
    const void* in;
    const void* w;
    const void* bias;
    double* out;
    int64_t total;
    int32_t abs_mode;
    int32_t depthwise;
    int32_t vec;    // channel vectors are whole, aligned 16-byte pieces
    // bounds mode without local_bound (tensor_ops.cpp:797-801, 1252-1256): every input element is replaced by the
    // largest magnitude of the input tensor, found by absmax_kernel; nullptr otherwise
    const double* input_abs_max;
};

// The largest |x| of a tensor into *out (zero before the launch; non-negative doubles order like their bit patterns).
template <typename T>
__global__ __launch_bounds__(256) void absmax_kernel(const void* x, int64_t n, double* out, int32_t blocks)
{
    __shared__ double red[256];
    double m             = 0.0;
    const int64_t stride = (int64_t)blocks * 256;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride)
        m = fmax(m, fabs(widen<T>(x, (size_t)i)));
    red[threadIdx.x] = m;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1)
    {
        if ((int)threadIdx.x < s)
            red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + s]);
        __syncthreads();
    }
    if (threadIdx.x == 0)
        atomicMax(reinterpret_cast<unsigned long long*>(out), (unsigned long long)__double_as_longlong(red[0]));
}

__global__ void store_zero_kernel(double* p)
{
    *p = 0.0;
}

template <typename T>
__global__ __launch_bounds__(256) void precise_conv_kernel(PreciseConvArgs a, int32_t blocks)
{
    const ConvGeom& g    = a.g;
    const int64_t stride = (int64_t)blocks * 256;
    const bool flat      = a.input_abs_max != nullptr;    // the input is one constant
    const double gmax    = flat ? *a.input_abs_max : 0.0;
    // (CONV2D's bounds pass multiplies the padding out, tensor_ops.cpp:845-852: an infinite weight there makes NaN)
    const bool outside_adds_nothing = a.depthwise || !a.abs_mode;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < a.total; i += stride)
    {
        const int oc      = (int)(i % g.OC);
        const int64_t pix = i / g.OC;
        const int ow      = (int)(pix % g.OW);
        const int oh      = (int)((pix / g.OW) % g.OH);
        const int n       = (int)(pix / ((int64_t)g.OW * g.OH));
        double acc        = 0.0;
        for (int ky = 0; ky < g.KH; ky++)
        {
            const int y     = oh * g.stride_y - g.pad_top + ky * g.dil_y;
            const bool y_in = y >= 0 && y < g.IH;
            if (!y_in && outside_adds_nothing)
                continue;
            for (int kx = 0; kx < g.KW; kx++)
            {
                const int x = ow * g.stride_x - g.pad_left + kx * g.dil_x;
                if (!y_in || x < 0 || x >= g.IW)
                {
                    if (!outside_adds_nothing)
                        for (int ic = 0; ic < g.IC; ic++)
                            acc = acc + 0.0 * fabs(widen<T>(a.w, (((size_t)oc * g.KH + ky) * g.KW + kx) * g.IC + ic));
                    continue;
                }
                const size_t in_base = (((size_t)n * g.IH + y) * g.IW + x) * g.IC;
                if (a.depthwise)
                {
                    // weight [KH, KW, C, M], output channel c * M + m
                    const int c = oc / g.M, m = oc - c * g.M;
                    double u = widen<T>(a.in, in_base + c);
                    double v = widen<T>(a.w, (((size_t)ky * g.KW + kx) * g.IC + c) * g.M + m);
                    if (a.abs_mode)
                        u = flat ? gmax : fabs(u), v = fabs(v);
                    acc = acc + u * v;
                }
                else
                {
                    const size_t w_base = (((size_t)oc * g.KH + ky) * g.KW + kx) * g.IC;
                    int ic              = 0;
                    if (a.vec)
                    {
                        // 16 bytes of both rows per step; the products still enter the sum one by one, in order
                        constexpr int V = 16 / (int)sizeof(T);
                        for (; ic + V <= g.IC; ic += V)
                        {
                            alignas(16) T xu[V], xw[V];
                            *reinterpret_cast<pr_v4i*>(xu) =
                                *reinterpret_cast<const pr_v4i*>(reinterpret_cast<const T*>(a.in) + in_base + ic);
                            *reinterpret_cast<pr_v4i*>(xw) =
                                *reinterpret_cast<const pr_v4i*>(reinterpret_cast<const T*>(a.w) + w_base + ic);
#pragma unroll
                            for (int e = 0; e < V; e++)
                            {
                                double u = widen<T>(xu, e), v = widen<T>(xw, e);
                                if (a.abs_mode)
                                    u = flat ? gmax : fabs(u), v = fabs(v);
                                acc = acc + u * v;
                            }
                        }
                    }
                    for (; ic < g.IC; ic++)
                    {
                        double u = widen<T>(a.in, in_base + ic);
                        double v = widen<T>(a.w, w_base + ic);
                        if (a.abs_mode)
                            u = flat ? gmax : fabs(u), v = fabs(v);
                        acc = acc + u * v;
                    }
                }
            }
        }
        double b = widen<T>(a.bias, g.bias_len == 1 ? 0 : oc);
        if (a.abs_mode)
            b = fabs(b);
        a.out[i] = acc + b;
    }
}

template <typename T>
__global__ __launch_bounds__(256) void precise_matmul_kernel(int32_t H, int32_t C, int32_t W, int64_t total,
                                                             const void* av, const void* bv, int32_t abs_mode,
                                                             int32_t vec, double* out, int32_t blocks)
{
    const int64_t stride = (int64_t)blocks * 256;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += stride)
    {
        const int w       = (int)(i % W);
        const int64_t row = i / W;    // n * H + h
        const int64_t n   = row / H;
        double acc        = 0.0;
        int c             = 0;
        if (vec)
        {
            constexpr int V = 16 / (int)sizeof(T);
            for (; c + V <= C; c += V)
            {
                alignas(16) T xu[V];
                *reinterpret_cast<pr_v4i*>(xu) =
                    *reinterpret_cast<const pr_v4i*>(reinterpret_cast<const T*>(av) + (size_t)row * C + c);
#pragma unroll
                for (int e = 0; e < V; e++)
                {
                    double u = widen<T>(xu, e);
                    double v = widen<T>(bv, ((size_t)n * C + c + e) * W + w);
                    if (abs_mode)
                        u = fabs(u), v = fabs(v);
                    acc = acc + u * v;
                }
            }
        }
        for (; c < C; c++)
        {
            double u = widen<T>(av, (size_t)row * C + c);
            double v = widen<T>(bv, ((size_t)n * C + c) * W + w);
            if (abs_mode)
                u = fabs(u), v = fabs(v);
            acc = acc + u * v;
        }
        out[i] = acc;
    }
}

static int grid_for(int64_t total)
{
    int64_t blocks = (total + 255) / 256;
    return (int)(blocks > 256 * 64 ? 256 * 64 : blocks);
}

const char* launch_conv_precise(hipStream_t st, int32_t in_dtype, bool depthwise, const ConvGeom& g, const void* in,
                                const void* w, const void* bias, int32_t abs_mode, double* abs_max_slot, double* out, void* copies)
{
    PreciseConvArgs a{};
    a.g = g, a.in = in, a.w = w, a.bias = bias, a.out = out, a.abs_mode = abs_mode, a.depthwise = depthwise ? 1 : 0;
    a.total = (int64_t)g.N * g.OH * g.OW * g.OC;
    const int eb = in_dtype == TMI_FP32 ? 4 : 2;
    a.vec        = ((int64_t)g.IC * eb) % 16 == 0 && (((uintptr_t)in | (uintptr_t)w) & 15) == 0;
    if (abs_mode && abs_max_slot)
    {
        // the bounds pass of an operator without local_bound: the input tensor's largest magnitude first
        const int64_t n_in = (int64_t)g.N * g.IH * g.IW * g.IC;
        const dim3 rgrid(grid_for(n_in)), rblock(256);
        hipLaunchKernelGGL(store_zero_kernel, dim3(1), dim3(1), 0, st, abs_max_slot);
        switch (in_dtype)
        {
            case TMI_FP16: hipLaunchKernelGGL(absmax_kernel<_Float16>, rgrid, rblock, 0, st, in, n_in, abs_max_slot, (int32_t)rgrid.x); break;
            case TMI_BF16: hipLaunchKernelGGL(absmax_kernel<bf16_t>, rgrid, rblock, 0, st, in, n_in, abs_max_slot, (int32_t)rgrid.x); break;
            case TMI_FP32: hipLaunchKernelGGL(absmax_kernel<float>, rgrid, rblock, 0, st, in, n_in, abs_max_slot, (int32_t)rgrid.x); break;
            default: return nullptr;
        }
        a.input_abs_max = abs_max_slot;
    }
    if (!depthwise && !copies && !a.input_abs_max && ordered_staged_leads(in_dtype, true, g, in, w) &&
        launch_ordered_conv_staged(st, in_dtype, true, g, in, w, bias, abs_mode != 0, out))
        return abs_mode ? "conv_bounds_ordered_staged_f64" : "conv_precise_ordered_staged_f64";
    if (!depthwise && copies && launch_ordered_conv_copied(st, in_dtype, true, g, in, w, bias, abs_mode != 0, a.input_abs_max, out, copies))
        return abs_mode ? "conv_bounds_copied_f64" : "conv_precise_copied_f64";
    if (!depthwise)
        switch (launch_ordered_conv(st, in_dtype, true, g, in, w, bias, abs_mode != 0, a.input_abs_max, out))
        {
            case OrderedForm::tiles: return abs_mode ? "conv_bounds_ordered_f64" : "conv_precise_ordered_f64";
            case OrderedForm::quarters: return abs_mode ? "conv_bounds_ordered_tail_f64" : "conv_precise_ordered_tail_f64";
            case OrderedForm::none: break;
        }
    switch (in_dtype)
    {
        case TMI_FP16: hipLaunchKernelGGL(precise_conv_kernel<_Float16>, dim3(grid_for(a.total)), dim3(256), 0, st, a, grid_for(a.total)); break;
        case TMI_BF16: hipLaunchKernelGGL(precise_conv_kernel<bf16_t>, dim3(grid_for(a.total)), dim3(256), 0, st, a, grid_for(a.total)); break;
        case TMI_FP32: hipLaunchKernelGGL(precise_conv_kernel<float>, dim3(grid_for(a.total)), dim3(256), 0, st, a, grid_for(a.total)); break;
        default: return nullptr;
    }
    return abs_mode ? "conv_bounds_f64" : "conv_precise_f64";
}

const char* launch_matmul_precise(hipStream_t st, int32_t in_dtype, int32_t N, int32_t H, int32_t C, int32_t W,
                                  const void* a, const void* b, int32_t abs_mode, double* out)
{
    switch (launch_ordered_matmul(st, in_dtype, true, N, H, C, W, a, b, abs_mode != 0, out))
    {
        case OrderedForm::tiles: return abs_mode ? "matmul_bounds_ordered_f64" : "matmul_precise_ordered_f64";
        case OrderedForm::quarters: return abs_mode ? "matmul_bounds_ordered_tail_f64" : "matmul_precise_ordered_tail_f64";
        case OrderedForm::none: break;
    }
    const int64_t total = (int64_t)N * H * W;
    const dim3 grid(grid_for(total)), block(256);
    const int eb      = in_dtype == TMI_FP32 ? 4 : 2;
    const int32_t vec = ((int64_t)C * eb) % 16 == 0 && ((uintptr_t)a & 15) == 0;
    switch (in_dtype)
    {
        case TMI_FP16: hipLaunchKernelGGL(precise_matmul_kernel<_Float16>, grid, block, 0, st, H, C, W, total, a, b, abs_mode, vec, out, (int32_t)grid.x); break;
        case TMI_BF16: hipLaunchKernelGGL(precise_matmul_kernel<bf16_t>, grid, block, 0, st, H, C, W, total, a, b, abs_mode, vec, out, (int32_t)grid.x); break;
        case TMI_FP32: hipLaunchKernelGGL(precise_matmul_kernel<float>, grid, block, 0, st, H, C, W, total, a, b, abs_mode, vec, out, (int32_t)grid.x); break;
        default: return nullptr;
    }
    return abs_mode ? "matmul_bounds_f64" : "matmul_precise_f64";
}

// ---- DOT_PRODUCT check ---------------------------------------------------------------------------------------
struct DpCheckArgs
{
    const void* imp;
    const double* ref;
    const double* bnd;
    int64_t n;
    int32_t abs_bound;
    int32_t normal_frac;
    double normal_min;
    DpPartial* partials;
};

template <typename T>
__device__ __forceinline__ bool overflows(double v);
template <>
__device__ __forceinline__ bool overflows<_Float16>(double v)
{
    return isinf((float)(_Float16)v);
}
template <>
__device__ __forceinline__ bool overflows<bf16_t>(double v)
{
    return isinf(bf16_to_float(float_to_bf16((float)v)));
}
template <>
__device__ __forceinline__ bool overflows<float>(double v)
{
    return isinf((float)v);
}

// Two elements per lane and pass (16-byte loads of both fp64 tensors where they are aligned), one partial result per
// workgroup written straight to `partials` - host memory that the device can write: atomics of 2048 workgroups on one line
// were nine tenths of the time (3.2 M fp32 elements, call to verdict: 140 -> 31 us).
template <typename T>
__global__ __launch_bounds__(256) void dp_check_kernel(DpCheckArgs a, int32_t blocks)
{
    __shared__ DpPartial red[4];
    double sum = 0.0, sumsq = 0.0, worst = 0.0;
    unsigned long long bad  = 0;
    const double unit_scale = exp2(-1.0 - a.normal_frac);
    auto one = [&](double ref, double bnd, double imp) {
        double err = 0.0;
        bool ok    = true;
        if (ref != ref)
            ok = imp != imp;    // a NaN reference must be matched
        else if (bnd != bnd)
            ok = true;          // no accuracy requirement under a NaN bound
        else if (overflows<T>(bnd * (1.0 + a.abs_bound * unit_scale)))
            ok = true;          // the dot product may overflow: no accuracy limit
        else if (bnd == 0.0)
            ok = ref == 0.0 && imp == 0.0;
        else
        {
            const double unit = fmax(bnd * unit_scale, a.normal_min);
            err               = (imp - ref) / unit;
            ok                = fabs(err) <= (double)a.abs_bound;
        }
        bad += ok ? 0 : 1;
        sum += err, sumsq += err * err;
        worst = fmax(worst, fabs(err));
    };
    const int64_t stride = (int64_t)blocks * 256, pairs = a.n / 2;
    const bool vec       = ((reinterpret_cast<uintptr_t>(a.ref) | reinterpret_cast<uintptr_t>(a.bnd)) & 15) == 0;
    int64_t i            = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (vec)
    {
        const double2* ref2 = reinterpret_cast<const double2*>(a.ref);
        const double2* bnd2 = reinterpret_cast<const double2*>(a.bnd);
        for (; i + stride < pairs; i += 2 * stride)
        {
            const double2 r0 = ref2[i], b0 = bnd2[i], r1 = ref2[i + stride], b1 = bnd2[i + stride];
            const double i0 = widen<T>(a.imp, (size_t)(2 * i)), i1 = widen<T>(a.imp, (size_t)(2 * i + 1));
            const double i2 = widen<T>(a.imp, (size_t)(2 * (i + stride))), i3 = widen<T>(a.imp, (size_t)(2 * (i + stride) + 1));
            one(r0.x, b0.x, i0), one(r0.y, b0.y, i1), one(r1.x, b1.x, i2), one(r1.y, b1.y, i3);
        }
        for (; i < pairs; i += stride)
        {
            const double2 r0 = ref2[i], b0 = bnd2[i];
            one(r0.x, b0.x, widen<T>(a.imp, (size_t)(2 * i))), one(r0.y, b0.y, widen<T>(a.imp, (size_t)(2 * i + 1)));
        }
        i = 2 * pairs + (int64_t)blockIdx.x * 256 + threadIdx.x;
    }
    for (; i < a.n; i += stride)
        one(a.ref[i], a.bnd[i], widen<T>(a.imp, (size_t)i));
    for (int s = 32; s > 0; s >>= 1)
    {
        sum += __shfl_xor(sum, s), sumsq += __shfl_xor(sumsq, s), bad += __shfl_xor(bad, s);
        worst = fmax(worst, __shfl_xor(worst, s));
    }
    if ((threadIdx.x & 63) == 0)
        red[threadIdx.x >> 6] = DpPartial{ sum, sumsq, worst, bad };
    __syncthreads();
    if (threadIdx.x == 0)
    {
        DpPartial t = red[0];
        for (int w = 1; w < 4; w++)
            t.sum += red[w].sum, t.sumsq += red[w].sumsq, t.worst = fmax(t.worst, red[w].worst), t.bad += red[w].bad;
        a.partials[blockIdx.x] = t;
    }
}

int dp_check_blocks(int64_t n)
{
    const int64_t blocks = (n + 511) / 512;
    return (int)(blocks > kDpCheckBlocks ? kDpCheckBlocks : blocks);
}

const char* launch_dp_check(hipStream_t st, int32_t out_dtype, int64_t n, const void* imp, const double* ref,
                            const double* bnd, int32_t abs_bound, DpPartial* partials)
{
    DpCheckArgs a{};
    a.imp = imp, a.ref = ref, a.bnd = bnd, a.n = n, a.abs_bound = abs_bound, a.partials = partials;
    const dim3 grid(dp_check_blocks(n)), block(256);
    switch (out_dtype)
    {
        case TMI_FP16:
            a.normal_frac = 10, a.normal_min = 0x1p-14;
            hipLaunchKernelGGL(dp_check_kernel<_Float16>, grid, block, 0, st, a, (int32_t)grid.x);
            break;
        case TMI_BF16:
            a.normal_frac = 7, a.normal_min = 0x1p-126;
            hipLaunchKernelGGL(dp_check_kernel<bf16_t>, grid, block, 0, st, a, (int32_t)grid.x);
            break;
        case TMI_FP32:
            a.normal_frac = 23, a.normal_min = 0x1p-126;
            hipLaunchKernelGGL(dp_check_kernel<float>, grid, block, 0, st, a, (int32_t)grid.x);
            break;
        default: return nullptr;
    }
    return "dot_product_check";
}

}    // namespace tmi
