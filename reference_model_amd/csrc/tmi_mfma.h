// Matrix-core plumbing shared by the MFMA kernels: vector types, the per-type 32x32 matrix instruction, and
// the small conversions their prologues and epilogues use.
#pragma once
#include "tmi_kernels.h"

namespace tmi
{

typedef int v2i __attribute__((ext_vector_type(2)));
typedef short v4s __attribute__((ext_vector_type(4)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef __bf16 v8b __attribute__((ext_vector_type(8)));

// One 32x32 MFMA step: 16 bytes of K per lane and operand (32 int8 or 16 half-precision values per row), lane
// half h = lane / 32 holding the K bytes [16h, 16h + 16) of row lane % 32.
template <typename T>
struct Mma;

template <>
struct Mma<int8_t>
{
    using acc_t                  = v16i;
    static constexpr bool is_int = true;
    __device__ static v16i mma(v4i a, v4i b, v16i c)
    {
        return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
    }
};
template <>
struct Mma<_Float16>
{
    using acc_t                  = v16f;
    static constexpr bool is_int = false;
    __device__ static v16f mma(v4i a, v4i b, v16f c)
    {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0,
                                                      0, 0);
    }
};
template <>
struct Mma<bf16_t>
{
    using acc_t                  = v16f;
    static constexpr bool is_int = false;
    __device__ static v16f mma(v4i a, v4i b, v16f c)
    {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8b, a), __builtin_bit_cast(v8b, b), c, 0,
                                                       0, 0);
    }
};

// The row of a weight operand's tile that lane rho reads: accumulator row 8q + 4h' + j is then channel 16h' + 4q + j, and a lane owns 16
// consecutive channels of one pixel
__device__ __forceinline__ int channel_of_row(int rho)
{
    return 16 * ((rho >> 2) & 1) + 4 * (rho >> 3) + (rho & 3);
}

// min(max(v, lo), hi) as one instruction; lo <= hi
__device__ __forceinline__ int32_t clamp_med3(int32_t v, int32_t lo, int32_t hi)
{
    int32_t r;
    asm("v_med3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "v"(lo), "v"(hi));
    return r;
}

__device__ __forceinline__ int dot4_ones(v4i v)
{
    int s = __builtin_amdgcn_sdot4(v.x, 0x01010101, 0, false);
    s     = __builtin_amdgcn_sdot4(v.y, 0x01010101, s, false);
    s     = __builtin_amdgcn_sdot4(v.z, 0x01010101, s, false);
    return __builtin_amdgcn_sdot4(v.w, 0x01010101, s, false);
}


template <typename T>
__device__ __forceinline__ float load_as_float(const void* p, int i);
template <>
__device__ __forceinline__ float load_as_float<_Float16>(const void* p, int i)
{
    return (float)reinterpret_cast<const _Float16*>(p)[i];
}
template <>
__device__ __forceinline__ float load_as_float<bf16_t>(const void* p, int i)
{
    return bf16_to_float(reinterpret_cast<const bf16_t*>(p)[i]);
}
template <>
__device__ __forceinline__ float load_as_float<int8_t>(const void*, int)
{
    return 0.0f;
}

__device__ __forceinline__ void store_from_float(_Float16* p, float v)
{
    *p = (_Float16)v;
}
__device__ __forceinline__ void store_from_float(bf16_t* p, float v)
{
    *p = float_to_bf16(v);
}
__device__ __forceinline__ void store_from_float(int8_t*, float)
{}

// 16 bytes from an address of no alignment (gfx950 takes global addresses of any)
__device__ __forceinline__ v4i load16(const uint8_t* p)
{
    v4i v;
    __builtin_memcpy(&v, p, 16);
    return v;
}
// v without its first n bytes, zeros behind (n < 16)
__device__ __forceinline__ v4i drop_bytes(v4i v, int n)
{
    uint64_t lo = (uint32_t)v[0] | (uint64_t)(uint32_t)v[1] << 32, hi = (uint32_t)v[2] | (uint64_t)(uint32_t)v[3] << 32;
    if (n & 8)
        lo = hi, hi = 0;
    const int bits = 8 * (n & 7);
    if (bits)
        lo = lo >> bits | hi << (64 - bits), hi >>= bits;
    return v4i{ (int)lo, (int)(lo >> 32), (int)hi, (int)(hi >> 32) };
}
// The same without 64-bit shifts, whose amount may not lie in a wave's last register (build.py).  In the kernels that use the other this one takes up to
// 15 registers more, two of them past the next border of occupancy.
__device__ __forceinline__ v4i drop_front(v4i v, int n)
{
    if (n & 8)
        v = v4i{ v[2], v[3], 0, 0 };
    if (n & 4)
        v = v4i{ v[1], v[2], v[3], 0 };
#pragma unroll
    for (int k = 0; k < 4; k++)
        v[k] = (int)__builtin_amdgcn_alignbyte(k < 3 ? v[k < 3 ? k + 1 : 3] : 0, v[k], n & 3);
    return v;
}
// the first n bytes of v, zeros behind (n may be negative)
__device__ __forceinline__ v4i keep_bytes(v4i v, int n)
{
#pragma unroll
    for (int k = 0; k < 4; k++)
    {
        const int m = n - 4 * k;
        v[k]        = m >= 4 ? v[k] : (m <= 0 ? 0 : v[k] & (int)((1u << (8 * m)) - 1u));
    }
    return v;
}

}    // namespace tmi
