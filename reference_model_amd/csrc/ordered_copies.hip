// The sums of ordered_gemm.hip for CONV2D (fp32, and the fp64 precise-mode and bounds-mode passes, in the reference's order) on copies of
// the operands that the matrix instructions can read as they lie.
//
// A first launch writes both operands widened to the type of the sums (bounds pass: their magnitudes), the image with its
// padding materialised, channel vectors filled up with zeros to granules of 64 bytes, and inside a granule the elements
// k % 4 = q side by side as chunk q of 16 bytes: one 16-byte read then gives a lane its operands of two (fp64) or four (fp32)
// consecutive instructions.  The second launch brings rows of 128 or 256 bytes straight into a ring of LDS stages
// (global_load_lds_dwordx4), several stages ahead, and its loop is LDS reads, matrix instructions and, in fp32, additions: no
// conversion, no mask, no register staging.  Adding zeros leaves a sum as it is (it starts at +0 and never becomes -0), so the
// results are those of ordered_gemm.hip bit for bit.
//
// What bounds it is the chain of a result: a 16x16x4 fp64 matrix instruction takes 64 clocks whether or not the next depends on it
// (28.7 ns alone, 30 with every CU at work), an fp32 step of four k 32 clocks and 64 of additions.  A layer of few tiles is that chain,
// K / 4 instructions: [..,288]->24 3x3 (K 2592, 4 tiles), fp64 34.4 us of which the instructions are 18.6 and the first launch 3 (51.0 by
// ordered_gemm.hip), and a wave must find its next operands in registers: without the fragments read a stage ahead it was 51.
// [4,56,56,256]->256 3x3, fp64: 232 us, 212 of them matrix instructions (256 by ordered_gemm.hip).
//
// A tap outside the image multiplies a zero by a weight; where some weight of a tile's channels is infinite or NaN (the
// first launch leaves a word per piece of a row that says so) the tile is summed again one result at a time without those taps.
#include <type_traits>

#include "tmi_mfma.h"

namespace tmi
{

typedef double v2d __attribute__((ext_vector_type(2)));
typedef double v4d __attribute__((ext_vector_type(4)));

struct CopyArgs
{
    const void *a, *b, *bias;    // input, weights, bias
    uint8_t *ca, *cb, *cbias;
    int32_t* bad;        // per weight row and piece: a weight is not finite
    const double* input_abs_max;    // bounds pass without local_bound: what replaces every input element
    uint32_t abs_mask;
    int32_t IC, OC, IH, IW, taps, bias_len;
    int32_t pad_top, pad_left;
    int32_t a_chunks;              // of the first operand
    int32_t a_blocks, b_blocks;    // workgroups of either part
    int32_t pieces;                // workgroups of a weight row
    int32_t granules, row_granules;    // of a weight row: with content, and with the zeros behind
    int32_t gp;                    // granules of a channel vector
    FastDiv div_gp4, div_w, div_h, div_pieces, div_gp;
};

struct CopiedArgs
{
    const uint8_t *a, *b, *bias;
    const int32_t* bad;
    void* out;
    int32_t M, OC;
    int32_t pitch_x, pitch_y;      // bytes from one output pixel / row to the next in the first operand's copy
    int32_t image;                 // and from one image to the next
    int32_t gp, KW, next_tap, next_row;    // a channel vector's granules; bytes from its end to the next tap, from a row's end to the next row
    int32_t granules, stages;
    int32_t zero_off;              // where the first operand's copy holds 64 bytes of zeros
    int32_t b_pitch;
    int32_t tiles, n_big;          // all; those not cut into quarters (a multiple of eight)
    int32_t big_first;             // which of them come first
    int32_t IC, IH, IW, KH, pieces;
    int32_t pad_top, pad_left, stride_y, stride_x, dil_y, dil_x;
    int32_t padded;                // a tap can fall outside the image, and adds nothing there
    FastDiv ow, oh, tiles_n;
};

template <typename T>
__device__ __forceinline__ float to_f32(T v);
template <>
__device__ __forceinline__ float to_f32<float>(float v)
{
    return v;
}
template <>
__device__ __forceinline__ float to_f32<_Float16>(_Float16 v)
{
    return (float)v;
}
template <>
__device__ __forceinline__ float to_f32<bf16_t>(bf16_t v)
{
    return bf16_to_float(v);
}

template <bool F64>
using sum_t = std::conditional_t<F64, double, float>;

// One chunk: elements q, q + 4, ... of a granule, the first `live` elements of the granule existing.
template <bool F64>
__device__ __forceinline__ void put_chunk(uint8_t* to, const float (&v)[4])
{
    if constexpr (F64)
        *reinterpret_cast<v2d*>(to) = v2d{ (double)v[0], (double)v[1] };
    else
        *reinterpret_cast<v4f*>(to) = v4f{ v[0], v[1], v[2], v[3] };
}

template <typename T, bool F64>
__global__ __launch_bounds__(256) void ordered_copy_kernel(CopyArgs p)
{
    constexpr int PER = F64 ? 2 : 4, KG = 4 * PER;    // elements of a chunk, of a granule
    __shared__ int any_bad;
    const int tid = threadIdx.x;
    auto widen    = [&](T v) { return __uint_as_float(__float_as_uint(to_f32<T>(v)) & p.abs_mask); };
    if (blockIdx.x < (uint32_t)p.a_blocks)
    {
        const uint32_t t = blockIdx.x * 256u + tid;
        if (t >= (uint32_t)p.a_chunks)
            return;
        const uint32_t pix = fdiv(t, p.div_gp4);
        const int r = (int)(t - pix * p.div_gp4.d), c0 = (r >> 2) * KG + (r & 3);
        const uint32_t row = fdiv(pix, p.div_w), n = fdiv(row, p.div_h);
        const int x = (int)(pix - row * p.div_w.d) - p.pad_left, y = (int)(row - n * p.div_h.d) - p.pad_top;
        const bool inside = (unsigned)x < (unsigned)p.IW && (unsigned)y < (unsigned)p.IH;
        const T* src      = reinterpret_cast<const T*>(p.a) + (inside ? (((size_t)n * p.IH + y) * p.IW + x) * p.IC : 0);
        const bool flat  = F64 && p.input_abs_max != nullptr;
        const float gmax = flat ? (float)*p.input_abs_max : 0.0f;    // a value of the storage type: exact
        float v[4]       = { 0, 0, 0, 0 };
#pragma unroll
        for (int i = 0; i < PER; i++)
            if (inside && c0 + 4 * i < p.IC)
                v[i] = flat ? gmax : widen(src[c0 + 4 * i]);
        put_chunk<F64>(p.ca + (size_t)t * 16, v);
        return;
    }
    const uint32_t blk = blockIdx.x - p.a_blocks;
    if (blk >= (uint32_t)p.b_blocks)
    {
        // the zeros behind the first operand, and the bias
        if (tid < 4)
            *reinterpret_cast<v4i*>(p.ca + (size_t)p.a_chunks * 16 + tid * 16) = v4i{ 0, 0, 0, 0 };
        for (int i = tid; i < p.OC; i += 256)
                reinterpret_cast<sum_t<F64>*>(p.cbias)[i] = (sum_t<F64>)widen(reinterpret_cast<const T*>(p.bias)[p.bias_len == 1 ? 0 : i]);
        return;
    }
    const uint32_t oc = fdiv(blk, p.div_pieces);
    const int at      = (int)(blk - oc * p.div_pieces.d) * 256 + tid;    // chunk of the row
    if (tid == 0)
        any_bad = 0;
    __syncthreads();
    if (at < p.row_granules * 4)
    {
        const int G = at >> 2, tap = (int)fdiv((uint32_t)G, p.div_gp), c0 = (G - tap * p.gp) * KG + (at & 3);
        float v[4]  = { 0, 0, 0, 0 };
        float zero  = 0.0f;    // stays zero while every weight is finite
        const T* src = reinterpret_cast<const T*>(p.b) + ((size_t)oc * p.taps + tap) * p.IC;
#pragma unroll
        for (int i = 0; i < PER; i++)
            if (G < p.granules && c0 + 4 * i < p.IC)
                v[i] = widen(src[c0 + 4 * i]), zero = __builtin_fmaf(v[i], 0.0f, zero);
        put_chunk<F64>(p.cb + ((size_t)oc * p.row_granules * 4 + at) * 16, v);
        if (zero != 0.0f)
            any_bad = 1;
    }
    __syncthreads();
    if (tid == 0)
        p.bad[blk] = any_bad;
}

// One workgroup of four waves, 2 x 2 of WT x WT results from (m0, n0) on.  WT 32: stages of two granules a row; WT 16: of four.
template <bool F64, int WT, int RING>
__device__ __forceinline__ void copied_tile(const CopiedArgs& p, int m0, int n0, uint8_t* lds)
{
    constexpr int PER = F64 ? 2 : 4;    // elements of a chunk
    constexpr int BM = 2 * WT, NGS = WT == 32 ? 2 : 4, RB = NGS * 64;    // rows of either operand, granules and bytes of a row's stage
    constexpr int STAGE = 2 * BM * RB, LANES = RB / 16, RPI = 64 / LANES;    // RPI: rows of a wave's load
    static_assert(STAGE == 16384, "sixteen loads of 1 KB a stage, four a wave: two of either operand");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave      = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint8_t *a_base = p.a, *b_base = p.b;
    // a row's chunks lie permuted, chunk c at c ^ turn(row), so that the 16 lanes the LDS serves together hit different banks
    auto turn = [](int row) { return WT == 32 ? (row >> 1) & 7 : row & 15; };

    uint32_t a_off[2], b_off[2];
    int a_gran[2];    // which granule of the stage the lane's chunk belongs to
#pragma unroll
    for (int j = 0; j < 2; j++)
    {
        const int row = (wave + 4 * j) * RPI + lane / LANES, c = (lane % LANES) ^ turn(row);
        int m         = m0 + row;
        m             = m < p.M ? m : p.M - 1;
        const uint32_t t = fdiv((uint32_t)m, p.ow), n = fdiv(t, p.oh);
        a_off[j]  = n * (uint32_t)p.image + (t - n * p.oh.d) * (uint32_t)p.pitch_y + ((uint32_t)m - t * p.ow.d) * (uint32_t)p.pitch_x + (c & 3) * 16;
        a_gran[j] = c >> 2;
        int oc    = n0 + row;
        oc        = oc < p.OC ? oc : p.OC - 1;
        b_off[j]  = (uint32_t)oc * (uint32_t)p.b_pitch + c * 16;
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds + wave * 1024;
    auto load = [&](uint32_t off, const uint8_t* base, uint32_t to) {
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "s"(to) : "memory");
    };
    // The next stage to request: its first granule's place in the channel vector, its tap's column, its offset.  Where a stage lies
    // inside one tap (whole: the channel vector is whole stages) that offset is scalar and the lanes' own never change.
    const bool whole = p.gp % NGS == 0;
    uint32_t a_lane[2];
#pragma unroll
    for (int j = 0; j < 2; j++)
        a_lane[j] = a_off[j] + (uint32_t)a_gran[j] * 64u;
    int piece = 0, kx = 0, next = 0;
    uint32_t walk = 0;
    auto request  = [&](int slot) {
        if (whole)
        {
            const uint8_t* base = a_base + walk;
            load(a_lane[0], base, lds0 + slot * STAGE);
            load(a_lane[1], base, lds0 + slot * STAGE + 4096);
            walk += RB;
            if ((piece += NGS) == p.gp)
            {
                piece = 0;
                walk += (uint32_t)p.next_tap;
                if (++kx == p.KW)
                    kx = 0, walk += (uint32_t)p.next_row;
            }
        }
        else
        {
            uint32_t off[NGS];
#pragma unroll
            for (int g = 0; g < NGS; g++)
            {
                off[g] = walk;
                walk += 64;
                if (++piece == p.gp)
                {
                    piece = 0;
                    walk += (uint32_t)p.next_tap;
                    if (++kx == p.KW)
                        kx = 0, walk += (uint32_t)p.next_row;
                }
            }
            const bool ragged = (next + 1) * NGS > p.granules;
#pragma unroll
            for (int j = 0; j < 2; j++)
            {
                uint32_t o = off[0];
#pragma unroll
                for (int g = 1; g < NGS; g++)
                    o = a_gran[j] == g ? off[g] : o;
                o += a_off[j];
                if (ragged && next * NGS + a_gran[j] >= p.granules)
                    o = (uint32_t)p.zero_off;
                load(o, a_base, lds0 + slot * STAGE + j * 4096);
            }
        }
#pragma unroll
        for (int j = 0; j < 2; j++)
            load(b_off[j], b_base, lds0 + slot * STAGE + 8192 + j * 4096);
        b_base += RB;
        next++;
    };

    const int wm = (wave >> 1) * WT, wn = (wave & 1) * WT, l16 = lane & 15, q = lane >> 4;
    using acc_t = sum_t<F64>;
    v4d acc64[WT == 32 ? 4 : 1];
    v16f acc32;
    v4f acc4 = { 0, 0, 0, 0 };
    if constexpr (F64)
    {
#pragma unroll
        for (int t = 0; t < (WT == 32 ? 4 : 1); t++)
            acc64[t] = v4d{ 0, 0, 0, 0 };
    }
    else
    {
#pragma unroll
        for (int t = 0; t < 16; t++)
            acc32[t] = 0.0f;
    }
    // fp32, 32 x 32 results: block q = lane / 16 of the operands is (row half q / 2, column half q % 2)
    const int arow = wm + (!F64 && WT == 32 ? 16 * (q >> 1) : 0) + l16, brow = wn + (!F64 && WT == 32 ? 16 * (q & 1) : 0) + l16;
    const uint8_t* arow_p = lds + arow * RB;
    const uint8_t* brow_p = lds + 8192 + brow * RB;
    const int S = p.stages;
    for (int s = 0; s < RING - 1 && s < S; s++)
        request(s);
    // The fragments of a step (fp64: a stage; fp32: sixteen instructions' worth) are read while the step before is multiplied, so
    // the wait and the barrier are for the stage after the present one.  Two sets of fragments; the ring is written out, so that
    // sets and stage addresses are constants.
    constexpr int T = F64 ? WT / 16 : 1, FR = F64 ? NGS : 4;    // fragments of either operand: FR x T
    constexpr int STEPS = !F64 && WT == 32 ? 2 : 1;
    static_assert(RING % 2 == 0, "two sets");
    using frag_t = std::conditional_t<F64, v2d, v4f>;
    frag_t fa[2][FR][T], fb[2][FR][T];
    const uint8_t *pa[STEPS * FR], *pb[STEPS * FR];
#pragma unroll
    for (int g = 0; g < STEPS * FR; g++)
    {
        // fp32, 32 x 32 results: a lane needs every k; else k % 4 = q
        const int c = STEPS == 2 ? g : 4 * g + q;
        pa[g] = arow_p + ((c ^ turn(arow)) << 4), pb[g] = brow_p + ((c ^ turn(brow)) << 4);    // (16 rows on, the permutation is the same)
    }
    auto fetch = [&](int set, int slot, int step) {
#pragma unroll
        for (int g = 0; g < FR; g++)
#pragma unroll
            for (int t = 0; t < T; t++)
            {
                fa[set][g][t] = *reinterpret_cast<const frag_t*>(pa[step * FR + g] + slot * STAGE + t * 16 * RB);
                fb[set][g][t] = *reinterpret_cast<const frag_t*>(pb[step * FR + g] + slot * STAGE + t * 16 * RB);
            }
    };
    // fp32: the products of the next k are under way while those of this one are added, also from one step to the next; the empty
    // asm keeps it at one product ahead
    v16f prod;
    auto product = [&](int set, int k) {
        const v16f zero = { 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0 };
        const int c = WT == 32 ? k & 3 : k >> 2, i = WT == 32 ? k >> 2 : k & 3;
        float x = (float)fa[set][c % FR][0][i % PER];
        if constexpr (WT == 32)
            asm volatile("" : "+v"(x), "+v"(acc32));
        else
            asm volatile("" : "+v"(x), "+v"(acc4));
        return __builtin_amdgcn_mfma_f32_16x16x1f32(x, (float)fb[set][c % FR][0][i % PER], zero, 0, 0, 0);
    };
    auto multiply = [&](int set, int g) {
        if constexpr (F64)
        {
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int t = 0; t < T * T; t++)
                    acc64[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[set][g][t / T][i], fb[set][g][t % T][i], acc64[t], 0, 0, 0);
        }
        else
        {
#pragma unroll
            for (int k = 4 * g; k < 4 * g + 4; k++)
            {
                const v16f ahead = k < 15 ? product(set, k + 1) : product(set ^ 1, 0);
#pragma unroll
                for (int t = 0; t < 16; t++)
                    if constexpr (WT == 32)
                        acc32[t] = acc32[t] + prod[t];
                    else
                        acc4[t & 3] = acc4[t & 3] + prod[t];    // the four blocks of an instruction are four k
                prod = ahead;
            }
        }
    };
    if (S >= RING - 1)
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((RING - 2) * 4) : "memory");
    else
        asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    fetch(0, 0, 0);
    if constexpr (!F64)
        prod = product(0, 0);
    for (int s0 = 0; s0 < S; s0 += RING)
    {
#pragma unroll
        for (int r = 0; r < RING; r++)
        {
            const int s = s0 + r;
            if (s >= S)
                break;
            // (every wave is past the stage before this one, whose slot the next request takes)
            if (s + RING - 1 <= S)
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((RING - 3) * 4) : "memory");
            else
                asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
            for (int step = 0; step < STEPS; step++)
            {
                const int set = STEPS == 2 ? step : r & 1;
                multiply(set, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (step == 0 && s + RING - 1 < S)
                    request((r + RING - 1) % RING);
                if (step + 1 < STEPS)
                    fetch(set ^ 1, r, step + 1);
                else
                    fetch(set ^ 1, (r + 1) % RING, 0);    // (behind the last stage: never used)
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int g = 1; g < FR; g++)
                    multiply(set, g);
            }
        }
    }

    auto store_result = [&](int m, int oc, acc_t v) {
        reinterpret_cast<acc_t*>(p.out)[(size_t)m * p.OC + oc] = v + reinterpret_cast<const acc_t*>(p.bias)[oc];
    };
    if (p.padded)
    {
        __syncthreads();    // the stages are free: the first word collects what the first launch met
        int& met = *reinterpret_cast<int*>(lds);
        if (tid == 0)
            met = 0;
        __syncthreads();
        const int rows = p.OC - n0 < BM ? p.OC - n0 : BM;
        int bad        = 0;
        for (int i = tid; i < rows * p.pieces; i += 256)
            bad |= p.bad[n0 * p.pieces + i];
        if (bad)
            met = 1;
        __syncthreads();
        if (met)
        {
            constexpr int KG = F64 ? 8 : 16;
            for (int t = tid; t < BM * BM; t += 256)
            {
                const int m = m0 + t / BM, oc = n0 + t % BM;
                if (m >= p.M || oc >= p.OC)
                    continue;
                const uint32_t r = fdiv((uint32_t)m, p.ow), n = fdiv(r, p.oh);
                const int oy = (int)(r - n * p.oh.d), ox = (int)((uint32_t)m - r * p.ow.d);
                const uint8_t* u = a_base + n * (uint32_t)p.image + oy * (uint32_t)p.pitch_y + ox * (uint32_t)p.pitch_x;
                const uint8_t* w = p.b + (uint32_t)oc * (uint32_t)p.b_pitch;
                acc_t sum        = 0;
                for (int ky = 0; ky < p.KH; ky++)
                {
                    for (int x = 0; x < p.KW; x++)
                    {
                        const int iy = oy * p.stride_y - p.pad_top + ky * p.dil_y, ix = ox * p.stride_x - p.pad_left + x * p.dil_x;
                        if ((unsigned)iy < (unsigned)p.IH && (unsigned)ix < (unsigned)p.IW)
                            for (int c = 0; c < p.IC; c++)
                            {
                                const int e = c % KG, at = c / KG * 64 + (e & 3) * 16 + (e >> 2) * (int)sizeof(acc_t);
                                sum         = sum + *reinterpret_cast<const acc_t*>(u + at) * *reinterpret_cast<const acc_t*>(w + at);
                            }
                        u += p.gp * 64 + p.next_tap, w += p.gp * 64;
                    }
                    u += p.next_row;
                }
                store_result(m, oc, sum);
            }
            return;
        }
    }
    if constexpr (F64)
    {
        // row lane / 16 + 4 r, column lane % 16
        constexpr int T = WT / 16;
#pragma unroll
        for (int t = 0; t < T * T; t++)
#pragma unroll
            for (int r = 0; r < 4; r++)
            {
                const int m = m0 + wm + 16 * (t / T) + q + 4 * r, oc = n0 + wn + 16 * (t % T) + l16;
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

// The first n_big tiles of 64 x 64 results whole, each of the others as four workgroups of 32 x 32.
template <bool F64, int RING>
__global__ __launch_bounds__(256, 2) void ordered_copied_kernel(CopiedArgs p)
{
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const uint32_t n_big = (uint32_t)p.n_big, n_quarters = 4 * ((uint32_t)p.tiles - n_big);
    if (p.big_first ? blockIdx.x < n_big : blockIdx.x >= n_quarters)
    {
        // neighbouring tiles share operand rows: a contiguous run of tiles for each of the eight L2s
        const uint32_t at = blockIdx.x - (p.big_first ? 0 : n_quarters), tile = (at & 7) * (n_big >> 3) + (at >> 3);
        const uint32_t tm = fdiv(tile, p.tiles_n), tn = tile - tm * p.tiles_n.d;
        copied_tile<F64, 32, RING>(p, (int)tm * 64, (int)tn * 64, lds);
        return;
    }
    const uint32_t quarter = blockIdx.x - (p.big_first ? n_big : 0), tile = n_big + (quarter >> 2);
    const uint32_t tm = fdiv(tile, p.tiles_n), tn = tile - tm * p.tiles_n.d;
    const int m0 = (int)tm * 64 + 32 * (int)((quarter >> 1) & 1), n0 = (int)tn * 64 + 32 * (int)(quarter & 1);
    if (m0 >= p.M || n0 >= p.OC)
        return;
    CopiedArgs half = p;    // (stages of four granules)
    half.stages     = (p.granules + 3) / 4;
    copied_tile<F64, 16, RING>(half, m0, n0, lds);
}

// Most bytes of the image's copy, and of the weights': what the caches behind the L2s keep until it is read again (fp32 [..]->8 3x3 with
// 80 MB of copies: 478 us, 343 by ordered_gemm.hip; at 28 and 41 MB the copies still lead, below).
constexpr int64_t kMostImage = 44 << 20;

struct CopyPlan
{
    size_t a_bytes, b_bytes, bias_bytes, bad_bytes, total;
    int64_t a_chunks, rows_y, rows_x, gp, granules, row_granules, pieces;
};
static size_t up256(size_t v)
{
    return (v + 255) / 256 * 256;
}
static bool plan_copies(CopyPlan& c, const ConvGeom& g, bool f64)
{
    const int64_t kg = f64 ? 8 : 16;
    c.gp           = (g.IC + kg - 1) / kg;
    c.granules     = (int64_t)g.KH * g.KW * c.gp;
    c.row_granules = (c.granules + 3) / 4 * 4;
    c.rows_y       = (int64_t)(g.OH - 1) * g.stride_y + (int64_t)(g.KH - 1) * g.dil_y + 1;
    c.rows_x       = (int64_t)(g.OW - 1) * g.stride_x + (int64_t)(g.KW - 1) * g.dil_x + 1;
    if (c.rows_y > INT32_MAX || c.rows_x > INT32_MAX || c.granules > INT32_MAX / 64 || g.N * c.rows_y > INT32_MAX / c.rows_x ||
        g.N * c.rows_y * c.rows_x > kMostImage / 64 / c.gp || g.OC > kMostImage / 64 / c.row_granules)
        return false;
    c.a_chunks   = g.N * c.rows_y * c.rows_x * c.gp * 4;
    c.pieces     = (c.row_granules * 4 + 255) / 256;
    c.a_bytes    = up256((size_t)c.a_chunks * 16 + 64);
    c.b_bytes    = up256((size_t)g.OC * c.row_granules * 64);
    c.bias_bytes = up256((size_t)g.OC * 8);
    c.bad_bytes  = up256((size_t)g.OC * c.pieces * 4);
    c.total      = c.a_bytes + c.b_bytes + c.bias_bytes + c.bad_bytes;
    return true;
}

// Whether the copies pay, for what ordered_staged.hip leaves (channel vectors of no whole units of eight; times of such vectors below are from
// before it): their launch costs 3 us and the bytes written, and gains what ordered_gemm.hip spends on conversions, on masks and
// on waiting for stages it fetches through registers; most for channel vectors that end inside a group of four, which it reads
// element by element.  us by ordered_gemm.hip / here, 3x3 unless noted, K = taps x channels:
//   fp64, IC % 4 != 0: K 225 17.4 / 12.2, 603 68 / 36, 1125 54 / 19, 1773 228 / 164, 3294 151 / 59; 135 11.0 / 9.4, 90 7.0 / 8.9, 81 10.1 /
//     14.4; 1x1: 145 11.3 / 10.4, 113 18.8 / 22.1
//   fp64, IC % 4 = 0: K 936 25.4 / 23.8, 1152 26 / 19, 2304 [4,56,56,256]->256 257 / 232, 2592 51 / 34 (few tiles) and 196.0 / 195.6 (495
//     tiles), 4392 121 / 72; 648 56 / 66 (355 tiles) and 20.0 / 17.2 (23), 504 25 / 30; 1x1 424 19.4 / 24.4
//   fp32, IC % 4 != 0: K 405 18.0 / 13.7, 846 50 / 41, 1125 44 / 23, 2178 (625 tiles) 276 / 223, 3114 282 / 187; 306 14.9 / 14.9
//   fp32, IC % 4 = 0, up to 64 tiles: K 1008 28.2 / 24.5, 1296 37 / 30, 2232 61 / 41, 3312 89 / 61, 504 and shorter 0.9x; channels of whole
//     stages (IC % 32 = 0, which ordered_gemm.hip reads without decodes): 1440 30.6 / 31.7, 1728 36.0 / 36.5, 3168 62 / 63; more tiles, whose
//     additions and products fill the SIMDs either way: 1944 (150) 77 / 82, 2304 (784) 272 / 302
static bool copies_lead(const ConvGeom& g, bool f64)
{
    const int64_t K = (int64_t)g.KH * g.KW * g.IC;
    if (g.KH * g.KW < 4)    // (an image that is read once or twice)
        return false;
    const int64_t tiles = (((int64_t)g.N * g.OH * g.OW + 63) / 64) * ((g.OC + 63) / 64);
    // Rows of both operands for half a tile of results, over and over: fp32 610 tiles, K 425 59 / 102, 923 tiles, K 909 133 / 182, fp64 990 tiles,
    // K 630 111 / 136, IC % 4 = 0: 632 tiles, K 1008 102 / 124, 875, K 1100 1.7 x; the other way fp32 571 tiles, K 1233 166 / 146, fp64 608, K 810 134 / 92.
    if (g.OC <= 32 && tiles > 600)
        return false;
    // The chain grows by what fills the granules up (8 elements in fp64, 16 in fp32).  Times of ordered_gemm.hip's by channels, large windows: fp32 3
    // channels 2.8, 6 1.3, 10 1.1 and from K 800 on 0.9, 11 0.9, 4 2.7, 8 1.4, 20 1.2, 12 and 24 1.0, 28 0.85; fp64 2 1.5, 3 1.1, 5 0.8, 4 1.4, 12 0.94, 20 0.85.
    const int64_t kg  = f64 ? 8 : 16;
    const double fill = (double)((g.IC + kg - 1) / kg * kg) / g.IC;
    if (fill > (g.IC % 4 != 0 ? (f64 ? 1.8 : (K >= 800 ? 2.2 : 1.6)) : (f64 ? 1.34 : 1.3)))
        return false;
    // (129 ... 192 tiles, all quarters, fp32: K 425 27.5 / 37.7, 475 30.5 / 39.5, 567 37.0 / 33.7)
    if (g.IC % 4 != 0)
        return K >= (f64 ? 200 : (tiles > 128 && tiles <= 192 ? 500 : 400));
    return K > 900 && (f64 || (tiles <= 64 && g.IC % 32 != 0));
}

size_t ordered_conv_copies_bytes(bool f64, const ConvGeom& g)
{
    CopyPlan c;
    return copies_lead(g, f64) && plan_copies(c, g, f64) ? c.total : 0;
}

// Splits `copies` into the parts of the plan and fills what both launches share.
static void place_copies(const CopyPlan& c, void* copies, CopyArgs& k, CopiedArgs& p)
{
    k.ca = (uint8_t*)copies, k.cb = k.ca + c.a_bytes, k.cbias = k.cb + c.b_bytes, k.bad = (int32_t*)(k.cbias + c.bias_bytes);
    k.a_chunks = (int32_t)c.a_chunks, k.a_blocks = (int32_t)((c.a_chunks + 255) / 256);
    k.gp = (int32_t)c.gp, k.granules = (int32_t)c.granules, k.row_granules = (int32_t)c.row_granules, k.pieces = (int32_t)c.pieces;
    k.div_gp4 = make_fastdiv((uint32_t)c.gp * 4), k.div_gp = make_fastdiv((uint32_t)c.gp), k.div_pieces = make_fastdiv((uint32_t)c.pieces);
    p.a = k.ca, p.b = k.cb, p.bias = k.cbias, p.bad = k.bad;
    p.gp = (int32_t)c.gp, p.granules = (int32_t)c.granules, p.stages = (int32_t)((c.granules + 1) / 2);
    p.zero_off = (int32_t)(c.a_chunks * 16), p.b_pitch = (int32_t)(c.row_granules * 64), p.pieces = (int32_t)c.pieces;
}

template <bool F64>
static bool launch_copied(hipStream_t st, CopiedArgs& p)
{
    // Whole tiles by rounds of one per CU, what is left over as quarters (see ordered_gemm.hip)
    const int64_t tn = (p.OC + 63) / 64, tiles = (int64_t)((p.M + 63) / 64) * tn, over = tiles % 256;
    if (tiles > INT32_MAX / 4 || !fastdiv_exact_up_to((uint64_t)tiles, (uint32_t)tn))
        return false;
    p.tiles   = (int32_t)tiles;
    p.tiles_n = make_fastdiv((uint32_t)tn);
    p.n_big   = tiles <= 192 || p.OC <= 32 ? 0 : (int32_t)(over <= 192 ? tiles - over : tiles / 8 * 8);
    const int64_t grid = p.n_big + 4 * (tiles - p.n_big);
    // Quarters first, whose chain of dependent instructions is as long as a whole tile's and runs beside those - but where all do not fit at once (two
    // workgroups a CU), for whole tiles would then wait for quarters to end.  us by ordered_gemm.hip / quarters first / whole tiles first: fp32 327 tiles,
    // K 525 57 / 75 / 56, 390 tiles, K 2225 228 / 219 / 169, fp64 364 tiles, K 1107 111 / 103 / 71, IC % 4 = 0: 420 tiles, K 1656 127 / 154 / 121.
    p.big_first = grid > 512;
    // few workgroups: a long ring, for the waves of one workgroup hide nothing of each other's loads
    const bool longer = grid <= 256 && ensure_dynamic_lds<ordered_copied_kernel<F64, 8>>(8 * 16384);
    if (longer)
        hipLaunchKernelGGL((ordered_copied_kernel<F64, 8>), dim3((unsigned)grid), dim3(256), 8 * 16384, st, p);
    else if (ensure_dynamic_lds<ordered_copied_kernel<F64, 4>>(4 * 16384))
        hipLaunchKernelGGL((ordered_copied_kernel<F64, 4>), dim3((unsigned)grid), dim3(256), 4 * 16384, st, p);
    else
        return false;
    return true;
}

static bool launch_copies(hipStream_t st, int32_t in_dtype, bool f64, const CopyArgs& k)
{
    const dim3 grid((unsigned)(k.a_blocks + k.b_blocks + 1));
    if (!f64)
    {
        if (in_dtype != TMI_FP32)
            return false;
        hipLaunchKernelGGL((ordered_copy_kernel<float, false>), grid, dim3(256), 0, st, k);
        return true;
    }
    switch (in_dtype)
    {
        case TMI_FP16: hipLaunchKernelGGL((ordered_copy_kernel<_Float16, true>), grid, dim3(256), 0, st, k); return true;
        case TMI_BF16: hipLaunchKernelGGL((ordered_copy_kernel<bf16_t, true>), grid, dim3(256), 0, st, k); return true;
        case TMI_FP32: hipLaunchKernelGGL((ordered_copy_kernel<float, true>), grid, dim3(256), 0, st, k); return true;
        default: return false;
    }
}

bool launch_ordered_conv_copied(hipStream_t st, int32_t in_dtype, bool f64, const ConvGeom& g, const void* in, const void* w,
                                const void* bias, bool abs_mode, const double* input_abs_max, void* out, void* copies)
{
    CopyPlan c;
    const int64_t pixels = (int64_t)g.N * g.OH * g.OW;
    if (!copies || !plan_copies(c, g, f64) || pixels > INT32_MAX - 64 || !fastdiv_exact_up_to((uint64_t)pixels, (uint32_t)g.OW) ||
        !fastdiv_exact_up_to((uint64_t)pixels / g.OW, (uint32_t)g.OH) || !fastdiv_exact_up_to((uint64_t)c.a_chunks + 256, (uint32_t)c.gp * 4) ||
        !fastdiv_exact_up_to((uint64_t)(g.N * c.rows_y * c.rows_x) + 64, (uint32_t)c.rows_x) ||
        !fastdiv_exact_up_to((uint64_t)(g.N * c.rows_y) + 64, (uint32_t)c.rows_y) || !fastdiv_exact_up_to((uint64_t)g.OC * c.pieces, (uint32_t)c.pieces) ||
        !fastdiv_exact_up_to((uint64_t)c.row_granules, (uint32_t)c.gp))
        return false;
    CopyArgs k{};
    CopiedArgs p{};
    place_copies(c, copies, k, p);
    k.a = in, k.b = w, k.bias = bias, k.input_abs_max = input_abs_max, k.abs_mask = abs_mode ? 0x7fffffffu : ~0u;
    k.IC = g.IC, k.OC = g.OC, k.IH = g.IH, k.IW = g.IW, k.taps = g.KH * g.KW, k.bias_len = g.bias_len;
    k.pad_top = g.pad_top, k.pad_left = g.pad_left;
    k.b_blocks = (int32_t)(g.OC * c.pieces);
    k.div_w = make_fastdiv((uint32_t)c.rows_x), k.div_h = make_fastdiv((uint32_t)c.rows_y);
    const int32_t pixel = (int32_t)(c.gp * 64), row = (int32_t)(c.rows_x * pixel);
    p.out = out, p.M = (int32_t)pixels, p.OC = g.OC, p.KW = g.KW, p.KH = g.KH;
    p.pitch_x = g.stride_x * pixel, p.pitch_y = g.stride_y * row, p.image = (int32_t)(c.rows_y * row);
    p.next_tap = (g.dil_x - 1) * pixel, p.next_row = g.dil_y * row - g.KW * g.dil_x * pixel;
    p.IC = g.IC, p.IH = g.IH, p.IW = g.IW, p.pad_top = g.pad_top, p.pad_left = g.pad_left;
    p.stride_y = g.stride_y, p.stride_x = g.stride_x, p.dil_y = g.dil_y, p.dil_x = g.dil_x;
    p.ow = make_fastdiv((uint32_t)g.OW), p.oh = make_fastdiv((uint32_t)g.OH);
    // (the bounds pass multiplies the padding out, tensor_ops.cpp:845-852: an infinite weight there makes NaN, as the zeros in the copy do)
    p.padded = !abs_mode && (g.pad_top > 0 || g.pad_left > 0 || c.rows_y - g.pad_top > g.IH || c.rows_x - g.pad_left > g.IW);
    if (!launch_copies(st, in_dtype, f64, k))
        return false;
    return f64 ? launch_copied<true>(st, p) : launch_copied<false>(st, p);
}

}    // namespace tmi
