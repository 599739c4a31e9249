// MATMUL int8 -> int32 and fp16 / bf16 -> fp32 of any size and alignment, for products the GEMM kernel does not read in place
// or that offer it too few tiles: rows that are no multiple of 64 bytes, columns that are no whole 16-byte pieces, few rows.
//
// A tile is 32 rows x 64 columns and SPLIT waves share its K, a block of 64 bytes of K (two matrix instructions deep) at a
// time, dealt round-robin.  Nothing is shared between waves before the end: a wave takes its part of the first operand
// straight into the registers the matrix instruction reads (lane = row lane % 32, 16 bytes of K of half lane / 32), and moves
// its part of the second operand, [K][W] as it lies, through a piece of LDS of its own, from which the transposing reads
// (ds_read_b64_tr_b16 / _b8) return K-contiguous fragments; the next block's loads are in flight meanwhile.  Loads are 16 bytes
// from any address (gfx950 takes global addresses of any alignment), the last of a tensor from its last 16 bytes.  The partial
// tiles meet in LDS.  Rows of the tile are rows of the result, so that 32 lanes store 128 neighbouring bytes.  Workgroups of
// neighbouring tiles share an L2 (us without / with: fp16 7 x [78,853]x[853,2096] 20.6 / 17.2, int8 [1,4096]x[4096,4096] 8.7 / 6.5; fp16
// the same 10.0 / 10.7).
//
// What bounds it: the first operand's fragments, a line per lane and load, for products of many tiles (fp16 at 130 TFLOP/s), the
// chain of a wave's blocks otherwise.  us transposed copy + patch or GEMM kernel -> here: fp16 96 x [197,64]x[64,197] 33.6 -> 8.2
// (34 MB with the next: 2.4 TB/s), 96 x [197,197]x[197,64] 45.3 -> 6.2, [1,4096]x[4096,4096] 49.7 -> 9.4, int8 4 x [700,701]x[701,703]
// 13.4 (20.8 before its ends were read in one piece, 13.4 before its rows were read from words), [64,512]x[512,512] 11.5 -> 4.8.
#include <type_traits>

#include "tmi_mfma.h"

namespace tmi
{

struct RaggedArgs
{
    const uint8_t* a;
    const uint8_t* b;
    uint8_t* out;    // 4-byte results
    int64_t a_total, b_total;    // bytes of the whole operands
    int32_t H, C, W;
    int32_t za, zb;
    int32_t odd;      // bit 0 / 1: rows of the first / second operand begin between words
    int32_t tiles;    // of all batches
    uint32_t per_xcd;    // workgroups / 8, rounded down
    FastDiv per_batch, tiles_w;
};

// the first n bytes at p (n may be 0 or negative), then zeros
template <int EB>
__device__ __forceinline__ v4i load_front(const uint8_t* p, int n)
{
    if (n >= 16)
        return load16(p);
    uint32_t d[4] = { 0, 0, 0, 0 };
#pragma unroll
    for (int i = 0; i < 16; i += EB)
        if (i < n)
        {
            const uint32_t e = EB == 1 ? *(p + i) : *reinterpret_cast<const uint16_t*>(p + i);
            d[i >> 2] |= e << (8 * (i & 3));
        }
    return v4i{ (int)d[0], (int)d[1], (int)d[2], (int)d[3] };
}

// bytes of LDS of a wave: a block of the second operand, then its partial tile
template <typename T, int SPLIT, int NC>
constexpr int ragged_wave_lds()
{
    constexpr int EB = (int)sizeof(T), block = 64 / EB * (32 * NC * EB + (NC == 2 ? 32 * EB : 0));
    return SPLIT > 1 && block < 4096 * NC ? 4096 * NC : block;
}

// NC: column blocks of 32 in a tile.  TINY: an operand of less than 16 bytes, or a tile beyond 32-bit offsets: 64-bit ones, and pieces of less than
// 16 bytes element by element
// ODD: rows of an operand begin between words
template <typename T, int SPLIT, int NC, bool TINY, bool ODD>
__global__ __launch_bounds__(SPLIT > 4 ? 64 * SPLIT : 256) void matmul_ragged_kernel(RaggedArgs p)
{
    using M             = Mma<T>;
    using acc_t         = typename M::acc_t;
    using word          = std::conditional_t<M::is_int, int32_t, float>;
    constexpr int EB    = (int)sizeof(T);
    constexpr int KB    = 64 / EB;              // k of a block
    constexpr int RB    = 32 * NC * EB;         // bytes of a k row of the tile
    constexpr int LD    = RB + (NC == 2 ? 32 * EB : 0);    // the 4 (8) k rows x 64 (32) bytes of a transposing read touch every bank once
    constexpr int CPR   = RB / 16;              // 16-byte pieces of a k row
    constexpr int NL    = KB * CPR / 64;        // loads of the second operand per lane and block
    constexpr int kWaves = SPLIT > 4 ? SPLIT : 4;
    constexpr int kWaveLds = ragged_wave_lds<T, SPLIT, NC>();
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];

    // The arguments at once.  (Left to the compiler they come where they are used, seven trips one after the other before the first load: int8
    // [249,64]x[64,96] 4.11 us, so 3.71.)
    asm volatile("" : "+s"(p.a_total), "+s"(p.b_total), "+s"(p.H), "+s"(p.C), "+s"(p.W), "+s"(p.za), "+s"(p.zb), "+s"(p.odd), "+s"(p.tiles), "+s"(p.per_xcd)
                 : "s"(p.a), "s"(p.b), "s"(p.out));

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r32 = lane & 31, half = lane >> 5;
    // a contiguous run of tiles for each of the eight L2s (workgroups go to them in turn)
    uint32_t bid = blockIdx.x;
    if (bid < p.per_xcd * 8)
        bid = (bid & 7) * p.per_xcd + (bid >> 3);
    const uint32_t tile = (bid * kWaves + wave) / SPLIT;
    if (SPLIT < kWaves && SPLIT == 1 && tile >= (uint32_t)p.tiles)
        return;
    const bool live      = tile < (uint32_t)p.tiles;
    const uint32_t t     = live ? tile : 0;
    const uint32_t batch = fdiv(t, p.per_batch), in_batch = t - batch * p.per_batch.d, th = fdiv(in_batch, p.tiles_w);
    const int h0 = (int)th * 32, w0 = (int)(in_batch - th * p.tiles_w.d) * 32 * NC;
    uint8_t* mine = lds + wave * kWaveLds;

    const int row_bytes = p.C * EB, piece = (lane & (CPR - 1)) * 16, krow = lane / CPR;    // (krow: k row of the lane's first load)
    const int rows      = p.H - h0 < 32 ? p.H - h0 : 32;
    const int64_t pitch = (int64_t)p.W * EB;
    const int64_t a_tile = ((int64_t)batch * p.H + h0) * row_bytes, b_tile = (int64_t)batch * p.C * pitch + (int64_t)w0 * EB;
    const uint32_t a_lane = (uint32_t)(r32 < rows ? r32 : rows - 1) * (uint32_t)row_bytes + 16 * half, b_lane = (uint32_t)krow * (uint32_t)pitch + piece;
    const int blocks = (p.C + KB - 1) / KB, first = wave % SPLIT;
    const int shares = live && first < blocks ? (blocks - first + SPLIT - 1) / SPLIT : 0;    // blocks of this wave

    // Loads are 16 bytes wherever they begin, at the last 16 bytes of the tensor at the latest; what they bring from behind a row of the
    // first operand, from behind K or from before their place (the end of the tensor) goes in finish(), which loads nothing.  (Where the
    // ends were read element by element, a wave waited for eight loads one after the other: us then / now, fp16 96 x [197,197]x[197,64]
    // 8.0 / 7.2, 10 x [55,40]x[40,55] 6.3 / 4.0, int8 8 x [4,125]x[125,922] 6.7 / 4.5.  Two and three blocks of registers instead of one: the
    // products of many tiles lose more to fewer waves than they gain, fp16 127 x [203,128]x[128,203] 15.5 / 19.1 with three.)
    struct Place
    {
        const uint8_t* base;
        uint32_t extra, most;    // what to add to an offset, and how large the sum may be
    };
    auto place = [&](const uint8_t* t, int64_t total, int64_t at) {
        const int64_t to = at < total - 16 ? at : total - 16, room = total - 16 - to;
        return Place{ t + to, (uint32_t)(at - to), room < INT32_MAX ? (uint32_t)room : (uint32_t)INT32_MAX };
    };
    // A 16-byte load from between words occupies the memory pipeline for two and a half times as long (64 lanes, two to a row: 246 clocks,
    // 92 from a word on).  Such rows are read from the word before; what a lane then lacks is the next piece's first word, which another
    // lane has, and for the last piece is loaded (112 clocks).  Where a row's pieces begin in a word does not change along K.
    // us before / now: bf16 2 x [64,2265]x[2265,796] 15.4 / 10.2, 2 x [14,2529]x[2529,160] 11.0 / 6.8, 2 x [758,191]x[191,1668] 13.5 / 9.6, fp16
    // 96 x [197,197]x[197,64] 7.4 / 6.2, int8 8 x [300,701]x[701,701] 15.0 / 12.2.  The second operand's rows, whose pieces lie side by side, gain
    // where a wave has a tile to itself, in 16 bits (fp16 96 x [197,64]x[64,197] 8.9 / 8.2, 8 x [1500,64]x[64,2001] 28.0 / 23.9); not where K is shared
    // (bf16 2 x [64,2272]x[2272,797] 8.7 / 9.3) nor in int8 (64 x [200,64]x[64,301] 7.7 / 8.0).
    constexpr bool kRealignB = SPLIT == 1 && EB == 2;
    const bool odd_a = ODD && (p.odd & 1), odd_b = ODD && kRealignB && (p.odd & 2), last_piece = (lane & (CPR - 1)) == CPR - 1;
    const int shift_a = odd_a ? (int)((uintptr_t)(p.a + a_tile + a_lane) & 3) : 0, shift_b = odd_b ? (int)((uintptr_t)(p.b + b_tile + b_lane) & 3) : 0;
    auto k_ends = [&](int k0) { return k0 + KB > p.C; };
    auto b_ends = [&](int k0) { return k_ends(k0) || b_tile + (k0 + KB - 1) * pitch + RB > p.b_total; };
    v4i av[2], bv[NL];
    int a_next = 0, b_next[NL] = {};    // the word behind a lane's last piece
    auto words  = [&](const uint8_t* at) {
        v4i v;
        __builtin_memcpy(&v, __builtin_assume_aligned(at, 4), 16);
        return v;
    };
    auto request = [&](int share) {
        const int k0 = (first + share * SPLIT) * KB;
        if constexpr (TINY)
        {
#pragma unroll
            for (int j = 0; j < 2; j++)
                av[j] = load_front<EB>(p.a + a_tile + (int64_t)(r32 < rows ? r32 : rows - 1) * row_bytes + 16 * half + k0 * EB + 32 * j, row_bytes - k0 * EB - 16 * half - 32 * j);
#pragma unroll
            for (int j = 0; j < NL; j++)
            {
                const int k      = k0 + krow + j * (64 / CPR);
                const int64_t at = b_tile + k * pitch + piece, left = p.b_total - at;
                bv[j]         = load_front<EB>(p.b + at, k < p.C ? (left < 16 ? (int)left : 16) : 0);
            }
            return;
        }
        const Place pa = place(p.a, p.a_total, a_tile + k0 * EB), pb = place(p.b, p.b_total, b_tile + k0 * pitch);
        if (odd_a && !k_ends(k0))
        {
            const uint8_t* at = pa.base + a_lane - shift_a;
            av[0] = words(at), av[1] = words(at + 32);
            if (half)
                a_next = *reinterpret_cast<const int*>(at + 32 + (shift_a ? 16 : 12));    // (a word of the row either way)
        }
        else
#pragma unroll
            for (int j = 0; j < 2; j++)
            {
                const uint32_t off = a_lane + pa.extra + 32 * j;
                av[j]           = load16(pa.base + (off < pa.most ? off : pa.most));
            }
        if (odd_b && !b_ends(k0))
        {
#pragma unroll
            for (int j = 0; j < NL; j++)
            {
                const uint8_t* at = pb.base + b_lane - shift_b + j * (64 / CPR) * (uint32_t)pitch;
                bv[j]             = words(at);
                if (last_piece)
                    b_next[j] = *reinterpret_cast<const int*>(at + (shift_b ? 16 : 12));
            }
        }
        else
#pragma unroll
            for (int j = 0; j < NL; j++)
            {
                const uint32_t off = b_lane + pb.extra + j * (64 / CPR) * (uint32_t)pitch;
                bv[j]           = load16(pb.base + (off < pb.most ? off : pb.most));
            }
    };
    auto shifted = [&](v4i v, int next, int by) {
#pragma unroll
        for (int k = 0; k < 4; k++)
            v[k] = (int)__builtin_amdgcn_alignbyte((uint32_t)(k < 3 ? v[k < 3 ? k + 1 : 3] : next), (uint32_t)v[k], by);
        return v;
    };
    auto finish = [&](int share) {
        int k0 = (first + share * SPLIT) * KB;
        asm volatile("" : "+s"(k0));    // (worked out again rather than kept from request())
        const bool k_tail = k_ends(k0);
        if (odd_a && !k_tail)
        {
            // pieces in K order: lower half's first, upper half's first, lower half's second, upper half's second
            const auto first_words = __builtin_amdgcn_permlane32_swap((uint32_t)av[0][0], (uint32_t)av[1][0], false, false);
            const auto upper_words = __builtin_amdgcn_permlane32_swap((uint32_t)av[1][0], (uint32_t)av[1][0], false, false);
            av[0] = shifted(av[0], (int)(half ? first_words[0] : first_words[1]), shift_a);
            av[1] = shifted(av[1], half ? a_next : (int)upper_words[1], shift_a);
        }
        if (odd_b && !b_ends(k0))
#pragma unroll
            for (int j = 0; j < NL; j++)
            {
                const int right = __builtin_amdgcn_update_dpp(0, bv[j][0], 0x101, 0xf, 0xf, true);    // (the lane to the right; pieces of a row are 2, 4 or 8 lanes)
                bv[j]           = shifted(bv[j], last_piece ? b_next[j] : right, shift_b);
            }
        if (k_tail)
        {
            const Place pa = place(p.a, p.a_total, a_tile + k0 * EB);
#pragma unroll
            for (int j = 0; j < 2; j++)
            {
                const uint32_t off = a_lane + pa.extra + 32 * j;
                if (off > pa.most)
                    av[j] = drop_bytes(av[j], (int)(off - pa.most) & 15);
                av[j] = keep_bytes(av[j], row_bytes - k0 * EB - 16 * half - 32 * j);
            }
        }
        if (b_ends(k0))
        {
            const Place pb = place(p.b, p.b_total, b_tile + k0 * pitch);
#pragma unroll
            for (int j = 0; j < NL; j++)
            {
                const uint32_t off = b_lane + pb.extra + j * (64 / CPR) * (uint32_t)pitch;
                if (off > pb.most)
                    bv[j] = drop_bytes(bv[j], (int)(off - pb.most) & 15);
                if (k0 + krow + j * (64 / CPR) >= p.C)
                    bv[j] = v4i{ 0, 0, 0, 0 };
            }
        }
    };

    acc_t acc[NC];
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
        for (int i = 0; i < 16; i++)
            acc[c][i] = 0;
    int sum_a = 0, sum_b[NC] = {};    // of the lane's row and columns (int8)
    const bool sums = M::is_int && (p.za | p.zb) != 0;

    // source of a transposing read: k row sl / 4 of four (sl / 2 of eight), 8 bytes of columns; see the GEMM kernel
    const int sl = lane & 15, cblk = (lane >> 4) & 1;
    const int tr = EB == 2 ? (8 * half + (sl >> 2)) * LD + (16 * cblk + 4 * (sl & 3)) * 2 : (16 * half + (sl >> 1)) * LD + 16 * cblk + 8 * (sl & 1);
    if (shares > 0)
        request(0);
    for (int i = 0; i < shares; i++)
    {
        if constexpr (!TINY)
            finish(i);
#pragma unroll
        for (int j = 0; j < NL; j++)
            *reinterpret_cast<v4i*>(mine + (krow + j * (64 / CPR)) * LD + (lane & (CPR - 1)) * 16) = bv[j];
        const v4i a0 = av[0], a1 = av[1];
        __builtin_amdgcn_wave_barrier();
        if (i + 1 < shares)
            request(i + 1);
#pragma unroll
        for (int s = 0; s < 2; s++)
        {
            const v4i a = s ? a1 : a0;
            if (sums)
                sum_a += dot4_ones(a);
#pragma unroll
            for (int c = 0; c < NC; c++)
            {
                v4i b;
#pragma unroll
                for (int r = 0; r < 2; r++)
                {
                    const uint8_t* src = mine + tr + (KB / 2 * s + KB / 8 * r) * LD + 32 * c * EB;
                    v2i part;
                    if constexpr (EB == 2)
                        part = __builtin_bit_cast(v2i, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s*)src));
                    else
                        part = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) v2i*)src);
                    b[2 * r] = part.x, b[2 * r + 1] = part.y;
                }
                if (sums)
                    sum_b[c] += dot4_ones(b);
                acc[c] = M::mma(a, b, acc[c]);
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
    if (sums)
    {
        // each share brings its own part of the correction
        sum_a += __shfl_xor(sum_a, 32);
#pragma unroll
        for (int c = 0; c < NC; c++)
        {
            const int col = p.za * (sum_b[c] + __shfl_xor(sum_b[c], 32)) - (first == 0 ? p.C * p.za * p.zb : 0);
#pragma unroll
            for (int i = 0; i < 16; i++)
                acc[c][i] -= (word)(col + p.zb * __shfl(sum_a, 8 * (i >> 2) + 4 * half + (i & 3)));
        }
    }
    word* out   = reinterpret_cast<word*>(p.out) + (int64_t)batch * p.H * p.W;
    auto store  = [&](int c, int i, word v) {
        const int r = h0 + 8 * (i >> 2) + 4 * half + (i & 3), col = w0 + 32 * c + r32;
        if (r < p.H && col < p.W)
            out[(int64_t)r * p.W + col] = v;
    };
    if constexpr (SPLIT == 1)
    {
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
            for (int i = 0; i < 16; i++)
                store(c, i, acc[c][i]);
    }
    else
    {
        // a wave's partial tile in its own 8 KB (its reads of the second operand are done), then 1 / SPLIT of the sums each
        word* part = reinterpret_cast<word*>(mine);
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
            for (int i = 0; i < 16; i++)
                part[(16 * c + i) * 64 + lane] = acc[c][i];
        __syncthreads();
        if (!live)
            return;
        const uint8_t* base = lds + wave / SPLIT * SPLIT * kWaveLds;
        constexpr int kEach = 16 * NC / SPLIT;
#pragma unroll
        for (int e = 0; e < kEach; e++)
        {
            const int j = first * kEach + e;
            word v      = reinterpret_cast<const word*>(base)[j * 64 + lane];
#pragma unroll
            for (int s = 1; s < SPLIT; s++)
                v += reinterpret_cast<const word*>(base + s * kWaveLds)[j * 64 + lane];
            store(j >> 4, j & 15, v);
        }
    }
}

// Aligned copies of both operands for the GEMM kernel, in one launch: rows of the first become CP elements (a multiple of 64 bytes), the second
// [N][C][W] becomes [N][CP][ldw bytes]; what is added holds the zero point, so that it contributes nothing.
struct PadArgs
{
    const uint8_t* a;
    const uint8_t* b;
    uint8_t* ap;
    uint8_t* bp;
    int64_t units_a, units_b;    // 16-byte units of the copies (units_a 0: the first operand is read in place)
    int32_t row_a, row_b;        // bytes of a row of each operand
    int32_t C;
    uint32_t fill_a, fill_b;     // zero points, replicated
    FastDiv ua, ub, cp;          // units per padded row, padded k rows per batch
};

template <int EB>
__global__ __launch_bounds__(256) void pad_operands_kernel(PadArgs p, int32_t blocks)
{
    for (int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x; u < p.units_a + p.units_b; u += (int64_t)blocks * 256)
    {
        const bool is_b   = u >= p.units_a;
        const int64_t v   = is_b ? u - p.units_a : u;
        const uint32_t d  = is_b ? p.ub.d : p.ua.d;
        const int64_t row = v / d;
        const int at      = (int)(v - row * d) * 16, bytes = is_b ? p.row_b : p.row_a;
        const uint32_t fill = is_b ? p.fill_b : p.fill_a;
        int64_t src_row   = row;
        int left          = bytes - at;
        if (is_b)
        {
            const int64_t n = row / p.cp.d;
            const int k     = (int)(row - n * p.cp.d);
            src_row         = n * p.C + k;
            left            = k < p.C ? left : 0;
        }
        v4i q = { (int)fill, (int)fill, (int)fill, (int)fill };
        if (left >= 16)
            q = load16((is_b ? p.b : p.a) + src_row * bytes + at);
        else if (left > 0)
        {
            q = load_front<EB>((is_b ? p.b : p.a) + src_row * bytes + at, left);
#pragma unroll
            for (int i = 0; i < 4; i++)
            {
                const int keep      = left - 4 * i;    // bytes of the word that are the operand's
                const uint32_t mask = keep >= 4 ? ~0u : (keep <= 0 ? 0u : (1u << (8 * keep)) - 1u);
                q[i]                = (int)(((uint32_t)q[i] & mask) | (fill & ~mask));
            }
        }
        *reinterpret_cast<v4i*>((is_b ? p.bp : p.ap) + v * 16) = q;
    }
}

// geometry of those copies; pad_a false: the first operand stays where it is
void matmul_padded_sizes(int32_t eb, int32_t N, int32_t H, int32_t C, int32_t W, MatmulPad& m)
{
    m.pad_a   = (int64_t)C * eb % 64 != 0;
    m.CP      = (int32_t)(((int64_t)C * eb + 63) / 64 * 64 / eb);
    m.ldw     = ((int64_t)W * eb + 15) / 16 * 16;
    m.a_bytes = m.pad_a ? (size_t)N * H * m.CP * eb : 0;
    m.b_bytes = (size_t)N * m.CP * m.ldw;
}

bool launch_matmul_pad(hipStream_t st, int32_t eb, int32_t N, int32_t H, int32_t C, int32_t W, const MatmulPad& m, const void* a, const void* b,
                       int32_t a_zp, int32_t b_zp, void* scratch)
{
    PadArgs p{};
    p.a = (const uint8_t*)a, p.b = (const uint8_t*)b, p.ap = (uint8_t*)scratch, p.bp = (uint8_t*)scratch + m.a_bytes;
    p.units_a = (int64_t)(m.a_bytes / 16), p.units_b = (int64_t)(m.b_bytes / 16);
    p.row_a = C * eb, p.row_b = W * eb, p.C = C;
    p.fill_a = (uint32_t)(a_zp & 255) * 0x01010101u, p.fill_b = (uint32_t)(b_zp & 255) * 0x01010101u;
    p.ua = make_fastdiv((uint32_t)(m.CP * eb / 16)), p.ub = make_fastdiv((uint32_t)(m.ldw / 16)), p.cp = make_fastdiv((uint32_t)m.CP);
    const int64_t blocks = (p.units_a + p.units_b + 255) / 256;
    const dim3 grid((unsigned)(blocks > 8192 ? 8192 : blocks));
    if (eb == 1)
        hipLaunchKernelGGL(pad_operands_kernel<1>, grid, dim3(256), 0, st, p, (int32_t)grid.x);
    else
        hipLaunchKernelGGL(pad_operands_kernel<2>, grid, dim3(256), 0, st, p, (int32_t)grid.x);
    return true;
}

template <typename T, int SPLIT, int NC, bool TINY, bool ODD>
static bool launch_split_form(hipStream_t st, RaggedArgs& p)
{
    constexpr int kWaves       = SPLIT > 4 ? SPLIT : 4;
    constexpr size_t lds_bytes = (size_t)kWaves * ragged_wave_lds<T, SPLIT, NC>();
    constexpr auto kern        = matmul_ragged_kernel<T, SPLIT, NC, TINY, ODD>;
    if (lds_bytes > 65536 && !ensure_dynamic_lds<kern>(lds_bytes))
        return false;
    const int64_t grid = ((int64_t)p.tiles * SPLIT + kWaves - 1) / kWaves;
    p.per_xcd          = (uint32_t)(grid / 8);
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(64 * kWaves), lds_bytes, st, p);
    return true;
}

template <typename T, int SPLIT, int NC = 2>
static bool launch_split(hipStream_t st, RaggedArgs& p)
{
    constexpr int EB = (int)sizeof(T);
    // (rows beyond 32-bit offsets, us with every piece element by element / now: int8 [1,66000001]x[66000001,1] 415800 / 72300, fp16
    // [1,33000001]x[33000001,1] 265000 / 48600)
    const bool tiny = p.a_total < 16 || p.b_total < 16 || (int64_t)p.C * EB > INT32_MAX / 33 || (int64_t)p.W * EB > INT32_MAX / 65;
    if (tiny)
        return launch_split_form<T, SPLIT, NC, true, false>(st, p);
    return p.odd & (SPLIT == 1 && EB == 2 ? 3 : 1) ? launch_split_form<T, SPLIT, NC, false, true>(st, p) : launch_split_form<T, SPLIT, NC, false, false>(st, p);
}

template <typename T>
static bool launch_ragged(hipStream_t st, RaggedArgs& p)
{
    const int blocks = (p.C * (int)sizeof(T) + 63) / 64;
    // K over as many waves as give the chip two thousand (two a SIMD), each with a block of its own at least.  us for 1024 / 2048 / 4096
    // waves: fp16 96 x [197,197]x[197,64] (672 tiles) 8.6 / 7.3 / 7.1, 96 x [197,64]x[64,197] (2688) 8.8 / 8.8 / 9.9, 64 x [8,512]x[512,512]
    // (512) 6.8 / 5.5 / 5.5, 7 x [78,853]x[853,2096] 22.5 / 17.2 / 16.8, 4 x [300,301]x[301,303] (200) 4.8 / 4.9 / 4.8; int8 in this order 6.7 / 5.9 /
    // 5.7, 7.2 / 7.3 / 7.2, 4.8 / 4.4 / 4.2; the other way [500,2000]x[2000,500] (128) fp16 7.6 / 8.3 / 8.1, int8 5.9 / 6.2 / 6.2.
    int split = 1;
    while (split < 16 && (int64_t)p.tiles * split < 2048 && split * 2 <= blocks)
        split *= 2;
    switch (split)
    {
        case 1: return launch_split<T, 1>(st, p);
        case 2: return launch_split<T, 2>(st, p);
        case 4: return launch_split<T, 4>(st, p);
        case 8: return launch_split<T, 8>(st, p);
        default: break;
    }
    // Sixteen waves a tile and still few tiles: a workgroup, and the lines its CU's L1 takes in, bound it; tiles of 32 columns then put
    // twice as many CUs to work, while those fit beside each other.  us 64 / 32 columns: fp16 [1,4096]x[4096,4096] (64 tiles of 64) 11.0 / 9.4,
    // [13,3215]x[3215,235] x 5 (20) 18.6 / 14.9, [64,4000]x[4000,64] (2) 11.2 / 8.9, [20,1500]x[1500,3000] x 2 (94) 7.7 / 6.0, int8 5.0 / 4.5;
    // [500,2000]x[2000,500] (128) 8.2 / 8.1, int8 6.2 / 6.4; the other way [100,1100]x[1100,700] x 3 (132) 5.8 / 7.4, 4.9 / 5.8.
    const int64_t wide = p.tiles_w.d, narrow = ((int64_t)p.W + 31) / 32, rows = p.tiles / wide;
    if (p.tiles > 112 || !fastdiv_exact_up_to((uint64_t)(rows * narrow), (uint32_t)(p.per_batch.d / wide * narrow)) ||
        !fastdiv_exact_up_to((uint64_t)(p.per_batch.d / wide * narrow), (uint32_t)narrow))
        return launch_split<T, 16>(st, p);
    p.per_batch = make_fastdiv((uint32_t)(p.per_batch.d / wide * narrow));
    p.tiles     = (int32_t)(rows * narrow);
    p.tiles_w   = make_fastdiv((uint32_t)narrow);
    return launch_split<T, 16, 1>(st, p);
}

const char* launch_matmul_ragged(hipStream_t st, int32_t in_dtype, int32_t N, int32_t H, int32_t C, int32_t W, const void* a, const void* b,
                                 int32_t a_zp, int32_t b_zp, void* out)
{
    const int eb        = in_dtype == TMI_INT8 ? 1 : 2;
    const int64_t tw = ((int64_t)W + 63) / 64, per = ((int64_t)H + 31) / 32 * tw, tiles = per * N;
    if (C < 1 || tiles > INT32_MAX / 16 || (int64_t)C * eb > INT32_MAX / 2 || !fastdiv_exact_up_to((uint64_t)tiles, (uint32_t)per) ||
        !fastdiv_exact_up_to((uint64_t)per, (uint32_t)tw) || (eb == 2 && (((uintptr_t)a | (uintptr_t)b) & 1)))
        return nullptr;
    RaggedArgs p{};
    p.a = (const uint8_t*)a, p.b = (const uint8_t*)b, p.out = (uint8_t*)out;
    p.a_total = (int64_t)N * H * C * eb, p.b_total = (int64_t)N * C * W * eb;
    p.H = H, p.C = C, p.W = W, p.za = a_zp, p.zb = b_zp, p.odd = ((C * eb | (int)((uintptr_t)a & 3)) % 4 ? 1 : 0) | ((W * eb | (int)((uintptr_t)b & 3)) % 4 ? 2 : 0), p.tiles = (int32_t)tiles;
    p.per_batch = make_fastdiv((uint32_t)per), p.tiles_w = make_fastdiv((uint32_t)tw);
    switch (in_dtype)
    {
        case TMI_INT8: return launch_ragged<int8_t>(st, p) ? "matmul_ragged_i8" : nullptr;
        case TMI_FP16: return launch_ragged<_Float16>(st, p) ? "matmul_ragged_f16" : nullptr;
        case TMI_BF16: return launch_ragged<bf16_t>(st, p) ? "matmul_ragged_bf16" : nullptr;
        default: return nullptr;
    }
}

}    // namespace tmi
