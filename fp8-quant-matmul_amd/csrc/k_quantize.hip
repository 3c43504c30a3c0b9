// Device-side quantisers: the producers of the GEMM's inputs.
//
//   1 x 128 groups along K per row   (to_float8_rowwise_scale, /root/reference/quantize.py:43-67)
//   128 x 128 blocks                 (to_float8_block_scale,   /root/reference/quantize.py:16-41)
//
// Arithmetic of both, with the OCP e4m3fn maximum 448:
//   scale = (1 / max(amax, 1e-12)) * 448;  q = fp8_rne(clamp(x * scale, -448, 448));  stored = 1 / scale
// (reciprocal first, then the product: that is how torch evaluates `finfo.max / amax`,
// quantize.py:28,54).  For an fp32 source every step is fp32.  For a bf16 source torch rounds
// every element-wise result to bf16 (1e-12, the reciprocal, the product with 448, x * scale);
// BF16MATH reproduces that, so that bytes and scales equal the reference's own outputs for
// either source type.  A bf16 source can also be quantised with fp32 arithmetic (more
// accurate, not what quantize.py computes).
//
// The source x is row-major [rows][K] (K contiguous), bf16 or fp32.  The outputs are written
// directly in the GEMM's layouts, which the reference produces with host-side transposes
// (/root/reference/check.cu:164-167):  q at row + k*rows, the 1 x 128 scales at row + kb*rows,
// the 128 x 128 scales at nb + kb*ceil(rows/128).
//
// One workgroup owns QTILE rows x 128 k (a 128 x 128 scale block, or QTILE scale groups).  A thread reads 8 k of
// four adjacent rows at a time (16 lanes take a row's 128 elements: whole cache lines) and converts pairs of ROWS, so
// that the four bytes of one k leave the conversion as the dword the transposed layout wants: the transposition costs
// eight dword writes into the LDS per 32 elements and no byte shuffling.  From there the tile leaves as 16-byte
// pieces of QTILE-byte row segments.  The kernel moves 2 (or 4) bytes in and 1 byte out per element: bound by HBM.
#include "device_common.h"
#include "launchers.h"

#include <type_traits>

namespace fp8gemm {

namespace {

// eight consecutive k of one row as they lie in memory: four words of bf16 pairs, or eight of fp32
// ONCE = the caches are told not to keep them
template <bool ONCE>
__device__ __forceinline__ v4i load_piece(const void* p)
{
    return ONCE ? __builtin_nontemporal_load(static_cast<const v4i*>(p)) : *static_cast<const v4i*>(p);
}
template <bool ONCE>
__device__ __forceinline__ void load_raw(const uint16_t* p, uint32_t (&w)[4])
{
    const v4i v = load_piece<ONCE>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i)
        w[i] = (uint32_t)v[i];
}
template <bool ONCE>
__device__ __forceinline__ void load_raw(const float* p, uint32_t (&w)[8])
{
    const v4i lo = load_piece<ONCE>(p), hi = load_piece<ONCE>(p + 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        w[i] = (uint32_t)lo[i];
        w[4 + i] = (uint32_t)hi[i];
    }
}
template <int J>
__device__ __forceinline__ float value(const uint32_t (&w)[4])
{
    return __uint_as_float((J & 1) ? w[J >> 1] & 0xFFFF0000u : w[J >> 1] << 16);
}
template <int J>
__device__ __forceinline__ float value(const uint32_t (&w)[8])
{
    return __uint_as_float(w[J]);
}

template <int J>
__device__ __forceinline__ float pair_value(const uint32_t (&w)[1])
{
    return __uint_as_float(J ? w[0] & 0xFFFF0000u : w[0] << 16);
}
template <int J>
__device__ __forceinline__ float pair_value(const uint32_t (&w)[2])
{
    return __uint_as_float(w[J]);
}

template <bool BF16MATH>
__device__ __forceinline__ float q_round(float v)
{
    return BF16MATH ? __uint_as_float(pack_bf16x2(v, 0.0f) << 16) : v;
}

// two scaled values (of two rows), rounded to bf16 first where the source's arithmetic does that, saturated (NaN
// becomes -448, as min(max(v, -448), 448) has it), as two fp8 bytes in the half of `old` that HIGH names
template <bool BF16MATH, bool HIGH>
__device__ __forceinline__ int q_pair(float x, float y, int old)
{
    if (BF16MATH) {
        const uint32_t u = pack_bf16x2(x, y);
        x = __uint_as_float(u << 16);
        y = __uint_as_float(u & 0xFFFF0000u);
    }
    return __builtin_amdgcn_cvt_pk_fp8_f32(__builtin_amdgcn_fmed3f(x, -448.0f, 448.0f),
                                           __builtin_amdgcn_fmed3f(y, -448.0f, 448.0f), old, HIGH);
}

// v of another lane of the same 16-lane row (rotation by N), or of lane J of the same group of four
template <int N>
__device__ __forceinline__ float row_rotate(float v)
{
    return __uint_as_float((uint32_t)__builtin_amdgcn_mov_dpp((int)__float_as_uint(v), 0x120 + N, 0xF, 0xF, true));
}
template <int J>
__device__ __forceinline__ float quad_lane(float v)
{
    return __uint_as_float((uint32_t)__builtin_amdgcn_mov_dpp((int)__float_as_uint(v), J * 0x55, 0xF, 0xF, true));
}

// v of lane l ^ X of the same group of four
template <int X>
__device__ __forceinline__ float quad_swap(float v)
{
    return __uint_as_float((uint32_t)__builtin_amdgcn_mov_dpp((int)__float_as_uint(v), X == 1 ? 0xB1 : 0x4E, 0xF, 0xF, true));
}

__device__ __forceinline__ float row_max(float a)
{
    a = fmaxf(a, row_rotate<1>(a));
    a = fmaxf(a, row_rotate<2>(a));
    a = fmaxf(a, row_rotate<4>(a));
    return fmaxf(a, row_rotate<8>(a));
}
template <int J>
using Index = std::integral_constant<int, J>;

template <bool BF16MATH>
__device__ __forceinline__ float scale_of(float amax)
{
    const float recip = q_round<BF16MATH>(1.0f / fmaxf(amax, q_round<BF16MATH>(1e-12f)));
    return q_round<BF16MATH>(recip * 448.0f);
}

// BLOCK = false: one scale per row and 128 k (1 x 128).  BLOCK = true: one per 128 x 128.
// QTILE = rows of a workgroup's tile, 16 per wave (4 rows x 8 k per thread).
// ONCE = x is read past the caches.
template <typename TIn, bool BLOCK, bool BF16MATH, int QTILE, bool ONCE>
__global__ void __launch_bounds__(QTILE * 4)
quantize_kernel(const TIn* __restrict__ x, uint8_t* __restrict__ q, float* __restrict__ scale_out,
                int rows, int K, int grid)
{
    constexpr int NT = QTILE * 4, NW = NT / 64;
    static_assert(!BLOCK || QTILE == 128, "one scale block");
    // LDS: one row of QTILE bytes per k, its 16-byte chunks (four dwords: the rows of one wave) permuted by
    // k so that the dword writes of a wave -- 16 k that are 8 apart, one chunk -- go to as many banks as there are
    constexpr int CH = QTILE / 16;                        // chunks per k-row
    constexpr int STRIDE = QTILE == 64 ? 80 : QTILE;
    constexpr int KSH = QTILE == 64 ? 4 : 3;
    __shared__ __attribute__((aligned(16))) uint8_t tile[128 * STRIDE];
    __shared__ float s_red[NW];

    const int t = threadIdx.x;
    const int lane = t & 63, wave = t >> 6;
    const int c = lane & 15;   // 8-element piece of the row's 128
    const int g = lane >> 4;   // four rows
    const int row0 = blockIdx.x * QTILE;
    const int kb = blockIdx.y;

    // rows past the last are read as the last one: no branch around a load, all of them are in flight together (they
    // do not change the block's amax, and their bytes are not stored)
    uint32_t raw[4][2 * sizeof(TIn)];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = row0 + 16 * wave + 4 * g + i;
        load_raw<ONCE>(x + (size_t)(row < rows ? row : rows - 1) * K + (size_t)kb * 128 + 8 * c, raw[i]);
    }

    float amax[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        auto mag = [&](auto j) __attribute__((always_inline)) { return __builtin_fabsf(value<decltype(j)::value>(raw[i])); };
        const float lo = fmaxf(fmaxf(mag(Index<0>{}), mag(Index<1>{})), fmaxf(mag(Index<2>{}), mag(Index<3>{})));
        const float hi = fmaxf(fmaxf(mag(Index<4>{}), mag(Index<5>{})), fmaxf(mag(Index<6>{}), mag(Index<7>{})));
        amax[i] = fmaxf(fmaxf(lo, hi), 0.0f);  // a group of NaNs has amax 0
    }

    float scale[4];
    if (BLOCK) {
        float a = fmaxf(fmaxf(amax[0], amax[1]), fmaxf(amax[2], amax[3]));
        a = row_max(a);
        a = fmaxf(a, __shfl_xor(a, 16));
        a = fmaxf(a, __shfl_xor(a, 32));
        if (lane == 0)
            s_red[wave] = a;
        __syncthreads();
        a = s_red[0];
#pragma unroll
        for (int w = 1; w < NW; ++w)
            a = fmaxf(a, s_red[w]);
        const float mine = scale_of<BF16MATH>(a);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            scale[i] = mine;
        if (t == 0)
            scale_out[(size_t)kb * gridDim.x + blockIdx.x] = 1.0f / mine;
    } else {
        // lane c works out the scale of row c & 3 of its four, the others take it over from there
        const float a0 = row_max(amax[0]), a1 = row_max(amax[1]), a2 = row_max(amax[2]), a3 = row_max(amax[3]);
        const float lo = (c & 1) ? +a1 : +a0, hi = (c & 1) ? +a3 : +a2;
        const float mine = scale_of<BF16MATH>((c & 2) ? +hi : +lo);
        scale[0] = quad_lane<0>(mine);
        scale[1] = quad_lane<1>(mine);
        scale[2] = quad_lane<2>(mine);
        scale[3] = quad_lane<3>(mine);
        const int row = row0 + 16 * wave + 4 * g + c;
        if (c < 4 && row < rows)
            scale_out[(size_t)kb * rows + row] = 1.0f / mine;
    }

    auto put = [&](auto jc) __attribute__((always_inline)) {
        constexpr int j = decltype(jc)::value;
        int w = q_pair<BF16MATH, false>(value<j>(raw[0]) * scale[0], value<j>(raw[1]) * scale[1], 0);
        w = q_pair<BF16MATH, true>(value<j>(raw[2]) * scale[2], value<j>(raw[3]) * scale[3], w);
        const int k = 8 * c + j;
        *reinterpret_cast<int*>(tile + k * STRIDE + ((wave ^ ((k >> KSH) & (CH - 1))) << 4) + 4 * g) = w;
    };
    put(Index<0>{});
    put(Index<1>{});
    put(Index<2>{});
    put(Index<3>{});
    put(Index<4>{});
    put(Index<5>{});
    put(Index<6>{});
    put(Index<7>{});
    __syncthreads();

    // k-row kk of the tile: QTILE bytes, one per source row; a lane takes 16 of them
    const int dq = t % CH, first = row0 + 16 * dq;
    auto piece = [&](int kk) __attribute__((always_inline)) { return tile + kk * STRIDE + ((dq ^ ((kk >> KSH) & (CH - 1))) << 4); };
    if (grid == 16) {  // every k-row starts on a 16-byte boundary
#pragma unroll
        for (int pass = 0; pass < 128 * CH / NT; ++pass) {
            const int kk = t / CH + (NT / CH) * pass;
            const uint4 v = *reinterpret_cast<const uint4*>(piece(kk));
            if (first < rows)
                *reinterpret_cast<uint4*>(q + (size_t)(kb * 128 + kk) * rows + first) = v;
        }
        return;
    }
    // The small tiles: the same, since a store takes any address, and of a row's last bytes what there is.  Where the memory
    // system is not what bounds the launch that is the shortest way (128 rows of a tile, shifted into aligned pieces as
    // below / this, bf16 from the Infinity Cache: 100 x 7168 4.18 / 2.95 us, 333 x 2048 4.29 / 3.07, 1023 x 7168 8.48 / 7.14,
    // blocks of 4607 x 7168 27.1 / 24.7; 256 rows: 4095 x 7168 22.3 / 23.6, fp32 34.6 / 38.5).
    if (QTILE != 256) {
#pragma unroll
        for (int pass = 0; pass < 128 * CH / NT; ++pass) {
            const int kk = t / CH + (NT / CH) * pass;
            const uint8_t* const from = piece(kk);
            uint8_t* const to = q + (size_t)(kb * 128 + kk) * rows + first;
            if (first + 16 <= rows) {
                const uint4 v = *reinterpret_cast<const uint4*>(from);
                __builtin_memcpy(to, &v, 16);
            } else if (first < rows) {
                const int left = rows - first;
                int at = 0;
                if (left & 8) {
                    __builtin_memcpy(to, __builtin_assume_aligned(from, 8), 8);
                    at = 8;
                }
                if (left & 4) {
                    __builtin_memcpy(to + at, __builtin_assume_aligned(from + at, 4), 4);
                    at += 4;
                }
                if (left & 2) {
                    __builtin_memcpy(to + at, __builtin_assume_aligned(from + at, 2), 2);
                    at += 2;
                }
                if (left & 1)
                    to[at] = from[at];
            }
        }
        return;
    }
    if (grid == 8) {  // in pieces of 8 bytes
#pragma unroll 4
        for (int idx = t; idx < 128 * 2 * CH; idx += NT) {
            const int kk = idx / (2 * CH), h = idx % (2 * CH), first = row0 + 8 * h;
            const uint2 v = *reinterpret_cast<const uint2*>(tile + kk * STRIDE +
                                                            (((h >> 1) ^ ((kk >> KSH) & (CH - 1))) << 4) + 8 * (h & 1));
            if (first < rows)
                *reinterpret_cast<uint2*>(q + (size_t)(kb * 128 + kk) * rows + first) = v;
        }
        return;
    }
    // A row count off the 16-byte grid (a ragged token count): the segment starts at any byte.  The 16-byte pieces of
    // MEMORY that lie inside it are shifted into place and leave as whole stores; the fewer than 16 bytes before the
    // first and behind the last of them leave byte by byte, a lane each.
    const int len = rows - row0 < QTILE ? rows - row0 : QTILE;
    auto at = [&](int kk, int byte) __attribute__((always_inline)) {
        return tile + kk * STRIDE + (((byte >> 4) ^ ((kk >> KSH) & (CH - 1))) << 4) + (byte & 15);
    };
#pragma unroll 2
    for (int idx = t; idx < 128 * CH; idx += NT) {
        const int kk = idx / CH, slot = idx % CH;
        uint8_t* seg = q + (size_t)(kb * 128 + kk) * rows + row0;
        const int o = 16 * slot + ((0 - (int)reinterpret_cast<uintptr_t>(seg)) & 15);  // the piece's first byte, in the segment
        if (o + 16 <= len) {
            uint32_t in[5], w[4];
#pragma unroll
            for (int i = 0; i < 5; ++i)
                in[i] = *reinterpret_cast<const uint32_t*>(at(kk, ((o & ~3) + 4 * i) & (QTILE - 1)));
#pragma unroll
            for (int i = 0; i < 4; ++i)
                w[i] = __builtin_amdgcn_alignbyte(in[i + 1], in[i], (uint32_t)o & 3);
            *reinterpret_cast<uint4*>(seg + o) = make_uint4(w[0], w[1], w[2], w[3]);
        }
    }
#pragma unroll 4
    for (int idx = t; idx < 128 * 32; idx += NT) {
        const int kk = idx >> 5, e = idx & 31;
        uint8_t* seg = q + (size_t)(kb * 128 + kk) * rows + row0;
        int head = (0 - (int)reinterpret_cast<uintptr_t>(seg)) & 15;
        head = head < len ? head : len;
        const int tail = (len - head) & 15;
        if (e < head + tail) {
            const int byte = e < head ? e : len - tail + e - head;
            seg[byte] = *at(kk, byte);
        }
    }
}

// 1 x 128 groups of a decode batch, up to 4 * NW <= 64 rows: a workgroup owns a K block of all of them, whose output, [128][rows]
// bytes, is one contiguous piece of memory (q on a 16-byte boundary).  Bound by a chain, launch, load, arithmetic, store, of which
// only the arithmetic can be shortened: a wave takes four rows, a lane two k of each (the tile kernel's lanes: eight), and the
// condition for the rows that do not exist is the wave's, so that no lane is masked.  The four bytes of one k leave the
// conversion as a dword again; the 16-byte pieces of the output are permuted in the LDS, low four bits of a piece's number
// by the next four, which spreads the lanes' writes, rows bytes apart, over 16 banks.
template <typename TIn, bool BF16MATH, int NW>
__global__ void __launch_bounds__(64 * NW)
quantize_batch_kernel(const TIn* __restrict__ x, uint8_t* __restrict__ q, float* __restrict__ scale_out, int rows, int K)
{
    __shared__ __attribute__((aligned(16))) uint8_t tile[128 * 4 * NW];
    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int kb = blockIdx.x;
    const int row0 = 4 * wave;
    if (row0 < rows) {
        constexpr int WORDS = sizeof(TIn) / 2;  // of two values
        uint32_t raw[4][WORDS];
#pragma unroll
        for (int i = 0; i < 4; ++i) {  // rows past the last are read as the last one, and their bytes are not stored
            const int row = row0 + i < rows ? row0 + i : rows - 1;
            __builtin_memcpy(raw[i], x + (size_t)row * K + (size_t)kb * 128 + 2 * lane, sizeof(raw[i]));
        }
        float v[4][2], amax[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i][0] = pair_value<0>(raw[i]);
            v[i][1] = pair_value<1>(raw[i]);
            amax[i] = fmaxf(fmaxf(__builtin_fabsf(v[i][0]), __builtin_fabsf(v[i][1])), 0.0f);  // a group of NaNs has amax 0
        }
        // lane l ends with the maximum of row l & 3: two exchanges that halve the rows, then over the 16 lanes that have it
        const bool odd = lane & 1, high = lane & 2;
        const float lo = fmaxf(odd ? amax[1] : amax[0], quad_swap<1>(odd ? amax[0] : amax[1]));
        const float hi = fmaxf(odd ? amax[3] : amax[2], quad_swap<1>(odd ? amax[2] : amax[3]));
        float a = fmaxf(high ? hi : lo, quad_swap<2>(high ? lo : hi));
        a = fmaxf(a, row_rotate<4>(a));
        a = fmaxf(a, row_rotate<8>(a));
        const auto p16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(a), false, false);
        a = fmaxf(__uint_as_float(p16[0]), __uint_as_float(p16[1]));
        const auto p32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(a), false, false);
        a = fmaxf(__uint_as_float(p32[0]), __uint_as_float(p32[1]));
        const float mine = scale_of<BF16MATH>(a);
        const float scale[4] = {quad_lane<0>(mine), quad_lane<1>(mine), quad_lane<2>(mine), quad_lane<3>(mine)};
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            int w = q_pair<BF16MATH, false>(v[0][j] * scale[0], v[1][j] * scale[1], 0);
            w = q_pair<BF16MATH, true>(v[2][j] * scale[2], v[3][j] * scale[3], w);
            const int at = (2 * lane + j) * rows + row0;  // in the packed block
            auto place = [](int byte) { return byte ^ ((byte >> 4) & 0xF0); };
            if ((rows & 3) == 0) {
                *reinterpret_cast<int*>(tile + place(at)) = w;
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (row0 + i < rows)
                        tile[place(at + i)] = (uint8_t)((uint32_t)w >> (8 * i));
            }
        }
        if (lane < 4 && row0 + lane < rows)
            scale_out[(size_t)kb * rows + row0 + lane] = 1.0f / mine;
    }
    __syncthreads();
    for (int idx = t; idx < 8 * rows; idx += 64 * NW)
        reinterpret_cast<uint4*>(q + (size_t)kb * 128 * rows)[idx] = reinterpret_cast<const uint4*>(tile)[idx ^ ((idx >> 4) & 15)];
}

// the boundary that every k-row of the output starts on, if that is one of 16 or 8 bytes, else 0
int output_grid(const uint8_t* q, int rows)
{
    const uintptr_t ends = reinterpret_cast<uintptr_t>(q) | (uintptr_t)rows;
    return ends % 16 == 0 ? 16 : ends % 8 == 0 ? 8 : 0;
}

template <typename TIn, bool BLOCK, bool BF16MATH, int QTILE, bool ONCE = false>
void launch_quantize_tile(const TIn* x, uint8_t* q, float* scale_out, int rows, int k, hipStream_t s)
{
    const int grid = output_grid(q, rows);
    launch_kernel((quantize_kernel<TIn, BLOCK, BF16MATH, QTILE, ONCE>), dim3((rows + QTILE - 1) / QTILE, k / 128),
                       dim3(QTILE * 4), 0, s, x, q, scale_out, rows, k, grid);
}

template <typename TIn, bool BF16MATH, int NW>
void launch_quantize_batch(const TIn* x, uint8_t* q, float* scale_out, int rows, int k, hipStream_t s)
{
    launch_kernel((quantize_batch_kernel<TIn, BF16MATH, NW>), dim3(k / 128), dim3(64 * NW), 0, s, x, q, scale_out, rows, k);
}

// Tile sizes, measured with every operand from HBM (us, previous kernel -> this one):
//   128 x 128 blocks: 128 rows, eight waves of 16, whatever the size (512 x 2048 6.5 -> 3.5, 4608 x 7168 28.8 -> 22.0 =
//   4.5 TB/s; 256-row tiles 4.5 and 23.3).
//   1 x 128 groups, up to 64 rows: quantize_batch_kernel (previous forms -> it, from the Infinity Cache, in a graph whose empty kernel
//   takes 1.83: 1 x 7168 3.15 -> 2.12, 16 x 7168 2.48 -> 2.13, 24 x 7168 2.77 -> 2.21, 31 x 7168 3.19 -> 2.34, 50 x 7168 3.27 -> 2.68,
//   64 x 7168 2.83 -> 2.55; fp32 the same to 0.05).  Its way of taking 65 rows and more, two passes over 128: 100 x 7168 3.37 against 2.92
//   in tiles of 64.
//   More rows: 256-row tiles once they make 256 workgroups, whose k-rows leave in pieces of 256 bytes (8192 x 7168
//   46.3 -> 37.1 = 4.7 TB/s, 8191 x 7168 75 -> 48.6 against 54.1 with 128 rows).  Fewer than that: 64 rows
//   up to 1024 tiles (1024 x 2048 5.7 -> 3.8, with 128 rows 4.2), off the grid up to 384 (128 / 64 rows: 130 x 512 3.59 / 2.94, 333 x
//   2048 3.78 / 3.21, 777 x 2048 4.03 / 3.68, 333 x 7168, 336 tiles, 4.62 / 4.60, 500 x 7168, 448, 4.79 / 4.98, fp32 1023 x 7168 10.9 /
//   14.3), else 128.  Multiples of 8 rows count as on the grid (8184 x 1536 x 2048 with its GEMM 46.4 -> 45.3).
//   Values and codes of 115 MB or more together, nearly half of the Infinity Cache, do not stay there beside whatever else
//   runs: the values are read past it (kept / not kept, us, three sets in turn, 1 x 128 with the GEMM behind it: bf16 129 MB
//   6000 x 1536 x 7168 114.5 / 100.8, 176 MB 8192 x 512 x 7168 71.7 / 65.5; blocks of bf16 99 MB 4608 x 7168 17.88 / 18.17,
//   176 MB 8192 x 7168 36.6 / 31.0; fp32 84 MB 8192 x 576 x 2048 36.3 / 40.3, 147 MB 4096 x 1536 x 7168 79.9 / 80.2, 168 MB
//   8192 x 576 x 4096 75.4 / 74.0, 215 MB 6000 x 1536 x 7168 131.8 / 119.2; blocks of fp32 106 MB 4608 x 4608 20.6 / 22.7, 126
//   MB 8192 x 3072 27.5 / 26.5, 165 MB 4608 x 7168 34.3 / 32.5.  bf16 with its GEMM gains from 97 MB on: 4500 x 4608 x 7168
//   182.7 / 178.8).  The price: the same 8192 x 7168 quantised over and over, nothing between, 27.2 / 30.6.
template <typename TIn, bool BF16MATH>
void launch_quantize_typed(const TIn* x, uint8_t* q, float* scale_out, int rows, int k, bool block128, hipStream_t s)
{
    const bool on_grid = rows % 16 == 0 || output_grid(q, rows) == 8;
    const long nkb = k / 128;
    auto tiles = [&](int qtile) { return (rows + qtile - 1) / qtile * nkb; };
    const bool once = (double)rows * k * (sizeof(TIn) + 1) >= 115e6;
    if (block128 && once)
        launch_quantize_tile<TIn, true, BF16MATH, 128, true>(x, q, scale_out, rows, k, s);
    else if (block128)
        launch_quantize_tile<TIn, true, BF16MATH, 128>(x, q, scale_out, rows, k, s);
    else if (rows <= 64 && reinterpret_cast<uintptr_t>(q) % 16 == 0)
        rows <= 16   ? launch_quantize_batch<TIn, BF16MATH, 4>(x, q, scale_out, rows, k, s)
        : rows <= 32 ? launch_quantize_batch<TIn, BF16MATH, 8>(x, q, scale_out, rows, k, s)
                     : launch_quantize_batch<TIn, BF16MATH, 16>(x, q, scale_out, rows, k, s);
    else if (rows <= 64 || tiles(64) <= (on_grid ? 1024 : 384))
        launch_quantize_tile<TIn, false, BF16MATH, 64>(x, q, scale_out, rows, k, s);
    else if (tiles(256) < 256)
        launch_quantize_tile<TIn, false, BF16MATH, 128>(x, q, scale_out, rows, k, s);
    else if (once)
        launch_quantize_tile<TIn, false, BF16MATH, 256, true>(x, q, scale_out, rows, k, s);
    else
        launch_quantize_tile<TIn, false, BF16MATH, 256>(x, q, scale_out, rows, k, s);
}

}  // namespace

hipError_t launch_quantize(const void* x, QuantSource source, uint8_t* q, float* scale_out, int rows,
                           int k, bool block128, hipStream_t s)
{
    switch (source) {
    case QUANT_SOURCE_BF16:
        launch_quantize_typed<uint16_t, true>(static_cast<const uint16_t*>(x), q, scale_out, rows, k, block128, s);
        break;
    case QUANT_SOURCE_F32:
        launch_quantize_typed<float, false>(static_cast<const float*>(x), q, scale_out, rows, k, block128, s);
        break;
    case QUANT_SOURCE_BF16_F32MATH:
        launch_quantize_typed<uint16_t, false>(static_cast<const uint16_t*>(x), q, scale_out, rows, k, block128, s);
        break;
    default:
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace fp8gemm
