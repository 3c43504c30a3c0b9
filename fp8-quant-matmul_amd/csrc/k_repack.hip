// Padding copies for shapes the MFMA kernels cannot take as they are.
//
// The tile kernels move 16-byte pieces of A's and B's columns, which start at k*M and k*N:
// they need M and N to be multiples of 16 (and 16-byte aligned bases; some tiles have a form that
// takes any M).  The reference asks
// for multiples of 64 or 32 and reads out of bounds otherwise (/root/reference/mn_large.hip:16).
// For any other shape the operands are copied into buffers whose leading dimension is rounded
// up to 16 (new rows zero), the GEMM runs on the padded problem into a padded C, and C's
// m x n corner is copied out.  All of it is plain data movement: 2 bytes moved per byte of a
// padded operand, 4 per element of C.
#include "device_common.h"
#include "launchers.h"

namespace fp8gemm {

namespace {

// 16 bytes of a padded row: dst[16 * ch ..] = src[16 * ch ..] of a row of ld_src bytes, zeros beyond it.  Whatever the
// alignment of the row, the bytes lie in one or two aligned 16-byte pieces of memory, which are loaded whole and shifted
// into place.  What such a piece holds beside the row is not used, and it lies on a page of the matrix.
struct PadPiece {
    v4i lo, hi;     // the aligned pieces
    uint32_t sh;    // where the row's bytes start in them
    int valid;      // bytes that belong to the row

    __device__ __forceinline__ void load(const uint8_t* src, uint32_t row, uint32_t ch, uint32_t ld_src)
    {
        valid = (int)ld_src - 16 * (int)ch;
        const uintptr_t ad = reinterpret_cast<uintptr_t>(src) + (size_t)row * ld_src + (size_t)ch * 16;
        sh = (uint32_t)(ad & 15);
        // no branch around a load: each would be waited for before the next is asked for.  A piece that holds none of the
        // row's bytes is replaced by one that does (the other piece, or where the row starts: rows are not empty).
        const uintptr_t p = valid > 0 ? ad - sh : (reinterpret_cast<uintptr_t>(src) + (size_t)row * ld_src) & ~(uintptr_t)15;
        const bool both = (int)sh + (valid < 16 ? valid : 16) > 16;
        lo = *reinterpret_cast<const __attribute__((address_space(1))) v4i*>(p);
        hi = *reinterpret_cast<const __attribute__((address_space(1))) v4i*>(p + (both ? 16 : 0));
    }

    __device__ __forceinline__ v4i bytes() const
    {
        const uint32_t w[8] = {(uint32_t)lo[0], (uint32_t)lo[1], (uint32_t)lo[2], (uint32_t)lo[3],
                               (uint32_t)hi[0], (uint32_t)hi[1], (uint32_t)hi[2], (uint32_t)hi[3]};
        // bit selects: a choice between two elements of an array becomes an indexed access, by way of the LDS
        const uint32_t by2 = 0u - ((sh >> 3) & 1u), by1 = 0u - ((sh >> 2) & 1u);
        uint32_t two[6], one[5];
#pragma unroll
        for (int i = 0; i < 6; ++i)
            two[i] = (w[i + 2] & by2) | (w[i] & ~by2);
#pragma unroll
        for (int i = 0; i < 5; ++i)
            one[i] = (two[i + 1] & by1) | (two[i] & ~by1);
        v4i out;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t v = __builtin_amdgcn_alignbyte(one[i + 1], one[i], sh & 3);
            const int left = valid - 4 * i;  // bytes of this dword that belong to the row
            out[i] = (int)(left >= 4 ? v : (left <= 0 ? 0u : (v & ((1u << (8 * left)) - 1u))));
        }
        return out;
    }
};

// All padding copies of a call in one launch: a workgroup moves PER_THREAD * 256 pieces of 16 bytes of one job.
//
// Bound by memory: 2 bytes move per byte of the operand.  All loads of a thread are out before the first is needed, indices
// are 32 bits wide (an operand has less than 2^27 pieces), and a large grid holds the pieces that there are (a small one:
// JOB_ROWS_MAX_WORKGROUPS below).  Against one piece
// per thread by five dword loads and a 64-bit division on a grid as large for every job as for the largest: 8191 x 7168
// 25.0 -> 22.1 us (5.3 TB/s), eight groups of 250 ... 2051 rows x 2048 12.9 -> 9.6 us, thirty of 200 rows 8.6 -> 7.6 us;
// a single operand of up to 3 MB, where the launch is what it takes, is level (333 x 7168: 5.0 us).
template <int MAX, int PER_THREAD, bool JOB_ROWS>
__global__ void __launch_bounds__(256) pad_kernel(const PadJobs<MAX> jobs)
{
    const uint32_t block = blockIdx.x;
    int job = 0;
    if (JOB_ROWS) {
        job = blockIdx.y;
    } else if (MAX <= 4) {
#pragma unroll
        for (int j = 1; j < MAX; ++j)
            job += j < jobs.count && block >= jobs.first_block[j];
    } else {  // first_block ascends: how many jobs start at or before this workgroup, looked up by a lane each
        const int lane = threadIdx.x & 63;
        int upto = 0;
#pragma unroll
        for (int j = 0; j < MAX; j += 64)
            upto += __builtin_popcountll(
                __builtin_amdgcn_ballot_w64(j + lane < jobs.count && jobs.first_block[j + lane] <= block));
        job = __builtin_amdgcn_readfirstlane(upto) - 1;
    }
    const uint8_t* const src = static_cast<const uint8_t*>(jobs.src[job]);
    uint8_t* const dst = jobs.base + (size_t)jobs.dst256[job] * 256;
    const uint32_t chunks = jobs.chunks[job], ld_src = jobs.ld_src[job], pieces = jobs.rows[job] * chunks;
    const uint32_t first = (block - (JOB_ROWS ? 0u : jobs.first_block[job])) * (256u * PER_THREAD), at = first + threadIdx.x;
    if (JOB_ROWS && first >= pieces)
        return;
    PadPiece piece[PER_THREAD];
#pragma unroll
    for (int u = 0; u < PER_THREAD; ++u) {
        const uint32_t idx = min(at + 256u * u, pieces - 1), row = idx / chunks;
        piece[u].load(src, row, idx - row * chunks, ld_src);
    }
#pragma unroll
    for (int u = 0; u < PER_THREAD; ++u) {
        const uint32_t idx = at + 256u * u;
        if (idx < pieces)
            *(__attribute__((address_space(1))) v4i*)(dst + (size_t)idx * 16) = piece[u].bytes();
    }
}

// Four pieces to a thread from this many on (4 MB: four workgroups of 256 threads for every CU with one each): below, CUs
// would be left without a workgroup.
constexpr size_t PIECES_FOR_FOUR = (size_t)1 << 18;

// The copies of a grouped call: up to this many workgroups the grid has a row as long as the largest job's for every job
// (JOB_ROWS), so that a workgroup knows its job without looking it up, a trip to the kernel arguments in front of the one
// for the job itself; the surplus workgroups, at most 16 for a CU, leave at once.  39 grouped calls with 60 ... 4096 of
// them, with the GEMM behind it: up to 13 % ahead of the looked-up form, 2 % behind at worst (eight groups of 87 - 166
// rows, 2112 x 256, from HBM 11.84 -> 10.49 us; 59 of 2 - 16 rows, 3632 x 128, 15.54 -> 14.65); beyond, where the grid
// would be mostly surplus, the two are level and the looked-up form 1 % ahead.
constexpr uint32_t JOB_ROWS_MAX_WORKGROUPS = 4096;

template <int MAX, int PER_THREAD>
hipError_t launch_pad_typed(PadJobs<MAX>& jobs, hipStream_t s)
{
    uint32_t blocks = 0, most = 0;
    for (int j = 0; j < jobs.count; ++j) {
        const uint32_t mine = (jobs.rows[j] * jobs.chunks[j] + 256 * PER_THREAD - 1) / (256 * PER_THREAD);
        jobs.first_block[j] = blocks;
        blocks += mine;
        most = mine > most ? mine : most;
    }
    if constexpr (MAX > 4)
        if ((uint64_t)most * jobs.count <= JOB_ROWS_MAX_WORKGROUPS) {
            launch_kernel((pad_kernel<MAX, PER_THREAD, true>), dim3(most, jobs.count), dim3(256), 0, s, jobs);
            return hipGetLastError();
        }
    launch_kernel((pad_kernel<MAX, PER_THREAD, false>), dim3(blocks), dim3(256), 0, s, jobs);
    return hipGetLastError();
}

// dst[m][n] (dense) = src[m][0..n) of a matrix with ld_src elements per row (a multiple of 8, base
// 16-byte aligned).  One thread moves 8 elements of a row: one 16-byte load, and one store as
// wide as the destination's alignment allows.
__device__ __forceinline__ void crop_piece(const uint16_t* __restrict__ src, uint16_t* __restrict__ dst, int m, int n,
                                           int ld_src, size_t idx)
{
    const int chunks = (n + 7) / 8;
    if (idx >= (size_t)m * chunks)
        return;
    const int r = (int)(idx / chunks), ch = (int)(idx - (size_t)r * chunks);
    const uint4 v = *reinterpret_cast<const uint4*>(src + (size_t)r * ld_src + (size_t)ch * 8);
    uint16_t* d = dst + (size_t)r * n + (size_t)ch * 8;
    const int count = n - 8 * ch < 8 ? n - 8 * ch : 8;
    const uintptr_t ad = reinterpret_cast<uintptr_t>(d);
    const uint32_t wv[4] = {v.x, v.y, v.z, v.w};
    if (count == 8 && (ad & 15) == 0) {
        *reinterpret_cast<uint4*>(d) = v;
    } else if (count == 8 && (ad & 3) == 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            reinterpret_cast<uint32_t*>(d)[i] = wv[i];
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (i < count)
                d[i] = (uint16_t)(wv[i >> 1] >> (16 * (i & 1)));
    }
}

// a problem per blockIdx.y
__global__ void __launch_bounds__(256) crop_batched_kernel(const CropTable tab)
{
    const int g = blockIdx.y;
    crop_piece(static_cast<const uint16_t*>(tab.src[g]), static_cast<uint16_t*>(tab.dst[g]), tab.m[g], tab.n, tab.ld_src,
               (size_t)blockIdx.x * blockDim.x + threadIdx.x);
}

__global__ void __launch_bounds__(256)
crop_kernel(const uint16_t* __restrict__ src, uint16_t* __restrict__ dst, int m, int n, int ld_src)
{
    crop_piece(src, dst, m, n, ld_src, (size_t)blockIdx.x * blockDim.x + threadIdx.x);
}

inline unsigned crop_blocks(int m, int n) { return (unsigned)(((size_t)m * ((n + 7) / 8) + 255) / 256); }

}  // namespace

template <int MAX>
hipError_t launch_pad(PadJobs<MAX>& jobs, hipStream_t s)
{
    if (jobs.count < 0 || jobs.count > MAX)
        return hipErrorInvalidValue;
    size_t pieces = 0;
    for (int j = 0; j < jobs.count; ++j)
        pieces += (size_t)jobs.rows[j] * jobs.chunks[j];
    if (pieces == 0)
        return hipSuccess;
    return pieces >= PIECES_FOR_FOUR ? launch_pad_typed<MAX, 4>(jobs, s) : launch_pad_typed<MAX, 1>(jobs, s);
}
template hipError_t launch_pad<PAD_JOBS_SINGLE>(PadJobs<PAD_JOBS_SINGLE>&, hipStream_t);
template hipError_t launch_pad<PAD_JOBS_GROUPED>(PadJobs<PAD_JOBS_GROUPED>&, hipStream_t);

hipError_t launch_crop_bf16(const uint16_t* src, uint16_t* dst, int m, int n, int ld_src, hipStream_t s)
{
    if (m == 0 || n == 0)
        return hipSuccess;
    launch_kernel(crop_kernel, dim3(crop_blocks(m, n)), dim3(256), 0, s, src, dst, m, n, ld_src);
    return hipGetLastError();
}

hipError_t launch_crop_bf16_batched(const CropTable& tab, hipStream_t s)
{
    if (tab.groups < 1 || tab.groups > CropTable::MAX_GROUPS)
        return hipErrorInvalidValue;
    unsigned most = 0;
    for (int g = 0; g < tab.groups; ++g) {
        const unsigned blocks = crop_blocks(tab.m[g], tab.n);
        most = blocks > most ? blocks : most;
    }
    if (most == 0)
        return hipSuccess;
    launch_kernel(crop_batched_kernel, dim3(most, (unsigned)tab.groups), dim3(256), 0, s, tab);
    return hipGetLastError();
}

}  // namespace fp8gemm
