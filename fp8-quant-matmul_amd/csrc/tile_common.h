// Pieces shared by the tile kernels (k_tile.hip, k_tile_persistent.hip): LDS stage geometry,
// the chunk swizzle, the explicit wait on the copy counter.
#pragma once
#include "device_common.h"
#include "launchers.h"

#include <type_traits>

namespace fp8gemm {
namespace {

constexpr int NTHREADS = 512;
constexpr int GROUP_M = 8;  // tile rows per L2 locality group

// NW = waves of the workgroup (all of them copy): eight, or four for the kernels that run one wave
// per SIMD with twice the registers.
template <int BM, int BN, int WM, int WN, int NS, int NW = 8>
struct TileShape {
    static constexpr int RSA = BM > 128 ? 256 : (BM > 64 ? 128 : 64);  // LDS bytes per k-row of the A tile
    static constexpr int RSB = BN > 128 ? 256 : (BN > 64 ? 128 : 64);
    static constexpr int MAT_A = KBLOCK * RSA;
    static constexpr int MAT_B = KBLOCK * RSB;
    static constexpr int SCALE_OFF = MAT_A + MAT_B;       // BM a_scale floats
    static constexpr int SB_OFF = SCALE_OFF + 1024;       // four waves per workgroup, or four multiplying ones: 64 dwords,
                                                          // the first few = b_scale of the tile's columns
    static constexpr bool SB_STAGED = NW == 4 || WM * WN == 4;
    static constexpr int STAGE = MAT_A + MAT_B + 1024 + (SB_STAGED ? 256 : 0);
    static constexpr int LDS_BYTES = NS * STAGE;
    static constexpr int NA = RSA / (8 * NW);             // copy instructions per wave, A tile
    static constexpr int NB = RSB / (8 * NW);
    static constexpr int NCOPY = NA + NB + 1;             // + the a_scale slice (one wave); where it is staged,
                                                          // another wave brings b_scale as well
    static_assert(NW == 4 || NW == 8, "four or eight waves");
    static_assert(NA * 8 * NW == RSA && NB * 8 * NW == RSB, "whole copy instructions per wave");
    // A wave's copy instructions of one matrix lie 4 (256-byte rows), 8 (128-byte rows) or 16
    // (64-byte rows) k-rows apart.  Instructions 8 rows apart share the chunk swizzle and hence
    // the per-lane offset: only NV distinct offsets are kept in registers, the row distance goes
    // into the instruction's scalar offset.
    static constexpr int NVA = RSA == 256 ? 2 : 1;
    static constexpr int NVB = RSB == 256 ? 2 : 1;
    // instruction q of a matrix with row stride RS: which kept offset, and how many k-rows on top
    template <int RS> static constexpr int voff_index(int q) { return RS == 256 ? (q & 1) : 0; }
    template <int RS> static constexpr int extra_rows(int q)
    {
        return RS == 256 ? (q >> 1) * 8 : q * (1024 / RS);
    }
    // lane of a copy instruction -> k-row within the instruction's 1 KiB and chunk position in it
    template <int RS> static __device__ __forceinline__ int copy_row(int lane) { return lane / (RS / 16); }
    template <int RS> static __device__ __forceinline__ int copy_pos(int lane) { return lane % (RS / 16); }
    static_assert(LDS_BYTES <= 160 * 1024, "stages exceed the 160 KiB of LDS");
};

// chunk swizzle of k-row r (0 .. 127) for a row stride of RS bytes: the 16 rows whose pieces of one chunk are read
// together (frag_row: eight adjacent rows and the eight 64 further on) lie in 16 different 16-byte bank groups.  The rows
// that a wave copies agree in r >> 6.
template <int RS>
__device__ __forceinline__ int row_swizzle(int r)
{
    return (RS == 256 ? 2 * (r & 7) : (RS == 128 ? 2 * ((r >> 1) & 3) : 2 * ((r >> 2) & 1))) + (r >> 6);
}

// ---- operand fragments of v_mfma_f32_16x16x128_f8f6f4 out of a stage: 16 rows of m or n (one 16-byte chunk) x 128 k in
// four transposing reads.  In read t lane 16 * g + i supplies the half (i & 1) of the chunk in k-row frag_row + 8 * t and
// receives 8 k of row i; the k order inside the instruction is permuted alike for both operands.
__device__ __forceinline__ int frag_row(int lane)
{
    const int g = lane >> 4, i = lane & 15;
    return 64 * (g & 1) + 32 * (g >> 1) + (i >> 1);
}
// LDS offset of a lane's first read of chunk `chunk` of a matrix with rows of RS bytes
template <int RS>
__device__ __forceinline__ uint32_t frag_addr(int lane, int chunk)
{
    const int r = frag_row(lane);
    return (uint32_t)(r * RS + (lane & 1) * 8 + ((chunk ^ row_swizzle<RS>(r)) * 16));
}
template <int RS, typename Lds>
__device__ __forceinline__ v8i read_frag(Lds first)  // the lane's first read
{
    const v2i r0 = __builtin_amdgcn_ds_read_tr8_b64_v2i32(LDS_PTR(v2i, first));
    const v2i r1 = __builtin_amdgcn_ds_read_tr8_b64_v2i32(LDS_PTR(v2i, first + 8 * RS));
    const v2i r2 = __builtin_amdgcn_ds_read_tr8_b64_v2i32(LDS_PTR(v2i, first + 16 * RS));
    const v2i r3 = __builtin_amdgcn_ds_read_tr8_b64_v2i32(LDS_PTR(v2i, first + 24 * RS));
    return (v8i){r0.x, r0.y, r1.x, r1.y, r2.x, r2.y, r3.x, r3.y};
}
// the block sum of a 16 x 16 patch: rows = n (4 * (lane >> 4) + register), columns = m (lane & 15)
__device__ __forceinline__ v4f block_sum(v8i b, v8i a)
{
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(b, a, (v4f){0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0);
}

// One problem of a launch as the persistent kernels see it.
struct TileProblem {
    const uint8_t* a;
    const uint8_t* b;
    const float* a_scale;
    const float* b_scale;
    uint16_t* c;
    int M;
    int lda;  // elements between consecutive k-rows of a and of a_scale (>= M, a multiple of 16)
};

// Which part of a launch a walk covers.  All tiles of BM x BN; or, of a grid of such tiles, the rounds in which every
// workgroup of an XCD gets one; or the ones left over, each cut into sub-tiles of SM x SN.
template <int BM_, int BN_>
struct AllTiles {
    static constexpr int BM = BM_, BN = BN_, SM = BM_, SN = BN_;
    static constexpr bool FULL_ROUNDS = false, LEFT_OVER = false;
};
template <int BM_, int BN_>
struct FullRounds {
    static constexpr int BM = BM_, BN = BN_, SM = BM_, SN = BN_;
    static constexpr bool FULL_ROUNDS = true, LEFT_OVER = false;
};
template <int BM_, int BN_, int SM_, int SN_>
struct LeftOver {
    static constexpr int BM = BM_, BN = BN_, SM = SM_, SN = SN_;
    static constexpr bool FULL_ROUNDS = false, LEFT_OVER = true;
};

// The tiles of one persistent workgroup.  Workgroup ids go round the 8 XCDs (id % 8); each XCD owns a contiguous run
// of the tile order (groups of GROUP_M tile rows, as in k_tile.hip) and its workgroups take the run's tiles in turn, so that
// the tiles an XCD works on at any moment are neighbours and share A and B panels in its L2.
// GROUPED = false: one problem, tiles_m x tiles_n tiles.  GROUPED = true: the problems of `tab` (same N and K, own M),
// whose tiles are numbered one group after the other.
template <typename SHARE, bool GROUPED>
struct TileWalk {
    static constexpr int BM = SHARE::BM, BN = SHARE::BN, SUBS_N = BN / SHARE::SN, SUBS = BM / SHARE::SM * SUBS_N;
    const TileProblem& one;
    const GroupTable* tab;
    int tiles_m, tiles_n;
    int per_xcd, run0, run_len, li;
    __device__ __forceinline__ TileWalk(const TileProblem& p, const GroupTable* t, int tm, int tn)
        : one(p), tab(t), tiles_m(tm), tiles_n(tn)
    {
        const int T = GROUPED ? tab->tile_start[tab->groups] : tiles_m * tiles_n;
        const int pid = blockIdx.x;
        per_xcd = gridDim.x >> 3;  // gridDim.x is a multiple of 8
        const int xcd = pid & 7, q8 = T >> 3, r8 = T & 7;
        run0 = xcd * q8 + (xcd < r8 ? xcd : r8);
        run_len = q8 + (xcd < r8 ? 1 : 0);
        li = pid >> 3;
        if (SHARE::FULL_ROUNDS || SHARE::LEFT_OVER) {
            const int in_rounds = run_len / per_xcd * per_xcd;
            if (SHARE::FULL_ROUNDS) {
                run_len = in_rounds;
            } else {
                run0 += in_rounds;
                run_len = (run_len - in_rounds) * SUBS;
            }
        }
    }
    __device__ __forceinline__ int count() const { return li < run_len ? (run_len - li + per_xcd - 1) / per_xcd : 0; }
    // tile number j of this workgroup: its problem and its origin in that problem's C
    __device__ __forceinline__ void origin(int j, TileProblem& pr, int& m0, int& n0) const
    {
        const int per_group = GROUP_M * tiles_n;
        const int number = li + j * per_xcd;
        int logical = run0 + number / SUBS;
        int tm = tiles_m;
        if (GROUPED) {
            int g = 0;
            while (g + 1 < tab->groups && logical >= tab->tile_start[g + 1])
                ++g;
            logical -= tab->tile_start[g];
            pr = TileProblem{tab->a[g], tab->b[g], tab->a_scale[g], tab->b_scale[g], tab->c[g], tab->m[g], tab->lda[g]};
            tm = (pr.M + BM - 1) / BM;
        } else {
            pr = one;
        }
        const int group = logical / per_group;
        const int first_m = group * GROUP_M;
        const int gsz = (tm - first_m < GROUP_M) ? (tm - first_m) : GROUP_M;
        const int in_group = logical - group * per_group;
        const int sub = number % SUBS;
        m0 = (first_m + in_group % gsz) * BM + sub / SUBS_N * SHARE::SM;
        n0 = (in_group / gsz) * BN + sub % SUBS_N * SHARE::SN;
    }
};

template <int N>
__device__ __forceinline__ void wait_vmcnt()
{
    static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit field");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

}  // namespace
}  // namespace fp8gemm
