// Persistent form of the MFMA tile kernel for shapes with more tiles than compute units (256 x 192 and 256 x 256 tiles have a
// body of their own: k_tile_large.hip).
//
// The plain kernel (k_tile.hip) runs one tile per workgroup: with one workgroup per CU (the LDS
// ring fills the CU) every round of 256 tiles pays the launch of a new workgroup, an empty
// ring (one global round trip before the first MFMA) and an output burst during which no MFMA
// runs.  Here a workgroup walks through its tiles itself and the ring never drains: the K
// blocks of all its tiles form one stream, the copies for block g+NS-1 of the stream are
// issued while block g is multiplied, also across a tile boundary, so the first blocks of
// the next tile land while the finished tile is converted and stored.
//
// The finished tile cannot use the whole ring as its staging area (NS-1 slots hold the next
// tile's blocks): it leaves in pieces of PR rows through the one slot whose block was
// multiplied last.
//
// Data path, LDS layout, MFMA orientation and scale folding are those of k_tile.hip
// (successor of in_smem_kernel, /root/reference/mn_large.hip:11-128; the reference lists a
// persistent kernel that overlaps the epilogue with the next tile as future work,
// /root/reference/README.md:29).
#include "tile_persistent_body.h"

namespace fp8gemm {

namespace {

template <int BM, int BN, int WM, int WN, int NS, int PR>
__global__ void __launch_bounds__(64 * WM * WN)
tile_gemm_persistent_kernel(const uint8_t* __restrict__ a, const uint8_t* __restrict__ b,
                            const float* __restrict__ a_scale, const float* __restrict__ b_scale,
                            uint16_t* __restrict__ c, int M, int lda, int N, int K, int tiles_m, int tiles_n)
{
    const TileProblem one{a, b, a_scale, b_scale, c, M, lda};
    persistent_body<BM, BN, WM, WN, NS, PR, false>(one, nullptr, N, K, tiles_m, tiles_n, (int)threadIdx.x);
}

template <int BM, int BN, int WM, int WN, int NS, int PR>
__global__ void __launch_bounds__(64 * WM * WN)
tile_gemm_grouped_kernel(const GroupTable tab, int N, int K, int tiles_n)
{
    const TileProblem none{nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0};
    persistent_body<BM, BN, WM, WN, NS, PR, true>(none, &tab, N, K, 0, tiles_n, (int)threadIdx.x);
}

template <int BM, int BN, int WM, int WN, int NS, int PR>
hipError_t launch_persistent_variant(const GemmArgs& g, int workgroups, hipStream_t s)
{
    using S = TileShape<BM, BN, WM, WN, NS, WM * WN>;
    // four waves stage the finished tile beside the ring
    constexpr int LDS_TOTAL = S::LDS_BYTES + (WM * WN == 4 ? PR * BN * 2 : 0);
    const int tiles_m = (g.m + BM - 1) / BM, tiles_n = (g.n + BN - 1) / BN;
    constexpr auto kern = tile_gemm_persistent_kernel<BM, BN, WM, WN, NS, PR>;
    FP8GEMM_ALLOW_LDS(kern, LDS_TOTAL);
    launch_kernel(kern, dim3(workgroups), dim3(64 * WM * WN), LDS_TOTAL, s, g.a, g.b, g.a_scale,
                       g.b_scale, g.c, g.m, leading_dim(g), g.n, g.k, tiles_m, tiles_n);
    return hipGetLastError();
}

template <int BM, int BN, int WM, int WN, int NS, int PR>
hipError_t launch_grouped_variant(GroupTable& tab, int n, int k, int workgroups, hipStream_t s)
{
    using S = TileShape<BM, BN, WM, WN, NS>;
    constexpr int LDS_TOTAL = S::LDS_BYTES;
    const int tiles_n = (n + BN - 1) / BN;
    tab.tile_start[0] = 0;
    for (int g = 0; g < tab.groups; ++g)
        tab.tile_start[g + 1] = tab.tile_start[g] + ((tab.m[g] + BM - 1) / BM) * tiles_n;
    constexpr auto kern = tile_gemm_grouped_kernel<BM, BN, WM, WN, NS, PR>;
    FP8GEMM_ALLOW_LDS(kern, LDS_TOTAL);
    launch_kernel(kern, dim3(workgroups), dim3(NTHREADS), LDS_TOTAL, s, tab, n, k, tiles_n);
    return hipGetLastError();
}

// 128x256 tiles for groups of at most 128 rows, which bring more B than anything else: a launch streams every B once, from
// HBM, and is bound by the bytes that its CUs keep on their way there.  Tiles of 256x256 ask for B in the same whole pieces of
// 256 bytes, but half of their two slots is for rows that do not exist; here three slots fit, and a tile has half the MFMAs.
// A last round that leaves half of the workgroups idle is cut into 128x128 halves (large_tile_tail).  256x256 / this: 28 groups
// of 68 - 128 rows, 4608 x 7168, 229 / 206 us (925 MB of B: 4.5 TB/s); 64 of 3504 x 2944 208 / 185; 31 of 7168 x 2304 154 / 140; without
// halves 233 / 209 and 152 / 146.  B past the caches on top: -5.6 ... +2 %, +15 % where B fits the caches; not kept.
template <bool HALVES>
__global__ void __launch_bounds__(NTHREADS) tile_gemm_grouped_wide_kernel(const GroupTable tab, int N, int K, int tiles_n)
{
    const TileProblem none{nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0};
    using Whole = std::conditional_t<HALVES, FullRounds<128, 256>, AllTiles<128, 256>>;
    persistent_body<128, 256, 2, 4, 3, 64, true, Whole>(none, &tab, N, K, 0, tiles_n, (int)threadIdx.x);
    if constexpr (HALVES) {
        __syncthreads();  // nobody reads the ring any more
        persistent_body<128, 128, 2, 4, 4, 128, true, LeftOver<128, 256, 128, 128>>(none, &tab, N, K, 0, tiles_n, (int)threadIdx.x);
    }
}

hipError_t launch_grouped_wide(GroupTable& tab, int n, int k, int workgroups, hipStream_t s)
{
    constexpr int WHOLE = TileShape<128, 256, 2, 4, 3>::LDS_BYTES, PIECES = TileShape<128, 128, 2, 4, 4>::LDS_BYTES;
    constexpr int LDS_TOTAL = WHOLE > PIECES ? WHOLE : PIECES;
    const int tiles_n = (n + 255) / 256;
    tab.tile_start[0] = 0;
    for (int g = 0; g < tab.groups; ++g)
        tab.tile_start[g + 1] = tab.tile_start[g] + ((tab.m[g] + 127) / 128) * tiles_n;
    if (large_tile_tail(tab.tile_start[tab.groups], k, workgroups) == Tail::NONE) {
        constexpr auto kern = tile_gemm_grouped_wide_kernel<false>;
        FP8GEMM_ALLOW_LDS(kern, LDS_TOTAL);
        launch_kernel(kern, dim3(workgroups), dim3(NTHREADS), LDS_TOTAL, s, tab, n, k, tiles_n);
    } else {
        constexpr auto kern = tile_gemm_grouped_wide_kernel<true>;
        FP8GEMM_ALLOW_LDS(kern, LDS_TOTAL);
        launch_kernel(kern, dim3(workgroups), dim3(NTHREADS), LDS_TOTAL, s, tab, n, k, tiles_n);
    }
    return hipGetLastError();
}

int persistent_stages(int variant)
{
    switch (variant) {
    case TILE_128x256: return 4;  // of the halves
    case TILE_256x192: return 2;
    case TILE_256x128: return 3;
    case TILE_128x192: return 3;
    case TILE_128x128: return 4;
    case TILE_256x192_W4: return 2;
    case TILE_256x256: return 2;
    default: return 0;
    }
}

}  // namespace

bool tile_persistent_supports(const GemmArgs& g, int variant)
{
    const int stages = persistent_stages(variant);
    return stages > 0 && variant < TILE_VARIANT_COUNT && tile_supports(g) && g.k / KBLOCK >= stages - 1;
}

hipError_t launch_tile_persistent(const GemmArgs& g, int variant, int workgroups, hipStream_t s)
{
    if (workgroups <= 0 || workgroups % 8 != 0 || !tile_persistent_supports(g, variant))
        return hipErrorInvalidValue;
    switch (variant) {
    case TILE_256x192:
    case TILE_256x256: return launch_tile_large(g, variant, workgroups, s);
    case TILE_256x128: return launch_persistent_variant<256, 128, 4, 2, 3, 128>(g, workgroups, s);
    case TILE_128x192: return launch_persistent_variant<128, 192, 4, 2, 3, 128>(g, workgroups, s);
    case TILE_128x128: return launch_persistent_variant<128, 128, 2, 4, 4, 128>(g, workgroups, s);
    case TILE_256x192_W4: return launch_persistent_variant<256, 192, 2, 2, 2, 64>(g, workgroups, s);
    default: return hipErrorInvalidValue;
    }
}

// every group non-empty, aligned like a single problem, K long enough for the ring
bool tile_grouped_supports(const GroupTable& tab, int n, int k, int variant)
{
    const int stages = persistent_stages(variant);
    if (stages == 0 || variant == TILE_256x192_W4 ||  // the one-wave-per-SIMD loop is written for a single problem
        k / KBLOCK < stages - 1 || tab.groups < 1 || tab.groups > GroupTable::MAX_GROUPS)
        return false;
    for (int g = 0; g < tab.groups; ++g) {
        const GemmArgs ga{tab.a[g], tab.b[g], tab.a_scale[g], tab.b_scale[g], tab.c[g], tab.m[g], n, k, tab.lda[g]};
        if (tab.m[g] <= 0 || !tile_supports(ga))
            return false;
    }
    return true;
}

hipError_t launch_tile_grouped(GroupTable& tab, int n, int k, int variant, int workgroups, hipStream_t s)
{
    if (workgroups <= 0 || workgroups % 8 != 0 || !tile_grouped_supports(tab, n, k, variant))
        return hipErrorInvalidValue;
    switch (variant) {
    case TILE_256x192:
    case TILE_256x256: return launch_tile_large_grouped(tab, n, k, variant, workgroups, s);
    case TILE_256x128: return launch_grouped_variant<256, 128, 4, 2, 3, 128>(tab, n, k, workgroups, s);
    case TILE_128x192: return launch_grouped_variant<128, 192, 4, 2, 3, 128>(tab, n, k, workgroups, s);
    case TILE_128x128: return launch_grouped_variant<128, 128, 2, 4, 4, 128>(tab, n, k, workgroups, s);
    case TILE_128x256: return launch_grouped_wide(tab, n, k, workgroups, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace fp8gemm
