// The body of the persistent tile kernels with a ring of LDS stages (k_tile_persistent.hip tells what it does), also the
// second part of the large tiles' kernels (k_tile_large.hip).
#pragma once
#include "tile_common.h"

namespace fp8gemm {

namespace {

#include "w4_loop.inc"

// GROUPED = false: one problem (`one`), tiles_m x tiles_n tiles.  GROUPED = true: the problems of
// `tab` (same N and K, own M), whose tiles are numbered one group after the other.
// thread = the thread's number in the workgroup.  SHARE = which tiles (TileWalk), tiles_m and tiles_n count its walk's tiles.
template <int BM, int BN, int WM, int WN, int NS, int PR, bool GROUPED, typename SHARE = AllTiles<BM, BN>>
__device__ __forceinline__ void persistent_body(const TileProblem& one, const GroupTable* tab, int N, int K,
                                                int tiles_m, int tiles_n, int thread)
{
    constexpr int NW = WM * WN;    // waves per workgroup; four = one wave per SIMD (k_block_w4)
    constexpr int NTH = 64 * NW;
    using S = TileShape<BM, BN, WM, WN, NS, NW>;
    static_assert(NW == 8 || NW == 4, "eight or four waves per workgroup");
    static_assert(NS >= 2 && NS <= 4, "two to four LDS stages");
    constexpr int TM = BM / WM, TN = BN / WN;
    constexpr int MI = TM / 16, NJ = TN / 16;  // 16x16 patches
    static_assert(TM % 32 == 0 && TN % 32 == 0 && TN <= 128 && BM <= 256 && BN <= 256, "wave tile");
    constexpr int RSA = S::RSA, RSB = S::RSB, NA = S::NA, NB = S::NB, NCOPY = S::NCOPY;
    // Staging bytes per tile row.  16 rows x two 8-byte pieces of one chunk are written together: the chunks of a row are
    // permuted by the row (staged_chunk) so that they lie in different banks without any padding.
    constexpr int CROW = BN * 2;
    static_assert(BN % 128 == 0 || BN % 128 == 64, "rows that start on a multiple of half the banks");
    static_assert(PR % 16 == 0 && BM % PR == 0, "a piece is a whole number of patches");
    static_assert(PR * CROW <= S::STAGE, "a piece must fit one ring slot");
    // four waves: the finished tile is staged beside the ring, which then never pauses
    constexpr int STAGING_W4 = NS * S::STAGE;
    static_assert(NW == 8 || STAGING_W4 + PR * CROW <= 160 * 1024, "ring and staging area exceed the LDS");
    constexpr int CPR = BN / 8;               // 16-byte chunks per tile row
    constexpr int CHUNKS = PR * CPR;

    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    auto lds = LDS_PTR(uint8_t, smem);
    const uint32_t lds_base = (uint32_t)(uintptr_t)lds;

    const int lane = thread & 63;
    const int wave = __builtin_amdgcn_readfirstlane(thread >> 6);
    const int wm = wave % WM, wn = wave / WM;

    const TileWalk<SHARE, GROUPED> walk(one, tab, tiles_m, tiles_n);
    const int n_my = walk.count();
    if (n_my == 0)
        return;

    const int nkb = K / KBLOCK;
    const int sn = (N + KBLOCK - 1) / KBLOCK;
    // buffer resources of the copy stream's current tile (fixed for a single problem)
    v4i rsrc_a, rsrc_b, rsrc_s, rsrc_bs;
    int f_lda = one.lda;  // leading dimension of the problem the copy stream is in
    auto set_resources = [&](const TileProblem& pr) __attribute__((always_inline)) {
        rsrc_a = make_rsrc_words(pr.a, (uint32_t)pr.lda * (uint32_t)K);
        rsrc_b = make_rsrc_words(pr.b, (uint32_t)N * (uint32_t)K);
        rsrc_s = make_rsrc_words(pr.a_scale, (uint32_t)nkb * (uint32_t)pr.lda * 4u);
        rsrc_bs = make_rsrc_words(pr.b_scale, (uint32_t)nkb * (uint32_t)sn * 4u);
        f_lda = pr.lda;
    };

    // ---- the copy stream: K block f_kb of this workgroup's tile number f_tile is the next one
    // to be copied.  Per-lane offsets (copy plan of k_tile.hip) belong to that tile.
    uint32_t voff_a[S::NVA], voff_b[S::NVB], voff_s, voff_sb = 0x80000000u;
    int f_tile = 0, f_kb = 0;
    int fill_left = n_my * nkb;  // blocks not yet copied
    auto fill_setup = [&](int j) __attribute__((always_inline)) {
        TileProblem pr;
        int m0, n0;
        walk.origin(j, pr, m0, n0);
        if (GROUPED || j == 0)
            set_resources(pr);
        const int M = pr.M, lda = pr.lda;
#pragma unroll
        for (int q = 0; q < S::NVA; ++q) {
            const int r = RSA == 256 ? (NA * wave + q) * 4 + (lane >> 4) : (NA * wave + q) * 8 + (lane >> 3);
            const int cc = (RSA == 256 ? (lane & 15) : (lane & 7)) ^ row_swizzle<RSA>(r);
            const bool ok = (16 * cc < BM) && (m0 + 16 * cc < M);
            voff_a[q] = ok ? (uint32_t)(r * lda + m0 + 16 * cc) : 0x80000000u;
        }
#pragma unroll
        for (int q = 0; q < S::NVB; ++q) {
            const int r = RSB == 256 ? (NB * wave + q) * 4 + (lane >> 4) : (NB * wave + q) * 8 + (lane >> 3);
            const int cc = (RSB == 256 ? (lane & 15) : (lane & 7)) ^ row_swizzle<RSB>(r);
            const bool ok = (16 * cc < BN) && (n0 + 16 * cc < N);
            voff_b[q] = ok ? (uint32_t)(r * N + n0 + 16 * cc) : 0x80000000u;
        }
        voff_s = (4 * lane < BM && m0 + 4 * lane < M) ? (uint32_t)((m0 + 4 * lane) * 4) : 0x80000000u;
        if (NW == 4)  // lanes 0..3 bring b_scale[kb][n0/128 + lane]
            voff_sb = (lane < 4 && (n0 >> 7) + lane < sn) ? (uint32_t)(((n0 >> 7) + lane) * 4) : 0x80000000u;
    };
    // copy instruction q of the stream's next block into ring slot `slot`
    auto fill_copy = [&](int slot, int q) __attribute__((always_inline)) {
        const uint32_t stage = lds_base + (uint32_t)(slot * S::STAGE);
        if (q < NA) {
            lds_dma16(rsrc_a, voff_a[S::template voff_index<RSA>(q)], stage + (uint32_t)((NA * wave + q) * 1024),
                      (uint32_t)(f_kb * KBLOCK + S::template extra_rows<RSA>(q)) * (uint32_t)f_lda);
        } else if (q < NA + NB) {
            lds_dma16(rsrc_b, voff_b[S::template voff_index<RSB>(q - NA)],
                      stage + S::MAT_A + (uint32_t)((NB * wave + (q - NA)) * 1024),
                      (uint32_t)(f_kb * KBLOCK + S::template extra_rows<RSB>(q - NA)) * (uint32_t)N);
        } else if (NW == 8) {
            lds_dma16_unless((uint32_t)wave, rsrc_s, voff_s, stage + S::SCALE_OFF, (uint32_t)f_kb * (uint32_t)f_lda * 4u);
        } else if (wave == 0) {
            lds_dma16(rsrc_s, voff_s, stage + S::SCALE_OFF, (uint32_t)f_kb * (uint32_t)f_lda * 4u);
        } else if (NW == 4 && wave == 1) {
            lds_dma4(rsrc_bs, voff_sb, stage + S::SB_OFF, (uint32_t)f_kb * (uint32_t)sn * 4u);
        }
    };
    auto fill_advance = [&]() __attribute__((always_inline)) {
        --fill_left;
        if (++f_kb == nkb) {
            f_kb = 0;
            ++f_tile;
            if (fill_left > 0)
                fill_setup(f_tile);
        }
    };

    // ---- LDS read addresses (k_tile.hip): they do not depend on the tile
    uint32_t addr_a[MI], addr_b[NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
        addr_a[i] = frag_addr<RSA>(lane, (wm * TM) / 16 + i);
#pragma unroll
    for (int j = 0; j < NJ; ++j)
        addr_b[j] = S::MAT_A + frag_addr<RSB>(lane, (wn * TN) / 16 + j);
    const uint32_t addr_s = S::SCALE_OFF + (uint32_t)((wm * TM + (lane & 15)) * 4);

    // ---- a finished tile: bf16, in pieces of PR rows through `staging` (LDS bytes that nobody
    // else touches meanwhile), 16 bytes per lane along whole tile rows.  A lane owns row
    // m = .. + (lane & 15) and, per patch, a run of 4 columns: stored straight from the
    // registers that would be 8-byte pieces of 16 different rows per instruction.
    // sum(i, jj, e) = running sum e of patch (i, jj)
    auto staged_chunk = [&](int row, int ch) __attribute__((always_inline)) {  // LDS offset of chunk ch of a piece's row
        return (uint32_t)(row * CROW + ((ch ^ (BN % 128 == 0 ? row & 15 : (row >> 1) & 7)) << 4));
    };
    auto store_tile = [&](auto sum, uint32_t staging, int m0, int n0, int M,
                          uint16_t* __restrict__ c) __attribute__((always_inline)) {
        // opaque copy of the thread id: keeps the address arithmetic below inside the tile loop
        // (hoisted, it would sit in registers the K loop needs and be spilled)
        int tid = thread;
        asm volatile("" : "+v"(tid));
        const int lane_e = tid & 63;
#pragma unroll
        for (int p = 0; p < BM / PR; ++p) {
            if (p > 0)
                __syncthreads();  // the previous piece has been read out
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                const int prow = wm * TM + 16 * i;
                if (prow / PR == p) {
                    const int row = prow - p * PR + (lane_e & 15);
#pragma unroll
                    for (int jj = 0; jj < NJ; ++jj) {
                        const int col = wn * TN + 16 * jj + 4 * (lane_e >> 4);
                        v2i pk = {(int)pack_bf16x2(sum(i, jj, 0), sum(i, jj, 1)),
                                  (int)pack_bf16x2(sum(i, jj, 2), sum(i, jj, 3))};
                        *LDS_PTR(v2i, lds + staging + staged_chunk(row, col >> 3) + (col & 4) * 2) = pk;
                    }
                }
            }
            __syncthreads();
#pragma unroll
            for (int it = 0; it < (CHUNKS + NTH - 1) / NTH; ++it) {
                const int idx = it * NTH + tid;
                const int row = idx / CPR, ch = idx - row * CPR;
                const int mrow = m0 + p * PR + row;
                const int ncol = n0 + ch * 8;
                if (idx < CHUNKS && mrow < M && ncol < N) {
                    *reinterpret_cast<v4i*>(c + (size_t)mrow * N + ncol) = *LDS_PTR(v4i, lds + staging + staged_chunk(row, ch));
                }
            }
        }
    };

    if constexpr (NW == 4) {
        // ================= one wave per SIMD =================
        // A wave owns a 128 x 96 patch grid (2.33 transposing reads per MFMA instead of the 3.33 of
        // a 64 x 96 wave tile) and all 512 registers of its SIMD lane.  Nobody else issues on the
        // SIMD, so the K blocks run as one assembly loop with every instruction placed by hand
        // (w4_loop.inc; schedule, register map and wait counts: gen_w4_loop.py).  What that loop
        // does differently from the eight-wave schedule below:
        //   * the barrier of a K block sits before its LAST patch column: by then all fragments of
        //     the block are in registers, so the slot is free for the block after next right away,
        //     and the fragments of the next block (landed a whole block ago) are read while the
        //     last column is multiplied -- no MFMA waits for an LDS round trip behind a barrier;
        //   * the fold of a block's last patch rides on the first MFMAs of the next block;
        //   * b_scale rides in the stage like a_scale (a scalar load in flight would turn the
        //     counted LDS waits into full ones);
        //   * the finished tile is staged beside the two ring slots: the copy stream never pauses.
        // This part only walks the tiles, keeps the copy stream's bookkeeping and stores the tiles.
        static_assert(BM == 256 && BN == 192 && WM == 2 && WN == 2 && NS == 2 && !GROUPED,
                      "the assembly loop is written for this shape");
        static_assert(S::STAGE == 66816 && NA == 8 && NB == 8, "ring geometry the assembly loop assumes");
        const uint32_t scale_kind = wave < 2 ? (uint32_t)wave : 2u;
        const uint32_t lds_wave = lds_base + (uint32_t)(NA * wave * 1024);
        const uint32_t lds_scale = lds_base + (wave == 0 ? S::SCALE_OFF : S::SB_OFF);
        // the even patch of each pair; the odd one's address differs in bit 4 (the pair's chunks are 2 i and 2 i + 1)
        const uint32_t vbase_a0 = lds_base + addr_a[0], vbase_a1 = lds_base + addr_a[2];
        const uint32_t vbase_a2 = lds_base + addr_a[4], vbase_a3 = lds_base + addr_a[6];
        const uint32_t vbase_b0 = lds_base + addr_b[0], vbase_b1 = lds_base + addr_b[2], vbase_b2 = lds_base + addr_b[4];
        const uint32_t vaddr_s = lds_base + addr_s;

        v32f sums[6], blk;
        v32i frag0 = {}, frag1 = {}, frag2 = {};
        v16i frag3 = {};
        v2f scale_carry = {0.f, 0.f};
#pragma unroll
        for (int r = 0; r < 32; ++r)
            blk[r] = 0.f;

        // once the stream has run dry its copy instructions stay in the loop with offsets outside
        // their buffers: they fetch nothing and write zeros into the slot nobody reads
        auto stream_dry = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int q = 0; q < S::NVA; ++q)
                voff_a[q] = 0x80000000u;
#pragma unroll
            for (int q = 0; q < S::NVB; ++q)
                voff_b[q] = 0x80000000u;
            voff_s = voff_sb = 0x80000000u;
        };
        fill_setup(0);
#pragma unroll
        for (int q = 0; q < NCOPY; ++q)
            fill_copy(0, q);
        fill_advance();
        if (fill_left > 0) {
#pragma unroll
            for (int q = 0; q < NCOPY; ++q)
                fill_copy(1, q);
            fill_advance();
            wait_vmcnt<NCOPY - 1>();  // block 0 landed (waves 0 and 1: and their first copy of block 1)
        } else {
            wait_vmcnt<0>();
        }
        if (fill_left == 0)
            stream_dry();
        __syncthreads();
        w4_first_reads(frag0, frag1, frag2, frag3, vbase_a0, vbase_a1, vbase_a2, vbase_a3, vbase_b0);

        uint32_t slot_off = 0;  // LDS offset of the ring slot of the block multiplied next
        for (int j = 0; j < n_my; ++j) {
            TileProblem pr;
            int m0, n0;
            walk.origin(j, pr, m0, n0);
            const int n_wave = n0 + wn * TN;
            // the stage holds b_scale[kb][n0/128 + 0..3]; a wave's n range touches at most two of them
            const uint32_t lds_sb_lo = lds_base + S::SB_OFF + 4u * (uint32_t)((n_wave >> 7) - (n0 >> 7));
            const uint32_t lds_sb_hi = lds_base + S::SB_OFF + 4u * (uint32_t)(((n_wave + TN - 1) >> 7) - (n0 >> 7));
            uint32_t hi_mask[NJ / 2];  // all ones when patch columns 2 jj and 2 jj + 1 lie in the wave's second b_scale block
#pragma unroll
            for (int jj = 0; jj < NJ / 2; ++jj)
                hi_mask[jj] = (uint32_t)-(int)(((n_wave + 32 * jj) >> 7) > (n_wave >> 7));
#pragma unroll
            for (int t = 0; t < 6; ++t)
#pragma unroll
                for (int r = 0; r < 32; ++r)
                    sums[t][r] = 0.f;

            int kb = 0;
            while (kb < nkb) {
                // as many blocks as the copy stream can take without leaving its tile
                int cnt = nkb - kb;
                if (fill_left > 0 && nkb - f_kb < cnt)
                    cnt = nkb - f_kb;
                uint32_t count = (uint32_t)cnt;
                const uint32_t str_a = (uint32_t)(KBLOCK * f_lda), str_b = (uint32_t)(KBLOCK * N);
                const uint32_t str_sc = wave == 0 ? (uint32_t)f_lda * 4u : (uint32_t)sn * 4u;
                uint32_t off_a = (uint32_t)f_kb * str_a, off_b = (uint32_t)f_kb * str_b, off_sc = (uint32_t)f_kb * str_sc;
                // wave-uniform operands of the loop must sit in scalar registers
                auto sgpr = [](uint32_t x) __attribute__((always_inline)) {
                    return (uint32_t)__builtin_amdgcn_readfirstlane((int)x);
                };
                off_a = sgpr(off_a), off_b = sgpr(off_b), off_sc = sgpr(off_sc), count = sgpr(count);
                slot_off = sgpr(slot_off);
                w4_k_blocks(sums[0], sums[1], sums[2], sums[3], sums[4], sums[5], blk, frag0, frag1, frag2, frag3,
                            scale_carry, vbase_a0, vbase_a1, vbase_a2, vbase_a3, vbase_b0, vbase_b1, vbase_b2,
                            vaddr_s, voff_a[0], voff_a[1], voff_b[0], voff_b[1], wave == 0 ? voff_s : voff_sb,
                            rsrc_a, rsrc_b, wave == 0 ? rsrc_s : rsrc_bs, off_a, off_b, off_sc, sgpr(str_a),
                            sgpr(str_b), sgpr(str_sc), sgpr((uint32_t)(8 * f_lda)), sgpr((uint32_t)(8 * N)), slot_off,
                            sgpr(lds_wave), sgpr(lds_scale), sgpr(scale_kind), sgpr(lds_sb_lo), sgpr(lds_sb_hi),
                            sgpr(hi_mask[0]), sgpr(hi_mask[1]), sgpr(hi_mask[2]), count);
                kb += cnt;
                if (fill_left > 0) {
                    fill_left -= cnt;
                    f_kb += cnt;
                    if (f_kb == nkb) {
                        f_kb = 0;
                        ++f_tile;
                        if (fill_left > 0)
                            fill_setup(f_tile);
                        else
                            stream_dry();
                    }
                }
            }
            // the last patch's fold, then the tile leaves through the staging area
            w4_last_fold(sums[5], blk, scale_carry);
            scale_carry = (v2f){0.f, 0.f};
#pragma unroll
            for (int r = 16; r < 32; ++r)
                blk[r] = 0.f;
            store_tile([&](int i, int jj, int r) __attribute__((always_inline)) {
                           const int q = (jj / 2) * (MI / 2) + i / 2;  // pair of patch rows and columns
                           return sums[q / 2][(q % 2) * 16 + 8 * (i % 2) + 4 * (jj % 2) + r];
                       },
                       (uint32_t)STAGING_W4, m0, n0, pr.M, pr.c);
        }
        return;
    }

    // ---- fill the ring: the first NS-1 blocks of the stream
    fill_setup(0);
#pragma unroll
    for (int p = 0; p < NS - 1; ++p)
        if (fill_left > 0) {
#pragma unroll
            for (int q = 0; q < NCOPY; ++q)
                fill_copy(p, q);
            fill_advance();
        }
    int slot = 0;            // ring slot of the block being multiplied
    int slot_fill = NS - 1;  // ring slot the stream's next block goes into

    for (int j = 0; j < n_my; ++j) {
        TileProblem pr;
        int m0, n0;
        walk.origin(j, pr, m0, n0);
        const float* __restrict__ b_scale = pr.b_scale;
        uint16_t* __restrict__ c = pr.c;
        const int M = pr.M;
        const int n_wave = n0 + wn * TN;
        int nb_lo = n_wave >> 7, nb_hi = (n_wave + TN - 1) >> 7;
        nb_lo = nb_lo < sn ? nb_lo : sn - 1;
        nb_hi = nb_hi < sn ? nb_hi : sn - 1;
        uint32_t hi_mask[NJ / 2];  // all ones when patch columns 2 jj and 2 jj + 1 lie in the wave's second b_scale block
#pragma unroll
        for (int jj = 0; jj < NJ / 2; ++jj)
            hi_mask[jj] = (uint32_t)-(int)(((n_wave + 32 * jj) >> 7) > (n_wave >> 7));

        v4f acc[MI][NJ];
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int jj = 0; jj < NJ; ++jj)
                acc[i][jj] = (v4f){0.f, 0.f, 0.f, 0.f};

        float next_lo = b_scale[__builtin_amdgcn_readfirstlane(nb_lo)];
        float next_hi = b_scale[__builtin_amdgcn_readfirstlane(nb_hi)];

        // One K block.  MORE = the stream has a block left to copy (always, except for the last
        // NS-1 blocks of the last tile).
        auto k_block = [&](auto more_tag, int kb) __attribute__((always_inline)) {
            constexpr bool more = decltype(more_tag)::value;
            // The first NS-1 blocks of a later tile were copied before the previous tile's
            // epilogue, which waited for them: no wait here, and none that would drag in that
            // epilogue's stores.  Otherwise at most the younger blocks may be outstanding.
            const bool landed = j > 0 && kb < NS - 1;
            if (!landed) {
                if (more) {
                    wait_vmcnt<(NS - 2) * (NCOPY - 1)>();
                } else {
                    const int younger = (nkb - 1 - kb < NS - 2) ? (nkb - 1 - kb) : (NS - 2);
                    if (NS >= 4 && younger >= 2)
                        wait_vmcnt<2 * (NCOPY - 1)>();
                    else if (NS >= 3 && younger >= 1)
                        wait_vmcnt<NCOPY - 1>();
                    else
                        wait_vmcnt<0>();
                }
            }
            __syncthreads();  // block landed for everyone; slot_fill is no longer read
            // b_scale of this block, asked for during the last one (k_tile.hip)
            const float sb_lo = next_lo, sb_hi = next_hi;
            asm volatile("" ::"s"(sb_lo), "s"(sb_hi));
            const uint32_t so = (uint32_t)(slot * S::STAGE);
            auto ask_next_scale = [&]() __attribute__((always_inline)) {
                int next = __builtin_amdgcn_readfirstlane(kb + 1 < nkb ? kb + 1 : kb);
                asm volatile("" : "+s"(next));
                next_lo = b_scale[__builtin_amdgcn_readfirstlane(next * sn + nb_lo)];
                next_hi = b_scale[__builtin_amdgcn_readfirstlane(next * sn + nb_hi)];
            };
            // fragments, steps and folds as in k_tile.hip
            v8i fa[MI], fb[NJ];
            fb[0] = read_frag<RSB>(lds + (addr_b[0] + so));
#pragma unroll
            for (int i = 0; i < MI; ++i)
                fa[i] = read_frag<RSA>(lds + (addr_a[i] + so));
            if (NJ > 1)
                fb[1] = read_frag<RSB>(lds + (addr_b[1] + so));
            float sa[MI], sc[MI];
#pragma unroll
            for (int i = 0; i < MI; ++i)
                sa[i] = *LDS_PTR(float, lds + so + addr_s + 64 * i);
            constexpr int T = MI * NJ, PER_MFMA = (NCOPY + T - 1) / T;
            constexpr int LAG = MI < 4 && T >= 12 ? 6 : MI;
            v4f blk[LAG];
            auto fold = [&](int t) __attribute__((always_inline)) {
                if (t % MI == 0) {
                    // wave-uniform choice of the b_scale value on the scalar unit (bit select), then one product per patch
                    const float sbj = __uint_as_float((__float_as_uint(sb_hi) & hi_mask[t / MI / 2]) |
                                                      (__float_as_uint(sb_lo) & ~hi_mask[t / MI / 2]));
#pragma unroll
                    for (int i = 0; i < MI; ++i)
                        sc[i] = sa[i] * sbj;
                }
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    acc[t % MI][t / MI][e] = fmaf(sc[t % MI], blk[t % LAG][e], acc[t % MI][t / MI][e]);
            };
#pragma unroll
            for (int t = 0; t < T; ++t) {
                if (t % MI == 0 && t > 0 && t / MI + 1 < NJ)
                    fb[t / MI + 1] = read_frag<RSB>(lds + (addr_b[t / MI + 1] + so));
                if (t >= LAG) {
                    fold(t - LAG);
                    if (t + 1 < T)
                        asm volatile("" : "+v"(acc[(t - LAG) % MI][(t - LAG) / MI]), "+v"(fa[(t + 1) % MI]));
                }
                blk[t % LAG] = block_sum(fb[t / MI], fa[t % MI]);
                if (more)
#pragma unroll
                    for (int q = t * PER_MFMA; q < (t + 1) * PER_MFMA; ++q)
                        if (q < NCOPY)
                            fill_copy(slot_fill, q);
                if (t == T - 1)
                    ask_next_scale();
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int t = T - LAG; t < T; ++t) {
                fold(t);
                asm volatile("" : "+v"(acc[t % MI][t / MI]));
            }
            if (more)
                fill_advance();
            slot_fill = slot;
            slot = (slot + 1 == NS) ? 0 : slot + 1;
        };

        // the host launches this kernel only for nkb >= NS-1: the stream then runs dry in the
        // last NS-1 blocks of the last tile and nowhere else
        const int tail = (j + 1 < n_my) ? 0 : NS - 1;
        int kb = 0;
        for (; kb < nkb - tail; ++kb)
            k_block(std::true_type{}, kb);
        for (; kb < nkb; ++kb)
            k_block(std::false_type{}, kb);

        // ---- epilogue: bf16, in pieces of PR rows through the ring slot of the block multiplied
        // last (slot_fill by now; the stream's next copy goes there, but not before the next
        // K block's barrier).  Every copy of the stream issued so far has to have landed before
        // the first store goes out: the next tile's first blocks are then known to be there
        // without a wait that would also cover these stores.
        wait_vmcnt<0>();
        __syncthreads();  // every wave has finished reading that slot
        // (the same steps as store_tile, written out: handed to that lambda through an accessor, the
        // running sums cost the K loop 9 more registers and the kernel 1-2 % on the headline shape)
        {
            const uint32_t staging = (uint32_t)(slot_fill * S::STAGE);
            int tid = thread;
            asm volatile("" : "+v"(tid));
            const int lane_e = tid & 63;
#pragma unroll
            for (int p = 0; p < BM / PR; ++p) {
                if (p > 0)
                    __syncthreads();  // the previous piece has been read out
#pragma unroll
                for (int i = 0; i < MI; ++i) {
                    const int prow = wm * TM + 16 * i;
                    if (prow / PR == p) {
                        const int row = prow - p * PR + (lane_e & 15);
#pragma unroll
                        for (int jj = 0; jj < NJ; ++jj) {
                            const int col = wn * TN + 16 * jj + 4 * (lane_e >> 4);
                            v2i pk = {(int)pack_bf16x2(acc[i][jj][0], acc[i][jj][1]),
                                      (int)pack_bf16x2(acc[i][jj][2], acc[i][jj][3])};
                            *LDS_PTR(v2i, lds + staging + staged_chunk(row, col >> 3) + (col & 4) * 2) = pk;
                        }
                    }
                }
                __syncthreads();
#pragma unroll
                for (int it = 0; it < (CHUNKS + NTH - 1) / NTH; ++it) {
                    const int idx = it * NTH + tid;
                    const int row = idx / CPR, ch = idx - row * CPR;
                    const int mrow = m0 + p * PR + row;
                    const int ncol = n0 + ch * 8;
                    if (idx < CHUNKS && mrow < M && ncol < N) {
                        *reinterpret_cast<v4i*>(c + (size_t)mrow * N + ncol) = *LDS_PTR(v4i, lds + staging + staged_chunk(row, ch));
                    }
                }
            }
        }
        // the next tile's first K block begins with a barrier: the slot is not written again
        // before every lane has read its chunks of the last piece
    }
}

}  // namespace
}  // namespace fp8gemm
