// Persistent form of the two large tiles (256 x 192, 256 x 256; eight waves of 64 x 96 / 64 x 128) for shapes with more
// tiles than compute units, and its grouped form.  Data path, fragments and fold are those of k_tile.hip (successor of
// in_smem_kernel, /root/reference/mn_large.hip:11-128; the reference lists a persistent kernel that overlaps the epilogue
// with the next tile as future work, /root/reference/README.md:29); the walk through the tiles is that of
// k_tile_persistent.hip: the K blocks of all tiles of a workgroup form one copy stream.
//
// Two slots of LDS are all that tiles of this size leave room for.  What the order of a K block is built around:
//   * The barrier of a block stands before its LAST TWO patch columns.  By then every fragment of the block is in
//     registers, so its slot is free for the block after next, whose copies go out right there; and the next block, asked for
//     one whole block earlier, has landed, so its first fragments are read under the last columns' MFMAs.  Those go row by
//     row, and a row of A is read as soon as the last MFMA that wants the old one is issued (no register on top): no MFMA
//     stands behind a barrier waiting for an LDS round trip.  With the barrier at the block's end all eight waves met there
//     with nothing in registers, and the matrix pipe idled for a quarter of the block.
//   * A patch is folded four MFMAs behind its own, across blocks too: every MFMA has four FMAs of another patch beside it,
//     none of which waits for its result.
//   * b_scale rides in the stage like a_scale: with a scalar load out, every wait for an LDS read is a wait for all.
//   * The loop knows its slot at compile time (two copies of the block): the slot is an immediate of every LDS read.
//   * A finished tile leaves through a staging area that each wave has to itself, beside the slots: no barrier, the copy
//     stream never pauses, and the copies of the next two blocks go out before the stores, so that no wait for them
//     is one for the stores (both count in vmcnt, in order; the stores are buffer stores that every wave issues, rows
//     and columns beyond C addressed outside the buffer, so their number is known).
//
// Bound by power on operands that toggle: 8192 x 4096 x 7168 (256 x 256) runs at a clock of 1.91 GHz with the matrix pipes
// 65 % busy; without its copies it takes 160 us.  Against 32x32x64 MFMAs with the barrier at the block's end and the
// tile leaving through a slot: 8192 x 4096 x 7168 212.7 -> 189 us = 51 % of 5033 TFLOP/s; 8192 x 4608 x 7168 (256 x 192) 252.8 ->
// 239; 8192 x 7168 x 2048 (256 x 192 and 256 x 256) 136.7 -> 129.5 and 123.8 -> 117; 8192 x 7168 x 256 32.8 -> 29; with C's
// stores past the caches (c_streams) 8192 x 4096 x 7168 180 us = 53 %.
#include "tile_persistent_body.h"

namespace fp8gemm {

namespace {

template <int BN>
struct LargeShape {
    static constexpr int BM = 256, WM = 4, WN = 2;
    using S = TileShape<BM, BN, WM, WN, 2>;
    static constexpr int TM = BM / WM, TN = BN / WN;
    static constexpr int MI = TM / 16, NJ = TN / 16;  // 16x16 patches of a wave
    static constexpr int MAT = KBLOCK * 256;          // one matrix of one slot: 128 k-rows of 256 bytes
    static constexpr int B_OFF = 2 * MAT;             // A of both slots, B of both slots (slot distance: a 16-bit immediate),
    static constexpr int SCALE_OFF = 4 * MAT;         // a_scale and b_scale of both slots
    static constexpr int SCALE_SLOT = 1024 + 256;
    // staging: 16 rows of a wave, all of its 96 columns or 64 of its 128
    static constexpr int SCOLS = TN == 96 ? 96 : 64;
    static constexpr int PARTS = TN / SCOLS;
    static constexpr int STORES = SCOLS * 2 * 16 / 1024;  // store instructions per part: 1 KiB each
    static constexpr int STAGING_OFF = SCALE_OFF + 2 * SCALE_SLOT;
    static constexpr int STAGING_WAVE = 16 * SCOLS * 2;
    static constexpr int LDS_BYTES = STAGING_OFF + 8 * STAGING_WAVE;
    static constexpr int TILE_STORES = MI * PARTS * STORES;
    static_assert(S::RSA == 256 && S::RSB == 256 && S::NA == 4 && S::NB == 4, "copy plan");
    static_assert(LDS_BYTES <= 160 * 1024, "slots and staging exceed the LDS");
    static_assert(TILE_STORES < 64, "vmcnt is a 6-bit field");
};

// The lane number, found out anew: what is worked out from it once per tile, or behind the tiles, is not kept through the
// K loop, which has no register left.
__device__ __forceinline__ int lane_now()
{
    uint32_t zero;
    asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
    return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, zero));
}

template <int BN, bool GROUPED, typename SHARE>
__device__ __forceinline__ void large_tile_body(const TileProblem& one, const GroupTable* tab, int N, int K, int tiles_m,
                                                int tiles_n, bool stream_c)
{
    using L = LargeShape<BN>;
    using S = typename L::S;
    constexpr int TM = L::TM, TN = L::TN, MI = L::MI, NJ = L::NJ, NA = S::NA, NB = S::NB;
    constexpr int NCOPY = NA + NB + 1;  // copy instructions of a wave per K block; the last one brings the scales
    constexpr bool STRADDLES = TN == 96;  // a wave's columns may lie in two b_scale blocks
    // A block's MFMAs: column by column of its patches, the last two columns row by row of theirs.
    constexpr int T = MI * NJ, BAR = MI * (NJ - 2);  // the barrier stands before MFMA number BAR
    auto row_of = [](int t) constexpr { return t < BAR ? t % MI : (t - BAR) / 2; };
    auto col_of = [](int t) constexpr { return t < BAR ? t / MI : NJ - 2 + (t - BAR) % 2; };
    constexpr int LAG = MI;  // a patch is folded LAG MFMAs behind its own, the last ones of a block in the next block
    // Copies of a block that go out behind the barrier of the block two before it (one MFMA each); the others ride on the
    // next block's first MFMAs.  The sooner they go out the sooner they land, and the closer together the more they hold each
    // other and the LDS reads up.  Grouped launches, whose operands come from HBM more than from the L2, want all of
    // them at once, single problems half of them (4 / 5 / 6 / 8 copies: eight groups of 250 - 2051 rows, 7168 x 2048 146.6 /
    // 143.9 / 143.5 / 142.2 us; 8192 x 4096 x 7168 189.7 / 190.8 / 194.4 / 195.9; 8192 x 7168 x 2048 119.8 / 118.8 / 119.3 / 119.0).
    constexpr int LATE = GROUPED ? 8 : 5;
    static_assert(T % LAG == 0 && T - BAR >= LATE, "schedule");

    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    auto lds = LDS_PTR(uint8_t, smem);
    const uint32_t lds_base = (uint32_t)(uintptr_t)lds;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave % L::WM, wn = wave / L::WM;

    const TileWalk<SHARE, GROUPED> walk(one, tab, tiles_m, tiles_n);
    const int n_my = walk.count();
    if (n_my == 0)
        return;
    const int nkb = K / KBLOCK;
    const int sn = (N + KBLOCK - 1) / KBLOCK;

    // ---- the copy stream: K block f_kb of this workgroup's tile number f_tile is the next one to be copied
    v4i rsrc_a, rsrc_b, rsrc_s, rsrc_bs;
    int f_lda = one.lda;
    uint32_t voff_a[2], voff_b[2], voff_sc = 0x80000000u;
    int f_tile = 0, f_kb = 0;
    int fill_left = n_my * nkb;
    auto fill_setup = [&](int j) __attribute__((always_inline)) {
        TileProblem pr;
        int m0, n0;
        walk.origin(j, pr, m0, n0);
        const int lane = lane_now();
        if (GROUPED || j == 0) {
            rsrc_a = make_rsrc_words(pr.a, (uint32_t)pr.lda * (uint32_t)K);
            rsrc_b = make_rsrc_words(pr.b, (uint32_t)N * (uint32_t)K);
            rsrc_s = make_rsrc_words(pr.a_scale, (uint32_t)nkb * (uint32_t)pr.lda * 4u);
            rsrc_bs = make_rsrc_words(pr.b_scale, (uint32_t)nkb * (uint32_t)sn * 4u);
            f_lda = pr.lda;
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int r = (NA * wave + q) * 4 + (lane >> 4);
            const int cc = (lane & 15) ^ row_swizzle<256>(r);
            voff_a[q] = m0 + 16 * cc < pr.M ? (uint32_t)(r * pr.lda + m0 + 16 * cc) : 0x80000000u;
            voff_b[q] = 16 * cc < BN && n0 + 16 * cc < N ? (uint32_t)(r * N + n0 + 16 * cc) : 0x80000000u;
        }
        if (wave == 0)  // wave 0 brings a_scale, 16 bytes per lane, wave 1 b_scale[kb][n0/128 + lane]
            voff_sc = m0 + 4 * lane < pr.M ? (uint32_t)((m0 + 4 * lane) * 4) : 0x80000000u;
        else
            voff_sc = lane < 4 && (n0 >> 7) + lane < sn ? (uint32_t)(((n0 >> 7) + lane) * 4) : 0x80000000u;
    };
    // copy instruction q of the stream's next block; a stream that has run dry reads outside its buffers (nothing) and
    // writes zeros to a slot that nobody reads any more
    auto fill_copy = [&](auto slot_tag, int q) __attribute__((always_inline)) {
        constexpr int slot = decltype(slot_tag)::value;
        if (q < NA) {
            lds_dma16(rsrc_a, voff_a[q & 1], lds_base + (uint32_t)(slot * L::MAT + (NA * wave + q) * 1024),
                      (uint32_t)(f_kb * KBLOCK + (q >> 1) * 8) * (uint32_t)f_lda);
        } else if (q < NA + NB) {
            const int p = q - NA;
            lds_dma16(rsrc_b, voff_b[p & 1], lds_base + (uint32_t)(L::B_OFF + slot * L::MAT + (NB * wave + p) * 1024),
                      (uint32_t)(f_kb * KBLOCK + (p >> 1) * 8) * (uint32_t)N);
        } else {
            const uint32_t at = lds_base + (uint32_t)(L::SCALE_OFF + slot * L::SCALE_SLOT);
            lds_dma16_unless((uint32_t)wave, rsrc_s, voff_sc, at, (uint32_t)f_kb * (uint32_t)f_lda * 4u);
            lds_dma4_unless((uint32_t)wave ^ 1u, rsrc_bs, voff_sc, at + 1024, (uint32_t)f_kb * (uint32_t)sn * 4u);
        }
    };
    auto fill_advance = [&]() __attribute__((always_inline)) {
        --fill_left;
        if (++f_kb == nkb) {
            f_kb = 0;
            ++f_tile;
            if (fill_left > 0) {
                fill_setup(f_tile);
            } else {
                voff_a[0] = voff_a[1] = voff_b[0] = voff_b[1] = voff_sc = 0x80000000u;
            }
        }
    };

    // ---- LDS read addresses of slot 0 (opaque: what is added to them stays the immediate of the read)
    using LdsBytes = __attribute__((address_space(3))) uint8_t*;
    auto opaque = [&](uint32_t offset) __attribute__((always_inline)) {
        uint32_t x = lds_base + offset;
        asm volatile("" : "+v"(x));
        return (LdsBytes)(uintptr_t)x;
    };
    LdsBytes addr_a[MI], addr_b[NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
        addr_a[i] = opaque(frag_addr<256>(lane, (wm * TM) / 16 + i));
#pragma unroll
    for (int jj = 0; jj < NJ; ++jj)
        addr_b[jj] = opaque(L::B_OFF + frag_addr<256>(lane, (wn * TN) / 16 + jj));
    auto read_b = [&](int jj, int slot) __attribute__((always_inline)) { return read_frag<256>(addr_b[jj] + slot * L::MAT); };
    const LdsBytes addr_sa = opaque(L::SCALE_OFF + (uint32_t)((wm * TM + (lane & 15)) * 4));

    // ---- what the multiplying side knows of its tile
    TileProblem pr;
    int m0 = 0, n0 = 0;
    uint32_t addr_sb = 0, hi_mask[NJ / 2] = {};
    auto enter_tile = [&](int j) __attribute__((always_inline)) {
        walk.origin(j, pr, m0, n0);
        const int n_wave = n0 + wn * TN;
        addr_sb = L::SCALE_OFF + 1024 + 4u * (uint32_t)((n_wave >> 7) - (n0 >> 7));
        if (STRADDLES)
#pragma unroll
            for (int p = 0; p < NJ / 2; ++p)  // all ones when patch columns 2 p and 2 p + 1 lie in the second b_scale block
                hi_mask[p] = (uint32_t)-(int)(((n_wave + 32 * p) >> 7) > (n_wave >> 7));
    };

    v4f acc[MI][NJ], blk[LAG];
    v8i fa[MI], fb_first;  // on entry to a block: its A fragments and those of its first column of B
    float sc[MI];          // scales of the block being folded
    auto sum_of = [&](int t) __attribute__((always_inline)) -> v4f& { return acc[row_of(t)][col_of(t)]; };
    auto fold = [&](int t) __attribute__((always_inline)) {  // the patch of MFMA number t
#pragma unroll
        for (int e = 0; e < 4; ++e)
            sum_of(t)[e] = fmaf(sc[row_of(t)], blk[t % LAG][e], sum_of(t)[e]);
    };

    // One K block in slot SLOT.  FIRST = the first one of a tile: the sums start here, and the block after it has been
    // asked for already.
    auto k_block = [&](auto slot_tag, auto first_tag, int outstanding_stores) __attribute__((always_inline)) {
        constexpr int SLOT = decltype(slot_tag)::value;
        constexpr bool FIRST = decltype(first_tag)::value;
        using Slot = std::integral_constant<int, SLOT>;
        using Other = std::integral_constant<int, 1 - SLOT>;
        v8i fb[NJ];
        fb[0] = fb_first;
        // scales of this block (the stage holds b_scale[kb][n0/128 + 0..3])
        float sa[MI];
#pragma unroll
        for (int i = 0; i < MI; ++i)
            sa[i] = *LDS_PTR(float, addr_sa + SLOT * L::SCALE_SLOT + 64 * i);
        const float sb_lo = *LDS_PTR(float, lds + addr_sb + SLOT * L::SCALE_SLOT);
        const float sb_hi = STRADDLES ? *LDS_PTR(float, lds + addr_sb + SLOT * L::SCALE_SLOT + 4) : 0.f;
        auto scale_for = [&](int jj) __attribute__((always_inline)) {
            const float sbj = STRADDLES ? __uint_as_float((__float_as_uint(sb_hi) & hi_mask[jj / 2]) |
                                                          (__float_as_uint(sb_lo) & ~hi_mask[jj / 2]))
                                        : sb_lo;
#pragma unroll
            for (int i = 0; i < MI; ++i)
                sc[i] = sa[i] * sbj;
        };
        auto step = [&](int t) __attribute__((always_inline)) {
            if (t >= LAG) {
                // one product per patch row, for a pair of columns
                if ((t - LAG) % MI == 0 && t - LAG <= BAR && (t == LAG || (STRADDLES && (t - LAG) / MI % 2 == 0)))
                    scale_for((t - LAG) / MI);
                if (FIRST)
                    sum_of(t - LAG) = (v4f){0.f, 0.f, 0.f, 0.f};
                fold(t - LAG);
            } else if (!FIRST) {
                fold(T + t - LAG);  // of the block before
            }
            // The next MFMA comes behind this fold (it reads what passes through here).  Left alone, the compiler issues all
            // MFMAs of a block first and all folds after them.
            if (t + 1 < T && (t >= LAG || !FIRST)) {
                v4f& sum = sum_of(t >= LAG ? t - LAG : T + t - LAG);
                if (t < BAR)
                    asm volatile("" : "+v"(sum), "+v"(fa[row_of(t + 1)]));
                else
                    asm volatile("" : "+v"(sum), "+v"(fb[col_of(t + 1)]));
            }
            blk[t % LAG] = block_sum(fb[col_of(t)], fa[row_of(t)]);
        };
        int cq = LATE;
#pragma unroll
        for (int t = 0; t < BAR; ++t) {
            // B two columns ahead (one at the start: the third buffer is in use until the block before ends)
            if (t == 0)
                fb[1] = read_b(1, SLOT);
            if (t == 2)
                fb[2] = read_b(2, SLOT);
            if (t % MI == 0 && t >= MI)
                fb[t / MI + 2] = read_b(t / MI + 2, SLOT);
            step(t);
            if (!FIRST && cq < NCOPY)
                fill_copy(Other{}, cq++);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (!FIRST)
            fill_advance();
        // every fragment of the block is in registers, the next block has landed
        if (FIRST && outstanding_stores > 0)
            wait_vmcnt<L::TILE_STORES>();
        else
            wait_vmcnt<0>();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        fb_first = read_b(0, 1 - SLOT);
#pragma unroll
        for (int t = BAR; t < T; ++t) {
            step(t);
            if (col_of(t) == NJ - 1)
                fa[row_of(t)] = read_frag<256>(addr_a[row_of(t)] + (1 - SLOT) * L::MAT);
            if (t - BAR < LATE)
                fill_copy(Slot{}, t - BAR);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (FIRST)  // folded behind the next block's first MFMAs, or behind the tile's last
#pragma unroll
            for (int t = T - LAG; t < T; ++t)
                sum_of(t) = (v4f){0.f, 0.f, 0.f, 0.f};
    };
    // ---- a finished tile: bf16, 16 rows of the wave at a time through its own staging area, 16 bytes per lane along rows.
    // A lane owns row m = .. + (lane & 15) and, per patch, a run of 4 columns; the chunks of a staged row are permuted
    // so that the 16 rows x two 8-byte pieces that are written together lie in different banks.
    auto store_tile = [&]() __attribute__((always_inline)) {
        const int ln = lane_now();
        constexpr int CPR = L::SCOLS / 8;  // 16-byte chunks per staged row
        const uint32_t staging = (uint32_t)(L::STAGING_OFF + wave * L::STAGING_WAVE);
        auto at = [&](int row, int ch) __attribute__((always_inline)) {
            return staging + (uint32_t)(row * (L::SCOLS * 2) + ((ch ^ (CPR == 8 ? (row >> 1) & 7 : (row >> 2) & 3)) << 4));
        };
        const __amdgpu_buffer_rsrc_t rc = make_rsrc(pr.c, (uint32_t)pr.M * (uint32_t)N * 2u);
        const int m_wave = m0 + wm * TM, n_wave = n0 + wn * TN;
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int part = 0; part < L::PARTS; ++part) {
#pragma unroll
                for (int jj = 0; jj < L::SCOLS / 16; ++jj) {
                    const v4f v = acc[i][part * (L::SCOLS / 16) + jj];
                    const v2i pk = {(int)pack_bf16x2(v[0], v[1]), (int)pack_bf16x2(v[2], v[3])};
                    *LDS_PTR(v2i, lds + at(ln & 15, 2 * jj + (ln >> 5)) + (ln & 16) / 2) = pk;
                }
                asm volatile("" ::: "memory");
#pragma unroll
                for (int it = 0; it < L::STORES; ++it) {
                    const int idx = it * 64 + ln;
                    const int row = idx / CPR, ch = idx - row * CPR;
                    const int mrow = m_wave + 16 * i + row, ncol = n_wave + part * L::SCOLS + 8 * ch;
                    const v4i v = *LDS_PTR(v4i, lds + at(row, ch));
                    const uint32_t off = mrow < pr.M && ncol < N ? ((uint32_t)mrow * (uint32_t)N + (uint32_t)ncol) * 2u : 0xFFFFFFF0u;
                    if (stream_c)
                        __builtin_amdgcn_raw_buffer_store_b128(v, rc, off, 0, 2);  // nt
                    else
                        __builtin_amdgcn_raw_buffer_store_b128(v, rc, off, 0, 0);
                }
                asm volatile("" ::: "memory");
            }
    };

    using Slot0 = std::integral_constant<int, 0>;
    using Slot1 = std::integral_constant<int, 1>;
    // ---- the first two blocks of the stream, the first one's fragments
    fill_setup(0);
#pragma unroll
    for (int q = 0; q < NCOPY; ++q)
        fill_copy(Slot0{}, q);
    fill_advance();
#pragma unroll
    for (int q = 0; q < NCOPY; ++q)
        fill_copy(Slot1{}, q);
    fill_advance();
    wait_vmcnt<NCOPY - 1>();  // waves that bring no scales: the first block; the others: and their first copy of the second
    asm volatile("s_barrier" ::: "memory");
    fb_first = read_b(0, 0);
#pragma unroll
    for (int i = 0; i < MI; ++i)
        fa[i] = read_frag<256>(addr_a[i]);

    int slot = 0;  // of the block multiplied next
    for (int j = 0; j < n_my; ++j) {
        enter_tile(j);
        int kb = 1;
        if (slot == 0) {
            k_block(Slot0{}, std::true_type{}, j);
            if (kb < nkb) {
                k_block(Slot1{}, std::false_type{}, 0);
                ++kb;
            } else {
                slot = 1;
            }
        } else {
            k_block(Slot1{}, std::true_type{}, j);
            slot = 0;
        }
        if (kb < nkb) {
            for (; kb + 1 < nkb; kb += 2) {
                k_block(Slot0{}, std::false_type{}, 0);
                k_block(Slot1{}, std::false_type{}, 0);
            }
            if (kb < nkb) {
                k_block(Slot0{}, std::false_type{}, 0);
                slot = 1;
            }
        }
#pragma unroll
        for (int t = T - LAG; t < T; ++t)
            fold(t);
        // the rest of the copies of the block after next, ahead of the stores
        if (slot == 0) {
#pragma unroll
            for (int q = LATE; q < NCOPY; ++q)
                fill_copy(Slot1{}, q);
        } else {
#pragma unroll
            for (int q = LATE; q < NCOPY; ++q)
                fill_copy(Slot0{}, q);
        }
        fill_advance();
        store_tile();
    }
    wait_vmcnt<0>();  // no copy may land in LDS that has been given to somebody else
}

template <Tail TAIL>
constexpr int tail_lds_bytes()
{
    return TAIL == Tail::NONE ? 0 : TAIL == Tail::HALVES ? TileShape<256, 128, 4, 2, 3>::LDS_BYTES : TileShape<128, 128, 2, 4, 4>::LDS_BYTES;
}

template <int BN, bool GROUPED, Tail TAIL>
__device__ __forceinline__ void large_kernel_body(const TileProblem& one, const GroupTable* tab, int N, int K, int tiles_m,
                                                  int tiles_n, bool stream_c)
{
    if constexpr (TAIL == Tail::NONE) {
        large_tile_body<BN, GROUPED, AllTiles<256, BN>>(one, tab, N, K, tiles_m, tiles_n, stream_c);
    } else {
        static_assert(BN == 256, "halves and quarters of 256x256");
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        large_tile_body<BN, GROUPED, FullRounds<256, BN>>(one, tab, N, K, tiles_m, tiles_n, stream_c);
        __syncthreads();  // nobody reads the slots any more
        const int thread = 64 * wave + lane_now();
        if constexpr (TAIL == Tail::HALVES)
            persistent_body<256, 128, 4, 2, 3, 128, GROUPED, LeftOver<256, 256, 256, 128>>(one, tab, N, K, tiles_m,
                                                                                                   tiles_n, thread);
        else
            persistent_body<128, 128, 2, 4, 4, 128, GROUPED, LeftOver<256, 256, 128, 128>>(one, tab, N, K, tiles_m,
                                                                                                   tiles_n, thread);
    }
}

template <int BN, Tail TAIL>
__global__ void __launch_bounds__(NTHREADS)
tile_gemm_large_kernel(const uint8_t* __restrict__ a, const uint8_t* __restrict__ b, const float* __restrict__ a_scale,
                       const float* __restrict__ b_scale, uint16_t* __restrict__ c, int M, int lda, int N, int K, int tiles_m,
                       int tiles_n, int stream_c)
{
    const TileProblem one{a, b, a_scale, b_scale, c, M, lda};
    large_kernel_body<BN, false, TAIL>(one, nullptr, N, K, tiles_m, tiles_n, stream_c != 0);
}

template <int BN, Tail TAIL>
__global__ void __launch_bounds__(NTHREADS)
tile_gemm_large_grouped_kernel(const GroupTable tab, int N, int K, int tiles_n, int stream_c)
{
    const TileProblem none{nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0};
    large_kernel_body<BN, true, TAIL>(none, &tab, N, K, 0, tiles_n, stream_c != 0);
}

// Whether C leaves with stores that tell the caches not to keep it (whole tiles; halves and quarters are stored as ever).  The tiles of a round are stored together, 32 MB in a few
// microseconds, and the lines that the L2s and the Infinity Cache then hold have to leave under the next rounds' reads.
// Where the launch's data are small enough to stay, so does C.  Kept / not kept, us, three sets of operands in turn,
// bytes of A, B and C together: 92 MB 8192 x 4096 x 2048 61.1 / 63.2; 108 MB 4608 x 4608 x 7168 139.0 / 137.0; 111 MB 8192 x
// 5120 x 2048 79.5 / 80.8; 117 MB 8192 x 4096 x 4096 112.2 / 108.1, 4096 x 8192 x 4096 113.3 / 108.4; 130 MB 8192 x 6144 x 2048
// 91.3 / 88.2; 155 MB 8192 x 4096 x 7168 187.7 / 180.2; 167 MB 8192 x 4608 x 7168 232.9 / 226.0; with the quantiser in front 8192
// x 7168 x 2048 129.4 / 120.6.
int c_streams(long rows, long weights, int n, int k)
{
    return (double)rows * k + (double)weights * n * k + 2.0 * rows * n >= 115e6 ? 1 : 0;
}

template <int BN, Tail TAIL>
hipError_t launch_large(const GemmArgs& g, int workgroups, hipStream_t s)
{
    constexpr int LDS = LargeShape<BN>::LDS_BYTES > tail_lds_bytes<TAIL>() ? LargeShape<BN>::LDS_BYTES : tail_lds_bytes<TAIL>();
    constexpr auto kern = tile_gemm_large_kernel<BN, TAIL>;
    FP8GEMM_ALLOW_LDS(kern, LDS);
    launch_kernel(kern, dim3(workgroups), dim3(NTHREADS), LDS, s, g.a, g.b, g.a_scale, g.b_scale, g.c, g.m,
                       leading_dim(g), g.n, g.k, (g.m + 255) / 256, (g.n + BN - 1) / BN, c_streams(g.m, 1, g.n, g.k));
    return hipGetLastError();
}

template <int BN, Tail TAIL>
hipError_t launch_large_grouped(const GroupTable& tab, int n, int k, int workgroups, hipStream_t s)
{
    constexpr int LDS = LargeShape<BN>::LDS_BYTES > tail_lds_bytes<TAIL>() ? LargeShape<BN>::LDS_BYTES : tail_lds_bytes<TAIL>();
    constexpr auto kern = tile_gemm_large_grouped_kernel<BN, TAIL>;
    FP8GEMM_ALLOW_LDS(kern, LDS);
    long rows = 0;
    for (int g = 0; g < tab.groups; ++g)
        rows += tab.m[g];
    launch_kernel(kern, dim3(workgroups), dim3(NTHREADS), LDS, s, tab, n, k, (n + BN - 1) / BN,
                       c_streams(rows, tab.groups, n, k));
    return hipGetLastError();
}

}  // namespace

// An XCD's run of tiles, less the rounds in which each of its workgroups gets one, cut so that every workgroup gets at most
// one piece.  Behind the full rounds a ring of stages starts anew, which halves need eight K blocks to make up for (full
// tiles / halves, 8192 x 7168, half a round left over: K = 512 42.7 / 44.1 us, 1024 69.6 / 69.2, 1536 92.7 / 90.9, 2048
// 118.0 / 114.0) and quarters none (8192 x 4608, a quarter left over: 512 29.8 / 29.2, 1024 45.2 / 43.4, 3072 115.1 /
// 106.0, 7168 251.7 / 233.2; 4096 x 4608, an eighth on top of one round: 2048 49.4 / 42.0, 4096 90.4 / 74.5).
Tail large_tile_tail(long tiles, int k, int workgroups)
{
    const int per_xcd = workgroups / 8, nkb = k / KBLOCK;
    const long most = (tiles + 7) / 8;  // the XCDs' runs differ by one
    const long left = most % per_xcd;
    if (most < per_xcd || left == 0 || tiles / 8 / per_xcd != most / per_xcd)
        return Tail::NONE;
    if (4 * left <= per_xcd && nkb >= 3)  // the ring's depth
        return Tail::QUARTERS;
    return 2 * left <= per_xcd && nkb >= 8 ? Tail::HALVES : Tail::NONE;
}

hipError_t launch_tile_large(const GemmArgs& g, int variant, int workgroups, hipStream_t s)
{
    if (variant == TILE_256x192)
        return launch_large<192, Tail::NONE>(g, workgroups, s);
    const long tiles = (long)((g.m + 255) / 256) * ((g.n + 255) / 256);
    switch (large_tile_tail(tiles, g.k, workgroups)) {
    case Tail::QUARTERS: return launch_large<256, Tail::QUARTERS>(g, workgroups, s);
    case Tail::HALVES: return launch_large<256, Tail::HALVES>(g, workgroups, s);
    default: return launch_large<256, Tail::NONE>(g, workgroups, s);
    }
}

hipError_t launch_tile_large_grouped(GroupTable& tab, int n, int k, int variant, int workgroups, hipStream_t s)
{
    const int bn = variant == TILE_256x192 ? 192 : 256, tiles_n = (n + bn - 1) / bn;
    tab.tile_start[0] = 0;
    for (int g = 0; g < tab.groups; ++g)
        tab.tile_start[g + 1] = tab.tile_start[g] + ((tab.m[g] + 255) / 256) * tiles_n;
    if (variant == TILE_256x192)
        return launch_large_grouped<192, Tail::NONE>(tab, n, k, workgroups, s);
    switch (large_tile_tail(tab.tile_start[tab.groups], k, workgroups)) {
    case Tail::QUARTERS: return launch_large_grouped<256, Tail::QUARTERS>(tab, n, k, workgroups, s);
    case Tail::HALVES: return launch_large_grouped<256, Tail::HALVES>(tab, n, k, workgroups, s);
    default: return launch_large_grouped<256, Tail::NONE>(tab, n, k, workgroups, s);
    }
}

}  // namespace fp8gemm
