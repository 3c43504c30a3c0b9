// MFMA tile kernel for gfx950: the successor of in_smem_kernel (/root/reference/mn_large.hip:11-128)
// and, with the K range split over workgroups, of k_large_kernel (/root/reference/mn_small.hip:10-137).
//
// Data path (all of it differs from the reference, which scatters single bytes into LDS):
//   * A ([K][M], m contiguous) and B ([K][N], n contiguous) tiles of 128 K-rows are copied
//     global -> LDS with 16-byte buffer loads that write LDS directly (no VGPR round trip),
//     keeping the global orientation: one LDS row per k, 128 or 256 bytes per row.  The
//     16-byte column chunk c of row r is stored at chunk position c ^ swizzle(r), which makes
//     the transposing reads below bank-conflict free (measured: the conflicts of a launch do not grow with K).
//   * Operands are fetched with ds_read_b64_tr_b8: 16 lanes read an 8(k) x 16(m|n) byte
//     patch and receive it transposed, i.e. lane i holds 8 consecutive k of column i.  Four
//     such reads give the 32 bytes per lane that v_mfma_f32_16x16x128_f8f6f4 consumes.
//     The k order inside the instruction is permuted identically for both operands, which
//     leaves the dot product unchanged.
//   * One MFMA covers a 128-wide scale block of one 16x16 patch; the block sum
//     lives in 4 registers for a moment and is folded into the running result with
//     a_scale[kb][m] * b_scale[kb][n/128] by one FMA per element (mn_large.hip:100-106,
//     mn_small.hip:85-88 do the same with a second full-size accumulator).  Why this instruction and not two of
//     32x32x64: with the fold beside them, on operands of quantised normal values, nothing else in the loop, it
//     sustains 65.5 % of the peak against 58.2 % (78.6 against 74.2 % on constant operands: the rest is power), from as
//     many LDS reads; its block sums are as far from the exact ones (2-norm 1.3e-5 and 2.3e-5 with outliers, both).
//   * The MFMA computes the transposed patch (rows = n, columns = m) as mn_small.hip does,
//     so that a lane owns one m (one a_scale value) and runs of 4 consecutive n.
//   * The finished tile goes through the idle LDS ring (row-major, padded rows) and leaves as
//     16 bytes per lane along whole tile rows; straight from the accumulators a store
//     instruction would write 8-byte pieces of 32 different rows.
//   * a_scale values of the tile travel through LDS with the stage (one extra 1 KiB copy), so
//     the K loop holds no compiler-visible global load and every wait on the copies is the
//     explicit one below.  b_scale is asked for by scalar loads one K block ahead: in the block that
//     needs it its trip to the L2 would stand in front of the MFMAs (from the Infinity Cache, 128 x 128
//     tiles, 336 x 4608 x 7168: 27.1 -> 22.6 us; 1024 x 1536 x 7168: 24.9 -> 21.6 us).  Where only four waves
//     multiply, a wave that does not copies b_scale into the stage (64x64 tiles, which are done before that
//     trip is: 48 x 4608 x 7168 14.2 -> 10.9 us).
//   * The two smaller tiles, 64x64 and 128x128, are multiplied by four waves, one per SIMD, and copied by the other
//     four (128x128 with short chains: by eight, see four_waves).  What bounds a K block of them is the
//     LDS: where a block stands by itself, the reads of all waves come first (640 clocks for 128x128 in eight waves of
//     64x32) and the MFMAs, 512 clocks, behind them.  Four waves of 64x64 read two thirds of that, and they read
//     block kb + 1 into a second set of registers between the MFMAs of block kb, so that a block takes the longer of
//     the two and not their sum; the folds of a block's last four sums cross the barrier.  Eight waves with the reads
//     at the head of the block / this, from the Infinity Cache: 5504 x 512 x 7168 30.7 / 26.4 us, 2048 x 2048 x 7168
//     36.1 / 32.0, 1024 x 1536 x 7168 21.4 / 19.1, 352 x 3072 x 1536 9.4 / 8.6, 350 x 3072 x 1536 (RAGGED) 11.3 / 10.4;
//     64x64 tiles 1024 x 512 x 2048 6.1 / 5.85, 64 x 4608 x 7168, bound by the copies, 10.4 / 10.6.  From HBM the
//     copies bound a block: 5504 x 512 x 7168 35.0 / 36.1, 2048 x 2048 x 7168 39.9 / 39.4, 1024 x 1536 x 7168 21.3 / 20.0.
//     Copies between the MFMAs of a lone wave hold them up (RAGGED with B copied there: 350 x 3072 x 1536 12.3 us), so
//     they are the other waves'.  Eight stages of 64x64 instead of four: 5.9 -> 6.8 us.
//   * NS LDS stages form a ring: the copies of K blocks kb+1 .. kb+NS-1 are in flight while
//     block kb is multiplied.  Large tiles fit two stages; smaller tiles get three or four,
//     which is what hides the global latency when a K block is only a few MFMAs long.
//   * Where all eight waves multiply, the copy instructions of a K block ride on the first MFMAs of an earlier block instead
//     of being issued in one burst after the barrier (a burst queues up in the address unit
//     and holds every wave back from its LDS reads).
//
//   * RAGGED: M is no multiple of 16, so A's k-rows start anywhere and 16-byte copies straight to LDS are out.  Four of
//     the eight waves (two of the four that do not multiply) load A's pieces into registers from where they lie (a load
//     takes any address; measured: no slower off the grid than on it) and write them to the ring a step before they are
//     read, two or three register sets ahead; the others copy B and the scales as ever.  Each kind has a loop of its own,
//     so that the compiler's waits count the loads of A alone.  A K block takes 0.05 - 0.1 us more than with copies
//     throughout (128 x 128 in eight waves, 336 x 4608 from the Infinity Cache: 0.53 -> 0.59 us), and the launch that
//     copied A into padded rows is gone: 121 x 7168 x 256 5.6 -> 3.8 us, 244 x 3072 x 1536 9.2 -> 7.0, 1021 x 512 x 2048
//     11.4 -> 7.7, 2204 x 512 x 7168 26.9 -> 21.2.
//
// Work decomposition: grid.x = tiles (XCD-aware order), grid.y = K splits.
#include "tile_common.h"

namespace fp8gemm {

namespace {

// v >> (8 * by) as one 128-bit number, by < 16
__device__ __forceinline__ v4i shift_right_bytes(v4i v, uint32_t by)
{
    const unsigned __int128 x = __builtin_bit_cast(unsigned __int128, v);
    return __builtin_bit_cast(v4i, x >> (8 * by));
}

// One tile of one problem, in K blocks blockIdx.y * kb_per_split ...: the tile at (m0, n0), number `pid` of the launch.
// RAGGED: M may be no multiple of 16 (see the head of this file)
template <int BM, int BN, int WM, int WN, int NS, bool SPLIT, bool RAGGED>
__device__ __forceinline__ void
tile_body(const uint8_t* __restrict__ a, const uint8_t* __restrict__ b, const float* __restrict__ a_scale,
          const float* __restrict__ b_scale, uint16_t* __restrict__ c, float* __restrict__ partial, float* mailbox,
          int M, int lda, int N, int K, int m0, int n0, int pid, int kb_per_split)
{
    using S = TileShape<BM, BN, WM, WN, NS>;
    // WM x WN waves multiply: all eight, or the first four of the two smaller tiles (AHEAD)
    static_assert(WM * WN == 8 || WM * WN == 4, "eight or four multiplying waves");
    constexpr int NCW = WM * WN;
    static_assert(NCW == 4 ? NS == 4 : NS >= 2 && NS <= 4, "LDS stages");
    constexpr int TM = BM / WM, TN = BN / WN;      // wave tile
    constexpr int MI = TM / 16, NJ = TN / 16;      // 16x16 patches per wave
    static_assert(TM % 16 == 0 && TN % 32 == 0, "wave tile is made of 16x16 patches, pairs of them along n");
    static_assert(TN <= 128, "a wave's n range touches at most two 128-wide scale blocks");
    static_assert(BM <= 256 && BN <= 256, "LDS rows hold at most 256 bytes");
    constexpr int RSA = S::RSA, RSB = S::RSB, NA = S::NA, NB = S::NB, NCOPY = S::NCOPY;
    static_assert(!RAGGED || NS >= 3, "A's registers are written a step ahead of the multiply");
    // Who copies: all eight waves; the four that do not multiply, if there are such.  RAGGED: waves 0 - 3 copy B and the
    // scales and waves 4 - 7 load A; where those do not multiply, waves 4 and 5 load A and waves 6 and 7 copy.
    constexpr bool AHEAD = NCW == 4;
    constexpr int A_WAVE = 4, A_WAVES = AHEAD ? 2 : 4, NAW = 8 / A_WAVES * NA;
    constexpr int COPIERS = !AHEAD && !RAGGED ? 8 : AHEAD && RAGGED ? 2 : 4;
    constexpr int NBW = 8 / COPIERS * NB, NAC = RAGGED ? 0 : 8 / COPIERS * NA;  // copies of such a wave per K block
    constexpr int SETS = NS - 1, LEAD = SETS + 1;  // register sets of A, and K blocks that they run ahead
    // RAGGED, eight waves multiply: A's registers are emptied behind the first MFMA of a block; with two sets only behind its
    // last one, a step is short for the loads' trip (128x192, per K block from the Infinity Cache: 0.83 us early, 0.76 us
    // late; 128x128 with three sets 0.59 and 0.61 us)
    constexpr bool A_EARLY = SETS >= 3;
    static_assert(!RAGGED || BM <= 64 * COPIERS, "a wave that copies for every 64 rows of a_scale");

    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    auto lds = LDS_PTR(uint8_t, smem);
    const uint32_t lds_base = (uint32_t)(uintptr_t)lds;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int copier = wave & (COPIERS - 1);
    const int wm = wave % WM, wn = (wave / WM) % WN;
    const bool compute = !AHEAD || wave < NCW;

    const int nkb = K / KBLOCK;
    const int kb0 = blockIdx.y * kb_per_split;
    const int kb1 = (kb0 + kb_per_split < nkb) ? (kb0 + kb_per_split) : nkb;

    // ---- global -> LDS copy plan.  One 16-byte load per lane fills 1 KiB of LDS (LDS address
    // = base + lane*16): 4 rows of 256 B, 8 rows of 128 B or 16 rows of 64 B.  Wave w owns instructions
    // NA*w .. NA*w+NA-1 of the A tile and likewise of B.  A lane writes chunk position p of
    // row r and therefore fetches column chunk p ^ swizzle(r).  Chunks outside the tile or the
    // matrix get an out-of-range offset: the buffer load then writes zeros and reads nothing.
    uint32_t voff_a[S::NVA], voff_b[S::NVB];  // RAGGED: voff_a is not used, voff_b by the waves that copy
#pragma unroll
    for (int q = 0; q < S::NVA; ++q) {
        const int r = (NAC * copier + q) * (1024 / RSA) + S::template copy_row<RSA>(lane);
        const int cc = S::template copy_pos<RSA>(lane) ^ row_swizzle<RSA>(r);
        const bool ok = (16 * cc < BM) && (m0 + 16 * cc < M);
        voff_a[q] = ok ? (uint32_t)(r * lda + m0 + 16 * cc) : 0x80000000u;
    }
#pragma unroll
    for (int q = 0; q < S::NVB; ++q) {
        const int r = (NBW * copier + q) * (1024 / RSB) + S::template copy_row<RSB>(lane);
        const int cc = S::template copy_pos<RSB>(lane) ^ row_swizzle<RSB>(r);
        const bool ok = (16 * cc < BN) && (n0 + 16 * cc < N);
        voff_b[q] = ok ? (uint32_t)(r * N + n0 + 16 * cc) : 0x80000000u;
    }
    const uint32_t a_bytes = (uint32_t)lda * (uint32_t)K, b_bytes = (uint32_t)N * (uint32_t)K;
    const uint32_t as_bytes = (uint32_t)nkb * (uint32_t)lda * 4u;
    // a_scale: 16 bytes per lane by one wave; rows that do not start on the 16-byte grid by 4 bytes per lane and a wave
    // for every 64 of them
    const int scale_m = RAGGED ? m0 + 64 * copier + lane : m0 + 4 * lane;
    const uint32_t voff_s = (RAGGED ? 64 * copier < BM : 4 * lane < BM) && scale_m < M ? (uint32_t)(scale_m * 4) : 0x80000000u;

    // RAGGED: the 16 bytes per lane that a copy instruction would bring, by a load from wherever they lie; pieces
    // without a row of the matrix bring the tile's first one instead
    uint32_t off_a[NAW];
    v4i set_a[SETS][NAW];
    const bool loads_a = wave >= A_WAVE && wave < A_WAVE + A_WAVES;
    const int a_first = NAW * (wave - A_WAVE);  // first KiB of the A tile that the wave brings
    if constexpr (RAGGED) {
#pragma unroll
        for (int q = 0; q < NAW; ++q) {
            const int r = (a_first + q) * (1024 / RSA) + S::template copy_row<RSA>(lane);
            const int cc = S::template copy_pos<RSA>(lane) ^ row_swizzle<RSA>(r);
            const bool ok = (16 * cc < BM) && (m0 + 16 * cc < M);
            off_a[q] = (uint32_t)r * (uint32_t)M + (uint32_t)(ok ? m0 + 16 * cc : m0);
        }
    }
    // Nothing beyond the matrix is read: a piece of its last row that would reach there is its last 16 bytes instead,
    // shifted into place behind the wait.
    const uint32_t last_piece = (uint32_t)KBLOCK * (uint32_t)M - 16u;  // where they start in the last K block
    auto load_a = [&](v4i(&set)[NAW], int kb) __attribute__((always_inline)) {
        const uint8_t* const block = a + (size_t)kb * KBLOCK * (uint32_t)M;
        const uint32_t last = kb == nkb - 1 ? last_piece : 0xFFFFFFFFu;
#pragma unroll
        for (int q = 0; q < NAW; ++q)
            __builtin_memcpy(&set[q], block + min(off_a[q], last), 16);
    };
    auto write_a = [&](auto inner_tag, v4i(&set)[NAW], int slot, int kb) __attribute__((always_inline)) {
        if (!decltype(inner_tag)::value && kb == nkb - 1) {
#pragma unroll
            for (int q = 0; q < NAW; ++q)
                set[q] = shift_right_bytes(set[q], off_a[q] > last_piece ? off_a[q] - last_piece : 0u);
        }
#pragma unroll
        for (int q = 0; q < NAW; ++q)
            *LDS_PTR(v4i, lds + (uint32_t)(slot * S::STAGE + (a_first + q) * 1024 + lane * 16)) = set[q];
    };

    // copy instruction q (0..NCOPY-1) of K block kb into ring slot `slot`.  The three buffer
    // resources stay fixed; the K block's byte offset rides in the scalar offset operand.
    const v4i rsrc_a = make_rsrc_words(a, a_bytes), rsrc_b = make_rsrc_words(b, b_bytes);
    const v4i rsrc_s = make_rsrc_words(a_scale, as_bytes);
    const int sn = (N + KBLOCK - 1) / KBLOCK;
    const v4i rsrc_bs = make_rsrc_words(b_scale, (uint32_t)nkb * (uint32_t)sn * 4u);
    const uint32_t voff_sb = lane == 0 ? (uint32_t)((n0 >> 7) * 4) : 0x80000000u;  // staged: the tile is at most 128 wide
    auto copy_b = [&](uint32_t stage, int kb, int q) __attribute__((always_inline)) {
        lds_dma16(rsrc_b, voff_b[S::template voff_index<RSB>(q)], stage + S::MAT_A + (uint32_t)((NBW * copier + q) * 1024),
                  (uint32_t)(kb * KBLOCK + S::template extra_rows<RSB>(q)) * (uint32_t)N);
    };
    auto copy_step = [&](int slot, int kb, int q) __attribute__((always_inline)) {
        const uint32_t stage = lds_base + (uint32_t)(slot * S::STAGE);
        if (q < NA) {
            lds_dma16(rsrc_a, voff_a[S::template voff_index<RSA>(q)], stage + (uint32_t)((NA * wave + q) * 1024),
                      (uint32_t)(kb * KBLOCK + S::template extra_rows<RSA>(q)) * (uint32_t)lda);
        } else if (q < NA + NB) {
            copy_b(stage, kb, q - NA);
        } else {
            lds_dma16_unless((uint32_t)wave, rsrc_s, voff_s, stage + S::SCALE_OFF, (uint32_t)kb * (uint32_t)lda * 4u);
        }
    };
    // RAGGED and AHEAD: all copies of a wave at once
    auto copy_all = [&](int slot, int kb) __attribute__((always_inline)) {
        const uint32_t stage = lds_base + (uint32_t)(slot * S::STAGE);
        if constexpr (!RAGGED) {
#pragma unroll
            for (int q = 0; q < NAC; ++q)
                lds_dma16(rsrc_a, voff_a[S::template voff_index<RSA>(q)], stage + (uint32_t)((NAC * copier + q) * 1024),
                          (uint32_t)(kb * KBLOCK + S::template extra_rows<RSA>(q)) * (uint32_t)lda);
        }
#pragma unroll
        for (int q = 0; q < NBW; ++q)
            copy_b(stage, kb, q);
        if constexpr (!RAGGED) {
            if (copier == 0)
                lds_dma16(rsrc_s, voff_s, stage + S::SCALE_OFF, (uint32_t)kb * (uint32_t)lda * 4u);
            else if (copier == 1)
                lds_dma4(rsrc_bs, voff_sb, stage + S::SB_OFF, (uint32_t)kb * (uint32_t)sn * 4u);
            return;
        }
        if (64 * copier < BM)
            lds_dma4(rsrc_s, voff_s, stage + S::SCALE_OFF + (uint32_t)(256 * copier), (uint32_t)kb * (uint32_t)M * 4u);
        if (S::SB_STAGED && copier == COPIERS - 1)
            lds_dma4(rsrc_bs, voff_sb, stage + S::SB_OFF, (uint32_t)kb * (uint32_t)sn * 4u);
    };

    // ---- transposing LDS reads: one address per patch row and column (frag_addr)
    uint32_t addr_a[MI], addr_b[NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
        addr_a[i] = frag_addr<RSA>(lane, (wm * TM) / 16 + i);
#pragma unroll
    for (int j = 0; j < NJ; ++j)
        addr_b[j] = S::MAT_A + frag_addr<RSB>(lane, (wn * TN) / 16 + j);
    const uint32_t addr_s = S::SCALE_OFF + (uint32_t)((wm * TM + (lane & 15)) * 4);

    // ---- scales.  One a_scale per lane and 16-row patch (the lane's m).  A wave's n range is at
    // most 128 wide, so it touches at most two 128-wide b_scale blocks (nb_lo, nb_hi); a pair of
    // patch columns (32 wide) never straddles a block boundary.
    const int n_wave = n0 + wn * TN;
    int nb_lo = n_wave >> 7, nb_hi = (n_wave + TN - 1) >> 7;
    nb_lo = nb_lo < sn ? nb_lo : sn - 1;
    nb_hi = nb_hi < sn ? nb_hi : sn - 1;
    uint32_t hi_mask[NJ / 2];  // all ones when patch columns 2 j and 2 j + 1 lie in the wave's second b_scale block
#pragma unroll
    for (int j = 0; j < NJ / 2; ++j)
        hi_mask[j] = (uint32_t)-(int)(((n_wave + 32 * j) >> 7) > (n_wave >> 7));

    v4f acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
            acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};

    if constexpr (AHEAD) {
        // Iteration kb multiplies what the last one read into registers and reads block kb + 1; the slot of block kb is
        // free behind its barrier and gets block kb + NS.
        constexpr int PER_BLOCK = NAC + NBW;  // copies of a wave per block, or one or two short
        auto wait_block = [&](int kb) __attribute__((always_inline)) {  // at most the copies of the younger blocks are out
            const int younger = kb1 - 1 - kb;
            if (younger >= NS - 2)
                wait_vmcnt<(NS - 2) * PER_BLOCK>();
            else if (younger == 1)
                wait_vmcnt<PER_BLOCK>();
            else
                wait_vmcnt<0>();
        };
        // The first blocks are copied by all waves that have nothing else to do: the first two by those that multiply
        // (RAGGED: by two of them each), the others by those that copy later on.
        if (compute) {
            if constexpr (RAGGED) {
                if (kb0 + (wave >> 1) < kb1)
                    copy_all(wave >> 1, kb0 + (wave >> 1));
                if (wave < 2)
                    wait_vmcnt<0>();
            } else {
                if (kb0 < kb1)
                    copy_all(0, kb0);
                if (kb0 + 1 < kb1) {
                    copy_all(1, kb0 + 1);
                    wait_vmcnt<PER_BLOCK>();
                } else {
                    wait_vmcnt<0>();
                }
            }
        } else if (!(RAGGED && loads_a)) {
#pragma unroll
            for (int p = 2; p < NS; ++p)
                if (kb0 + p < kb1)
                    copy_all(p, kb0 + p);
        }
        if (RAGGED && loads_a) {
#pragma unroll
            for (int p = 0; p < SETS; ++p)
                if (kb0 + p < kb1)
                    load_a(set_a[p], kb0 + p);
            write_a(std::false_type{}, set_a[0], 0, kb0);
            if (kb0 + SETS < kb1)
                load_a(set_a[0], kb0 + SETS);
            __syncthreads();
            int slot_w = 1;
            auto step = [&](auto more_tag, auto set_tag, int at) __attribute__((always_inline)) {  // block at into the ring
                constexpr int set = decltype(set_tag)::value;
                constexpr bool steady = decltype(more_tag)::value;
                if (steady || at < kb1)
                    write_a(more_tag, set_a[set], slot_w, at);
                if (steady || at + SETS < kb1)
                    load_a(set_a[set], at + SETS);
                slot_w = slot_w + 1 == NS ? 0 : slot_w + 1;
                if (steady || at <= kb1)
                    __syncthreads();
            };
            static_assert(SETS == 3, "unrolled");
            int at = kb0 + 1;
            for (; at + 2 + SETS < kb1; at += SETS) {
                step(std::true_type{}, std::integral_constant<int, 1>{}, at);
                step(std::true_type{}, std::integral_constant<int, 2>{}, at + 1);
                step(std::true_type{}, std::integral_constant<int, 0>{}, at + 2);
            }
            for (; at <= kb1; at += SETS) {
                step(std::false_type{}, std::integral_constant<int, 1>{}, at);
                step(std::false_type{}, std::integral_constant<int, 2>{}, at + 1);
                step(std::false_type{}, std::integral_constant<int, 0>{}, at + 2);
            }
        } else if (!compute) {
            __syncthreads();
            int slot = 0, kb = kb0;
            for (; kb < kb1; ++kb) {
                if (kb + 1 < kb1)
                    wait_block(kb + 1);
                __syncthreads();
                if (kb + NS < kb1)
                    copy_all(slot, kb + NS);
                slot = slot + 1 == NS ? 0 : slot + 1;
            }
        } else {
            constexpr int T = MI * NJ, LAG = 4, FRAGS = MI + NJ, PER_MFMA = T >= 16 ? 1 : 2;
            static_assert(T % LAG == 0, "sums keep their registers from block to block");
            v8i fa[2][MI], fb[2][NJ];
            float sa[2][MI], sb[2], sc[2][MI];
            v4f blk[LAG];
#pragma unroll
            for (int i = 0; i < MI; ++i)
                sc[0][i] = sc[1][i] = 0.f;
#pragma unroll
            for (int i = 0; i < LAG; ++i)
                blk[i] = (v4f){0.f, 0.f, 0.f, 0.f};
            auto read = [&](int set, int f, uint32_t so) __attribute__((always_inline)) {
                if (f == 0)
                    fb[set][0] = read_frag<RSB>(lds + (addr_b[0] + so));
                else if (f <= MI)
                    fa[set][f - 1] = read_frag<RSA>(lds + (addr_a[f - 1] + so));
                else
                    fb[set][f - MI] = read_frag<RSB>(lds + (addr_b[f - MI] + so));
            };
            auto read_scales = [&](int set, uint32_t so) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < MI; ++i)
                    sa[set][i] = *LDS_PTR(float, lds + so + addr_s + 64 * i);
                sb[set] = *LDS_PTR(float, lds + so + S::SB_OFF);
            };
            auto fold = [&](int set, int t) __attribute__((always_inline)) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    acc[t % MI][t / MI][e] = fmaf(sc[set][t % MI], blk[t % LAG][e], acc[t % MI][t / MI][e]);
            };
            __syncthreads();
#pragma unroll
            for (int f = 0; f < FRAGS; ++f)
                read(0, f, 0);
            read_scales(0, 0);
            int slot = 0;
            // The first block: the barrier, behind which the next one has landed, stands behind half of the MFMAs, which need
            // not wait for those copies (before / after: 352 x 3072 x 1536 8.87 / 8.60 us, 1024 x 512 x 2048 5.99 / 5.85, 5504 x 512
            // x 7168 26.7 / 26.4, 64 x 4608 x 7168 10.5 / 10.6)
            auto block = [&](auto set_tag, auto first_tag) __attribute__((always_inline)) {
                constexpr int s = decltype(set_tag)::value;
                constexpr bool first = decltype(first_tag)::value;
                constexpr int R0 = first ? T / 2 : 0;  // the MFMA that the reads start with
                static_assert((T - R0) * PER_MFMA >= FRAGS, "all fragments are read");
                if (!first)
                    __syncthreads();
                slot = slot + 1 == NS ? 0 : slot + 1;
                const uint32_t so = (uint32_t)(slot * S::STAGE);
#pragma unroll
                for (int i = 0; i < MI; ++i)
                    sc[s][i] = sa[s][i] * sb[s];
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    const int u = t < LAG ? T - LAG + t : t - LAG;
                    if (first && t == R0) {
                        wait_vmcnt<0>();
                        __syncthreads();
                    }
                    fold(t < LAG ? 1 - s : s, u);
                    if (t + 1 < T)
                        asm volatile("" : "+v"(acc[u % MI][u / MI]), "+v"(fa[s][(t + 1) % MI]));
                    else
                        asm volatile("" : "+v"(acc[u % MI][u / MI]));
                    blk[t % LAG] = block_sum(fb[s][t / MI], fa[s][t % MI]);
#pragma unroll
                    for (int f = (t - R0) * PER_MFMA; f < (t - R0 + 1) * PER_MFMA; ++f)
                        if (t >= R0 && f < FRAGS)
                            read(1 - s, f, so);
                    if (t - R0 == (FRAGS + PER_MFMA - 1) / PER_MFMA - 1)
                        read_scales(1 - s, so);
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            using Set0 = std::integral_constant<int, 0>;
            using Set1 = std::integral_constant<int, 1>;
            int kb = kb0;
            if (kb < kb1) {
                block(Set0{}, std::true_type{});
                ++kb;
            }
            for (; kb + 1 < kb1; kb += 2) {
                block(Set1{}, std::false_type{});
                block(Set0{}, std::false_type{});
            }
            if (kb < kb1) {
                block(Set1{}, std::false_type{});
#pragma unroll
                for (int t = T - LAG; t < T; ++t)
                    fold(1, t);
            } else {
#pragma unroll
                for (int t = T - LAG; t < T; ++t)
                    fold(0, t);
            }
        }
    } else {
        // ---- prologue: the first NS-1 K blocks go into ring slots 0 .. NS-2
#pragma unroll
        for (int p = 0; p < NS - 1; ++p)
            if (kb0 + p < kb1) {
                if constexpr (RAGGED) {
                    if (!loads_a)
                        copy_all(p, kb0 + p);
                } else {
#pragma unroll
                    for (int q = 0; q < NCOPY; ++q)
                        copy_step(p, kb0 + p, q);
                }
            }
        int slot = 0;             // ring slot of block kb
        int slot_fill = NS - 1;   // ring slot that block kb + NS - 1 goes into (= slot of kb - 1)

        // b_scale of the next block (wave-uniform addresses: scalar loads)
        float next_lo = 0.f, next_hi = 0.f;
        next_lo = b_scale[__builtin_amdgcn_readfirstlane(kb0 * sn + nb_lo)];
        next_hi = b_scale[__builtin_amdgcn_readfirstlane(kb0 * sn + nb_hi)];

        // One K block.  MORE = block kb+NS-1 exists and is copied here; two instantiations keep the
        // steady-state body free of branches.
        auto k_block = [&](auto more_tag, auto loads_tag, auto set_tag, int kb) __attribute__((always_inline)) {
            constexpr bool loads_a = decltype(loads_tag)::value;
            constexpr bool steady = decltype(more_tag)::value;
            const bool more = steady || (RAGGED && kb + NS - 1 < kb1);
            // RAGGED: A of the next block into its slot, and its registers filled again
            auto next_a = [&]() __attribute__((always_inline)) {
                if constexpr (loads_a) {
                    constexpr int set = (decltype(set_tag)::value + 1) % SETS;
                    if (steady || kb + 1 < kb1)
                        write_a(more_tag, set_a[set], slot + 1 == NS ? 0 : slot + 1, kb + 1);  // steady: not the last block
                    if (steady || kb + LEAD < kb1)
                        load_a(set_a[set], kb + LEAD);
                }
            };
            // Block kb has landed once at most the copies of the younger blocks in flight are
            // outstanding (loads complete in order).  NCOPY - 1 per block is exact for waves 1..7
            // and one short for wave 0, which then waits for one more copy than it must.
            // RAGGED: the waves that load A have written it, the others' copies are B's, two of which bring one more.
            constexpr int PER_BLOCK = RAGGED ? NBW : NCOPY - 1;
            if (loads_a) {
            } else if (steady) {
                wait_vmcnt<(NS - 2) * PER_BLOCK>();
            } else {
                const int younger = (kb1 - 1 - kb < NS - 2) ? (kb1 - 1 - kb) : (NS - 2);
                if (NS >= 4 && younger >= 2)
                    wait_vmcnt<2 * PER_BLOCK>();
                else if (NS >= 3 && younger >= 1)
                    wait_vmcnt<PER_BLOCK>();
                else
                    wait_vmcnt<0>();
            }
            __syncthreads();  // everyone's copies of block kb landed; slot_fill is no longer read
            // b_scale of this block, asked for during the last one: waited for here, before any LDS read is in flight (behind
            // a scalar load that is still out every wait for an LDS read is a wait for all of them)
            const float sb_lo = next_lo, sb_hi = next_hi;
            asm volatile("" ::"s"(sb_lo), "s"(sb_hi));
            const uint32_t so = (uint32_t)(slot * S::STAGE);
            // The first column's fragments of B and all of A's, then the second column's; the later ones a column ahead.
            v8i fa[MI], fb[NJ];
            fb[0] = read_frag<RSB>(lds + (addr_b[0] + so));
#pragma unroll
            for (int i = 0; i < MI; ++i)
                fa[i] = read_frag<RSA>(lds + (addr_a[i] + so));
            fb[1] = read_frag<RSB>(lds + (addr_b[1] + so));
            float sa[MI], sc[MI];
#pragma unroll
            for (int i = 0; i < MI; ++i)
                sa[i] = *LDS_PTR(float, lds + so + addr_s + 64 * i);

            // MFMA number t multiplies patch (t % MI, t / MI).  Patches are folded LAG MFMAs behind their own, in the order that
            // stands here (the next MFMA's operand passes through the fold's empty asm statement).  The wave's copy instructions
            // of block kb + NS - 1 ride on the first MFMAs.
            constexpr int T = MI * NJ, PER_MFMA = (NCOPY + T - 1) / T;
            // two patch rows: six behind (128x192: 300 x 12288 x 2048 17.16 -> 17.02 us, four behind 17.05)
            constexpr int LAG = MI < 4 ? 6 : MI;
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
                if (RAGGED) {
                    if (t == 1) {
                        if (loads_a && A_EARLY)
                            next_a();
                        if (!loads_a && more)
                            copy_all(slot_fill, kb + NS - 1);
                    }
                } else if (more) {
#pragma unroll
                    for (int q = t * PER_MFMA; q < (t + 1) * PER_MFMA; ++q)
                        if (q < NCOPY)
                            copy_step(slot_fill, kb + NS - 1, q);
                }
                if (t == T - 1) {
                    // the next block's b_scale, behind this block's last LDS read: its trip to the L2 (a block's values share
                    // no cache line with the next one's unless N is small) is covered by the folds and the barrier
                    int next = kb + 1 < kb1 ? kb + 1 : kb;
                    asm volatile("" : "+s"(next));
                    next_lo = b_scale[next * sn + nb_lo];
                    next_hi = b_scale[next * sn + nb_hi];
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int t = T - LAG; t < T; ++t) {
                fold(t);
                asm volatile("" : "+v"(acc[t % MI][t / MI]));
            }
            if (!A_EARLY)
                next_a();

            slot_fill = slot;
            slot = (slot + 1 == NS) ? 0 : slot + 1;
        };
        int kb = kb0;
        using Set0 = std::integral_constant<int, 0>;
        if constexpr (RAGGED) {
            // a loop for either kind of wave: with the loads of A in a branch of a common one, the compiler has to expect that
            // an earlier block's were not followed by any, and waits for all of them
            auto blocks = [&](auto loads_tag) __attribute__((always_inline)) {
                if constexpr (decltype(loads_tag)::value) {  // A: block 0 into its slot, the next ones on their way
#pragma unroll
                    for (int p = 0; p < SETS; ++p)
                        if (kb0 + p < kb1)
                            load_a(set_a[p], kb0 + p);
                    write_a(std::false_type{}, set_a[0], 0, kb0);
                    if (kb0 + SETS < kb1)
                        load_a(set_a[0], kb0 + SETS);
                }
                auto round = [&](auto more_tag, int at) __attribute__((always_inline)) {  // the sets are numbered at compile time
                    constexpr bool steady = decltype(more_tag)::value;
                    k_block(more_tag, loads_tag, Set0{}, at);
                    if (steady || at + 1 < kb1)
                        k_block(more_tag, loads_tag, std::integral_constant<int, 1>{}, at + 1);
                    if (SETS == 3 && (steady || at + 2 < kb1))
                        k_block(more_tag, loads_tag, std::integral_constant<int, SETS - 1>{}, at + 2);
                };
                static_assert(SETS == 2 || SETS == 3, "unrolled above");
                for (; kb + SETS - 1 + LEAD < kb1; kb += SETS)
                    round(std::true_type{}, kb);
                for (; kb < kb1; kb += SETS)
                    round(std::false_type{}, kb);
            };
            if (loads_a)
                blocks(std::true_type{});
            else
                blocks(std::false_type{});
        } else {
            for (; kb + NS - 1 < kb1; ++kb)
                k_block(std::true_type{}, std::false_type{}, Set0{}, kb);
            for (; kb < kb1; ++kb)
                k_block(std::false_type{}, std::false_type{}, Set0{}, kb);
        }
    }

    // ---- K splits added inside the kernel (mailbox != nullptr).  grid.x is a multiple of 8, so the
    // workgroups of one tile (same blockIdx.x) have linear ids that agree modulo 8 and share an XCD: what
    // they store and load meets in that XCD's L2.  The mailbox holds zeros between launches.  A wave of every
    // split but the last stores its accumulators there in register order (1 KiB per instruction) with
    // every +0.0 replaced by -0.0, so that no word it writes is zero, and is done.  The waves of the last
    // split -- the workgroup with the highest id of its tile, dispatched after the others -- load the other
    // splits' patches past their L1 until no word is zero, add them in split order, their own registers last (the
    // arithmetic of splitk_reduce_kernel: adding -0.0 changes nothing), the workgroup leaves through the bf16
    // epilogue, and zeros go back into the mailbox: behind it where all waves write C (in front of it, its first barrier
    // would wait until they are acknowledged), else beside it.  A wave that has polled for a second gives up and
    // writes NaN.
    bool as_partial = SPLIT;
    constexpr int PATCHES = NCW * MI * NJ;  // 16x16 patches of a tile: 1 KiB of fp32 each
    const int senders = (int)gridDim.y - 1;
    const size_t first = ((size_t)pid * senders * PATCHES + (size_t)(wave & (NCW - 1)) * (MI * NJ)) * 64;  // in 16-byte units
    constexpr uint32_t SUMS_OFF = BM * (BN * 2 + 16);  // behind the tile's bf16 rows (below)
    static_assert(!AHEAD || SUMS_OFF + 4 * (MI * NJ / 2) * 1024 <= S::LDS_BYTES, "sums behind the rows");
    const uint32_t mail_span = (uint32_t)senders * PATCHES * 1024u;
    auto mail_at = [&](int z, int patch) __attribute__((always_inline)) {
        return (uint32_t)((z * PATCHES + patch) * 64 + lane) * 16u;
    };
    if constexpr (SPLIT) {
        if (mailbox != nullptr) {
            as_partial = false;
            if ((int)blockIdx.y < senders) {
                if (compute) {
                    v4i* mine = reinterpret_cast<v4i*>(mailbox) + first + (size_t)blockIdx.y * PATCHES * 64 + lane;
#pragma unroll
                    for (int i = 0; i < MI; ++i)
#pragma unroll
                        for (int j = 0; j < NJ; ++j) {
                            v4i bits = __builtin_bit_cast(v4i, acc[i][j]);
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                bits[e] = bits[e] == 0 ? (int)0x80000000 : bits[e];
                            mine[(i * NJ + j) * 64] = bits;
                        }
                }
                return;
            }
            // Who gathers.  The hand-over is bound by what one workgroup keeps in flight to the L2: where four waves multiply,
            // the other four, idle since their last copy, take the second half of the patches of one of them each, hand
            // the sums over through the LDS (no wave needs a fragment from it behind the last block's barrier, nor the
            // scales) and put the zeros back while C is written.  By the four that multiply / by all eight: 64x64 tiles
            // 64 x 1536 x 7168 in eight 9.19 / 8.29 us, 96 x 576 x 7168 in seven 8.16 / 7.40, 48 x 3136 x 1664 in four 5.53 /
            // 5.09, 304 x 1536 x 7168 in two 14.39 / 14.16; 128x128 2464 x 512 x 7168 in three 19.35 / 18.85, 384 x 4608 x 7168 in two
            // 19.67 / 19.41.
            // PG patches at a time (all of them when there are at most eight: one trip to the L2 for everything that
            // is there), ZB splits at a time.  Two patches a wave: three splits or four alike, two 1.3 % and seven 1.2 %
            // behind (60 and 44 shapes).
            constexpr int MINE = AHEAD ? MI * NJ / 2 : MI * NJ;  // patches that a wave gathers
            constexpr int PG = MINE <= 8 ? MINE : 4, ZB = MINE <= 4 ? 3 : 2;
            static_assert(MINE % PG == 0, "whole groups of patches");
            const int part = AHEAD && !compute ? MINE : 0;  // its first patch
            const __amdgpu_buffer_rsrc_t rp = make_rsrc(reinterpret_cast<const v4i*>(mailbox) + first, mail_span);
            const unsigned long long t_first = __builtin_amdgcn_s_memrealtime();
            bool gave_up = false;
#pragma unroll
            for (int pg = 0; pg < MINE; pg += PG) {
                v4f sum[PG];
                auto gather = [&](auto count, int z0) __attribute__((always_inline)) {  // splits z0 .. z0 + ZC - 1
                    constexpr int ZC = decltype(count)::value;
                    v4i v[ZC][PG];
                    for (;;) {
                        asm volatile("" ::: "memory");  // the loads belong to this round of the loop
#pragma unroll
                        for (int z = 0; z < ZC; ++z)
#pragma unroll
                            for (int g = 0; g < PG; ++g)
                                v[z][g] = __builtin_amdgcn_raw_buffer_load_b128(rp, mail_at(z0 + z, part + pg + g), 0, 16);
                        bool missing = false;
#pragma unroll
                        for (int z = 0; z < ZC; ++z)
#pragma unroll
                            for (int g = 0; g < PG; ++g)
                                missing = missing | (v[z][g][0] == 0) | (v[z][g][1] == 0) | (v[z][g][2] == 0) |
                                          (v[z][g][3] == 0);
                        if (__builtin_amdgcn_ballot_w64(missing) == 0)
                            break;
                        if (__builtin_amdgcn_s_memrealtime() - t_first > 100000000ull) {  // one second at 100 MHz
                            gave_up = true;
                            break;
                        }
                    }
#pragma unroll
                    for (int z = 0; z < ZC; ++z)
#pragma unroll
                        for (int g = 0; g < PG; ++g) {
                            const v4f f = __builtin_bit_cast(v4f, v[z][g]);
                            sum[g] = z0 + z == 0 ? f : sum[g] + f;
                        }
                };
                int z0 = 0;
                for (; z0 + ZB <= senders; z0 += ZB)
                    gather(std::integral_constant<int, ZB>{}, z0);
                auto rest = [&](auto count) __attribute__((always_inline)) {
                    constexpr int ZC = decltype(count)::value;
                    if (ZB > ZC && senders - z0 == ZC)
                        gather(count, z0);
                };
                rest(std::integral_constant<int, 2>{});
                rest(std::integral_constant<int, 1>{});
#pragma unroll
                for (int g = 0; g < PG; ++g) {
                    if (gave_up)
                        sum[g] = (v4f){__builtin_nanf(""), __builtin_nanf(""), __builtin_nanf(""), __builtin_nanf("")};
                    if (AHEAD && !compute)
                        *LDS_PTR(v4f, lds + SUMS_OFF + (uint32_t)(((wave & 3) * MINE + pg + g) * 1024 + lane * 16)) = sum[g];
                    else
                        acc[(pg + g) / NJ][(pg + g) % NJ] = sum[g] + acc[(pg + g) / NJ][(pg + g) % NJ];
                }
            }
            if (AHEAD) {
                __syncthreads();
                if (compute) {
#pragma unroll
                    for (int g = 0; g < MINE; ++g) {
                        v4f& own = acc[(MINE + g) / NJ][(MINE + g) % NJ];
                        own = *LDS_PTR(v4f, lds + SUMS_OFF + (uint32_t)((wave * MINE + g) * 1024 + lane * 16)) + own;
                    }
                }
            }
        }
    }

    // ---- epilogue.  A lane owns row m = .. + (lane & 15) and, per patch, a run of 4 columns, 4 * (lane >> 4)
    // of the patch: stored straight from the registers that would be 8- or 16-byte pieces of 16 different
    // rows per instruction.  The tile therefore goes through the (now idle) LDS ring, row-major with a
    // padded row stride that keeps the writes conflict free, and leaves as 16 bytes per lane
    // along whole rows of the tile.  A tile larger than the ring is written in two halves.
    // PARTIAL = fp32 into this split's partial tile (the reduction kernel follows), else bf16 into c.
    auto zeros = [&]() __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t rp = make_rsrc(reinterpret_cast<const v4i*>(mailbox) + first, mail_span);
        for (int z = 0; z < senders; ++z)
#pragma unroll
            for (int patch = 0; patch < MI * NJ; ++patch)
                __builtin_amdgcn_raw_buffer_store_b128((v4i){0, 0, 0, 0}, rp, mail_at(z, patch), 0, 0);
    };
    auto write_tile = [&](auto partial_tag) __attribute__((always_inline)) {
        constexpr bool PARTIAL = decltype(partial_tag)::value;
        constexpr int ESZ = PARTIAL ? 4 : 2;
        constexpr int CROW = BN * ESZ + 16;                 // LDS bytes per tile row
        constexpr int HALVES = (BM * CROW <= S::LDS_BYTES) ? 1 : 2;
        constexpr int HROWS = BM / HALVES;
        static_assert(HROWS * CROW <= S::LDS_BYTES, "half a tile must fit the ring");
        static_assert(HROWS % 16 == 0, "a patch lies in one half");
        constexpr int CPR = BN * ESZ / 16;                 // 16-byte chunks per tile row
        constexpr int CHUNKS = HROWS * CPR;
        constexpr bool GATHERED = AHEAD && SPLIT && !PARTIAL;  // a barrier has passed since the ring was read
        constexpr int STORERS = GATHERED ? 64 * NCW : NTHREADS;
        static_assert(!GATHERED || HALVES == 1, "one pass");
#pragma unroll
        for (int h = 0; h < HALVES; ++h) {
            if (!GATHERED)
                __syncthreads();  // nobody reads the ring (or the previous half) any more
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                const int prow = wm * TM + 16 * i;  // first tile row of the patch
                if (compute && prow / HROWS == h) {
                    const uint32_t rbase = (uint32_t)((prow - h * HROWS + (lane & 15)) * CROW);
#pragma unroll
                    for (int j = 0; j < NJ; ++j) {
                        const int col = wn * TN + 16 * j + 4 * (lane >> 4);
                        const v4f v = acc[i][j];
                        if (PARTIAL) {
                            *LDS_PTR(v4f, lds + rbase + col * 4) = v;
                        } else {
                            v2i pk = {(int)pack_bf16x2(v[0], v[1]), (int)pack_bf16x2(v[2], v[3])};
                            *LDS_PTR(v2i, lds + rbase + col * 2) = pk;
                        }
                    }
                }
            }
            if (GATHERED) {
                if (!compute) {
                    zeros();
                    asm volatile("s_barrier" ::: "memory");
                    return;
                }
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // the rows are in the LDS
            } else {
                __syncthreads();
            }
#pragma unroll
            for (int it = 0; it < (CHUNKS + STORERS - 1) / STORERS; ++it) {
                const int idx = it * STORERS + (int)threadIdx.x;
                const int row = idx / CPR, ch = idx - row * CPR;
                const int mrow = m0 + h * HROWS + row;
                const int ncol = n0 + ch * (16 / ESZ);
                if (idx < CHUNKS && mrow < M && ncol < N) {
                    const size_t o = (size_t)mrow * N + ncol;
                    if (PARTIAL) {
                        const v4f v = *LDS_PTR(v4f, lds + row * CROW + ch * 16);
                        *reinterpret_cast<v4f*>(partial + (size_t)blockIdx.y * M * N + o) = v;
                    } else {
                        *reinterpret_cast<v4i*>(c + o) = *LDS_PTR(v4i, lds + row * CROW + ch * 16);
                    }
                }
            }
        }
    };
    if constexpr (SPLIT) {
        if (as_partial) {
            write_tile(std::true_type{});
        } else {
            write_tile(std::false_type{});
            if (!AHEAD)
                zeros();
        }
    } else {
        write_tile(std::false_type{});
    }
}

// Which tile: consecutive workgroup ids land on different XCDs (id % 8), so each XCD gets a contiguous run of tile
// numbers.  -1: grid.x is rounded up to a multiple of 8 when the K splits of a tile have to share an XCD.
__device__ __forceinline__ int tile_number(int T)
{
    const int pid = blockIdx.x;
    if (pid >= T)
        return -1;
    const int xcd = pid & 7, q8 = T >> 3, r8 = T & 7;
    return xcd * q8 + (xcd < r8 ? xcd : r8) + (pid >> 3);
}

// ... walked in groups of group_m rows so that the tiles an XCD works on together share A and B panels in its L2 (the host
// picks group_m so that an XCD's co-resident tiles form a block that is about square in bytes).
template <int BM, int BN>
__device__ __forceinline__ void tile_origin(int logical, int tiles_m, int tiles_n, int group_m, int& m0, int& n0)
{
    const int per_group = group_m * tiles_n;
    const int group = logical / per_group;
    const int first_m = group * group_m;
    const int gsz = (tiles_m - first_m < group_m) ? (tiles_m - first_m) : group_m;
    const int in_group = logical - group * per_group;
    m0 = (first_m + in_group % gsz) * BM;
    n0 = (in_group / gsz) * BN;
}

template <int BM, int BN, int WM, int WN, int NS, bool SPLIT, bool RAGGED>
__global__ void __launch_bounds__(NTHREADS)
tile_gemm_kernel(const uint8_t* __restrict__ a, const uint8_t* __restrict__ b,
                 const float* __restrict__ a_scale, const float* __restrict__ b_scale,
                 uint16_t* __restrict__ c, float* __restrict__ partial, float* mailbox,
                 int M, int lda, int N, int K, int tiles_m, int tiles_n, int kb_per_split, int group_m)
{
    const int logical = tile_number(tiles_m * tiles_n);
    if (logical < 0)
        return;
    int m0, n0;
    tile_origin<BM, BN>(logical, tiles_m, tiles_n, group_m, m0, n0);
    tile_body<BM, BN, WM, WN, NS, SPLIT, RAGGED>(a, b, a_scale, b_scale, c, partial, mailbox, M, lda, N, K, m0, n0,
                                                 blockIdx.x, kb_per_split);
}

// The problems of `tab` (same N and K, own M), a tile per workgroup and K split, tiles numbered one problem after the other.
// What small grouped launches of tall groups are bound by is latency and idle CUs: the persistent kernels want A's rows on the
// grid (a copy launch, 3 - 6 us), start in tiles of 128 rows and more, and don't split K, for which the groups used to run
// one by one.  Here A comes as it lies, in tiles of 64 or 128 rows, K split where the tiles are few; the look-up is one trip to
// the kernel arguments.  22 groups of 67 - 172 rows, 576 x 7168, 64.9 -> 53.7 us; nine of 2637 rows in all, 48.3 -> 36.8; three of 705,
// 448 x 5632, 27.0 -> 14.0; eight of 68 - 139, 832 x 384, 8.5 -> 4.5.  In more than a few rounds the persistent kernels, which
// copy the next tile's blocks while one is stored, are ahead again (seven groups of 4048 rows, 4608 x 7168, 170 against 190).
template <int BM, int BN, int WM, int WN, int NS, bool SPLIT, bool RAGGED>
__global__ void __launch_bounds__(NTHREADS)
tile_gemm_each_kernel(const GroupTable tab, float* mailbox, int N, int K, int tiles_n, int kb_per_split)
{
    int logical = tile_number(tab.tile_start[tab.groups]);
    if (logical < 0)
        return;
    // tile_start ascends: how many problems end at or before this tile, looked up by a lane each
    static_assert(GroupTable::MAX_GROUPS == 64, "a lane for every problem");
    const int lane = threadIdx.x & 63;
    const int g = __builtin_popcountll(__builtin_amdgcn_ballot_w64(lane < tab.groups && tab.tile_start[lane + 1] <= logical));
    logical -= tab.tile_start[g];
    const int M = tab.m[g];
    int m0, n0;
    tile_origin<BM, BN>(logical, (M + BM - 1) / BM, tiles_n, GROUP_M, m0, n0);
    tile_body<BM, BN, WM, WN, NS, SPLIT, RAGGED>(tab.a[g], tab.b[g], tab.a_scale[g], tab.b_scale[g], tab.c[g], nullptr,
                                                 mailbox, M, tab.lda[g], N, K, m0, n0, blockIdx.x, kb_per_split);
}

// sum of the K-split partials in split order, then bf16
__global__ void __launch_bounds__(256) splitk_reduce_kernel(const float* __restrict__ partial,
                                                            uint16_t* __restrict__ c, size_t mn,
                                                            int ksplit)
{
    size_t i4 = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (i4 >= mn)
        return;
    // four splits' loads in flight at a time (one after the other, each add waits a trip to the L2: 0.4 us per
    // split of a small problem); the sum keeps its order
    v4f s = *reinterpret_cast<const v4f*>(partial + i4);
    int z = 1;
    for (; z + 3 < ksplit; z += 4) {
        v4f p[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            p[u] = *reinterpret_cast<const v4f*>(partial + (size_t)(z + u) * mn + i4);
#pragma unroll
        for (int u = 0; u < 4; ++u)
            s += p[u];
    }
    for (; z < ksplit; ++z) {
        v4f p = *reinterpret_cast<const v4f*>(partial + (size_t)z * mn + i4);
        s += p;
    }
    uint2 pk;
    pk.x = pack_bf16x2(s[0], s[1]);
    pk.y = pack_bf16x2(s[2], s[3]);
    *reinterpret_cast<uint2*>(c + i4) = pk;
}

// Tile rows per locality group.  The kernel gives XCD x (workgroup id % 8) a contiguous run of the
// tile order, which walks the tile grid in groups of group_m rows, column by column.  The tiles an
// XCD works on together (its first 32: one per CU) then touch some rows of A and some of B; the
// group size that makes the eight XCDs touch the fewest bytes is found by walking the order, and
// remembered for the last few grids.
int choose_group_m(int tiles_m, int tiles_n, int bm, int bn)
{
    struct Entry { int tm, tn, bm, bn, g; };
    static thread_local Entry cache[8] = {};
    static thread_local int next = 0;
    for (const Entry& e : cache)
        if (e.tm == tiles_m && e.tn == tiles_n && e.bm == bm && e.bn == bn)
            return e.g;
    const int T = tiles_m * tiles_n;
    int best_g = GROUP_M;
    long best_cost = -1;
    for (int gm = 1; gm <= GROUP_M; ++gm) {
        long cost = 0;
        for (int xcd = 0; xcd < 8; ++xcd) {
            const int q8 = T >> 3, r8 = T & 7;
            const int start = xcd * q8 + (xcd < r8 ? xcd : r8);
            int len = q8 + (xcd < r8 ? 1 : 0);
            len = len < 32 ? len : 32;
            unsigned long long rows[4] = {0, 0, 0, 0}, cols[4] = {0, 0, 0, 0};  // up to 256 tile rows / columns tracked
            int nrows = 0, ncols = 0;
            for (int t = start; t < start + len; ++t) {
                const int per_group = gm * tiles_n, group = t / per_group, first_m = group * gm;
                const int gsz = tiles_m - first_m < gm ? tiles_m - first_m : gm;
                const int in_group = t - group * per_group;
                const int r = (first_m + in_group % gsz) & 255, c = (in_group / gsz) & 255;
                if (!(rows[r >> 6] >> (r & 63) & 1)) {
                    rows[r >> 6] |= 1ull << (r & 63);
                    ++nrows;
                }
                if (!(cols[c >> 6] >> (c & 63) & 1)) {
                    cols[c >> 6] |= 1ull << (c & 63);
                    ++ncols;
                }
            }
            cost += (long)nrows * bm + (long)ncols * bn;
        }
        if (best_cost < 0 || cost < best_cost) {
            best_cost = cost;
            best_g = gm;
        }
    }
    cache[next] = Entry{tiles_m, tiles_n, bm, bn, best_g};
    next = (next + 1) & 7;
    return best_g;
}

// the tile shapes that have a form for row counts off the 16-byte grid
constexpr bool tile_takes_ragged_rows(int bm, int ns) { return bm <= 128 && ns >= 3; }

template <int BM, int BN, int WM, int WN, int NS, bool SPLIT, bool RAGGED>
hipError_t launch_typed(const GemmArgs& g, int ksplit, float* partial, float* mailbox, hipStream_t s)
{
    using S = TileShape<BM, BN, WM, WN, NS>;
    constexpr int LDS_TOTAL = S::LDS_BYTES;
    const int tiles_m = (g.m + BM - 1) / BM, tiles_n = (g.n + BN - 1) / BN;
    const int nkb = g.k / KBLOCK;
    const int kb_per_split = (nkb + ksplit - 1) / ksplit;
    const int tiles = tiles_m * tiles_n;
    const int group_m = choose_group_m(tiles_m, tiles_n, BM, BN);
    // in-kernel reduction: the other splits' patches of every tile fit the mailbox
    if (SPLIT && mailbox && (size_t)tiles * (ksplit - 1) * BM * BN * 4 > SPLIT_MAILBOX_BYTES)
        return hipErrorInvalidValue;
    const dim3 grid(SPLIT && mailbox ? (tiles + 7) & ~7 : tiles, SPLIT ? ksplit : 1);
    constexpr auto kern = tile_gemm_kernel<BM, BN, WM, WN, NS, SPLIT, RAGGED>;
    FP8GEMM_ALLOW_LDS(kern, LDS_TOTAL);
    launch_kernel(kern, grid, dim3(NTHREADS), LDS_TOTAL, s, g.a, g.b, g.a_scale, g.b_scale, g.c, partial,
                       SPLIT ? mailbox : nullptr, g.m, leading_dim(g), g.n, g.k, tiles_m, tiles_n, kb_per_split, group_m);
    return hipGetLastError();
}

template <int BM, int BN, int WM, int WN, int NS>
hipError_t launch_variant(const GemmArgs& g, int ksplit, float* partial, float* mailbox, hipStream_t s)
{
    if (leading_dim(g) % 16 == 0)
        return ksplit > 1 ? launch_typed<BM, BN, WM, WN, NS, true, false>(g, ksplit, partial, mailbox, s)
                          : launch_typed<BM, BN, WM, WN, NS, false, false>(g, ksplit, partial, mailbox, s);
    if constexpr (tile_takes_ragged_rows(BM, NS)) {
        if (leading_dim(g) == g.m && g.m >= 16)
            return ksplit > 1 ? launch_typed<BM, BN, WM, WN, NS, true, true>(g, ksplit, partial, mailbox, s)
                              : launch_typed<BM, BN, WM, WN, NS, false, true>(g, ksplit, partial, mailbox, s);
    }
    return hipErrorInvalidValue;
}

// Whether 128x128 tiles are multiplied by four waves that read ahead, or by eight.  us by eight / by four:
//   K splits: four for long chains.  They start later (a K block more is read before the first MFMA) and, with rows of B that
//   share lines of 128 bytes with their neighbours' (N no multiple of 128), gain nothing per K block, which the copies
//   bound then.  Added in the kernel, rows on the grid, N a multiple of 128, 8 ... 15 K blocks to a split: 192 x 7168 x 2048 in
//   two 11.03 / 10.84, 256 x 7168 x 2048 11.17 / 10.89, 144 x 7168 x 2304 11.52 / 11.26 (18 of 20 ahead, 1.5 % on average);
//   other N 1504 x 832 x 2816 in two 12.55 / 12.94, 3728 x 288 x 2560 12.19 / 12.53, from 16 blocks on 2000 ... 3000 x 576
//   x 7168 1 - 3 % ahead.  Rows off the grid, where two of the copy waves bring A by way of registers, N a multiple of 128:
//   334 x 4608 x 7168 in two of 28 blocks 24.00 / 22.76, 2340 x 512 x 7168 in three 20.82 / 20.08, 397 x 1536 x 7168 in five of
//   twelve (reduction kernel) 18.25 / 17.81 (all of 150 workgroups and more; fewer than 128: as before, eight), 129 x 7168 x 2304 in two of nine 13.08 / 13.37; other N 1621 x 576 x 7168 21.03 /
//   21.42, 3065 x 576 x 7168 25.07 / 24.76 (30 shapes level).  With the reduction kernel behind them and rows on the grid,
//   four: 512 x 1024 x 7168 in five 14.77 / 13.99.
//   Unsplit, four: 500 x 4608 x 2048 (off the grid) 13.8 / 12.9 -- but for a single K block, where there is nothing to read
//   ahead of: 5104 x 720 x 128 4.41 / 4.72, 413 x 3824 x 128 4.37 / 4.47; two: 5104 x 720 x 256 5.19 / 5.14.
bool four_waves(const GemmArgs& g, int ksplit, bool fused)
{
    const int kb_per_split = (g.k / KBLOCK + ksplit - 1) / ksplit;
    const bool whole_lines = g.n % 128 == 0;
    if (ksplit == 1)
        return kb_per_split > 1;
    if (leading_dim(g) % 16 != 0) {
        const long tiles = (long)((g.m + 127) / 128) * ((g.n + 127) / 128);
        return whole_lines && kb_per_split >= 12 && tiles * ksplit >= 128;
    }
    return kb_per_split >= (!fused ? 2 : whole_lines ? 8 : 16);
}

}  // namespace

bool tile_supports(const GemmArgs& g)
{
    // 16-byte copies need every k-row of a, b and a_scale to start 16-byte aligned; rows of a
    // and a_scale beyond m, up to the leading dimension, are read (and must be finite: zeros)
    return leading_dim(g) % 16 == 0 && leading_dim(g) >= g.m && g.n % 16 == 0 &&
           (reinterpret_cast<uintptr_t>(g.a) % 16 == 0) &&
           (reinterpret_cast<uintptr_t>(g.b) % 16 == 0) &&
           (reinterpret_cast<uintptr_t>(g.a_scale) % 16 == 0) &&
           (reinterpret_cast<uintptr_t>(g.c) % 16 == 0);
}

bool tile_ragged_supports(const GemmArgs& g, int variant)
{
    return (variant == TILE_64x64 || variant == TILE_128x128 || variant == TILE_128x192) && g.m >= 16 && g.m % 16 != 0 &&
           leading_dim(g) == g.m && g.n % 16 == 0 && (reinterpret_cast<uintptr_t>(g.a) % 16 == 0) &&
           (reinterpret_cast<uintptr_t>(g.b) % 16 == 0) && (reinterpret_cast<uintptr_t>(g.a_scale) % 16 == 0) &&
           (reinterpret_cast<uintptr_t>(g.c) % 16 == 0);
}

const char* tile_variant_name(int variant)
{
    switch (variant) {
    case TILE_256x128: return "tile256x128";
    case TILE_128x128: return "tile128x128";
    case TILE_256x192: return "tile256x192";
    case TILE_128x192: return "tile128x192";
    case TILE_64x64: return "tile64x64";
    case TILE_256x192_W4: return "tile256x192w4";
    case TILE_256x256: return "tile256x256";
    case TILE_128x256: return "tile128x256";
    default: return "tile?";
    }
}

void tile_variant_dims(int variant, int* bm, int* bn)
{
    switch (variant) {
    case TILE_256x128: *bm = 256; *bn = 128; break;
    case TILE_256x192:
    case TILE_256x192_W4: *bm = 256; *bn = 192; break;
    case TILE_128x192: *bm = 128; *bn = 192; break;
    case TILE_64x64: *bm = 64; *bn = 64; break;
    case TILE_256x256: *bm = 256; *bn = 256; break;
    case TILE_128x256: *bm = 128; *bn = 256; break;
    default: *bm = 128; *bn = 128; break;
    }
}

size_t tile_mailbox_bytes(const GemmArgs& g, int variant, int ksplit)
{
    int bm, bn;
    tile_variant_dims(variant, &bm, &bn);
    const size_t tiles = (size_t)((g.m + bm - 1) / bm) * ((g.n + bn - 1) / bn);
    return ksplit > 1 ? tiles * (size_t)(ksplit - 1) * bm * bn * 4 : 0;
}

hipError_t launch_tile(const GemmArgs& g, int variant, int ksplit, float* partial, float* mailbox,
                       hipStream_t s)
{
    switch (variant) {
    case TILE_256x192: return launch_variant<256, 192, 4, 2, 2>(g, ksplit, partial, mailbox, s);
    case TILE_256x128: return launch_variant<256, 128, 4, 2, 3>(g, ksplit, partial, mailbox, s);
    case TILE_128x192: return launch_variant<128, 192, 4, 2, 3>(g, ksplit, partial, mailbox, s);
    case TILE_128x128:
        return four_waves(g, ksplit, mailbox != nullptr) ? launch_variant<128, 128, 2, 2, 4>(g, ksplit, partial, mailbox, s)
                                                         : launch_variant<128, 128, 2, 4, 4>(g, ksplit, partial, mailbox, s);
    case TILE_64x64: return launch_variant<64, 64, 2, 2, 4>(g, ksplit, partial, mailbox, s);
    default: return hipErrorInvalidValue;
    }
}

namespace {

template <int BM, int BN, int WM, int WN, int NS, bool SPLIT, bool RAGGED>
hipError_t launch_each_typed(GroupTable& tab, int n, int k, int ksplit, float* mailbox, hipStream_t s)
{
    using S = TileShape<BM, BN, WM, WN, NS>;
    const int tiles_n = (n + BN - 1) / BN, nkb = k / KBLOCK;
    tab.tile_start[0] = 0;
    for (int g = 0; g < tab.groups; ++g)
        tab.tile_start[g + 1] = tab.tile_start[g] + ((tab.m[g] + BM - 1) / BM) * tiles_n;
    const int tiles = tab.tile_start[tab.groups];
    if (SPLIT && (!mailbox || (size_t)tiles * (ksplit - 1) * BM * BN * 4 > SPLIT_MAILBOX_BYTES))
        return hipErrorInvalidValue;
    constexpr auto kern = tile_gemm_each_kernel<BM, BN, WM, WN, NS, SPLIT, RAGGED>;
    FP8GEMM_ALLOW_LDS(kern, S::LDS_BYTES);
    launch_kernel(kern, dim3(SPLIT ? (tiles + 7) & ~7 : tiles, ksplit), dim3(NTHREADS), S::LDS_BYTES, s, tab,
                  SPLIT ? mailbox : nullptr, n, k, tiles_n, (nkb + ksplit - 1) / ksplit);
    return hipGetLastError();
}

template <int BM, int BN, int WM, int WN, int NS>
hipError_t launch_each_variant(GroupTable& tab, bool ragged, int n, int k, int ksplit, float* mailbox, hipStream_t s)
{
    if (ragged)
        return ksplit > 1 ? launch_each_typed<BM, BN, WM, WN, NS, true, true>(tab, n, k, ksplit, mailbox, s)
                          : launch_each_typed<BM, BN, WM, WN, NS, false, true>(tab, n, k, 1, nullptr, s);
    return ksplit > 1 ? launch_each_typed<BM, BN, WM, WN, NS, true, false>(tab, n, k, ksplit, mailbox, s)
                      : launch_each_typed<BM, BN, WM, WN, NS, false, false>(tab, n, k, 1, nullptr, s);
}

}  // namespace

// every problem as a single one, for the form that takes it; one off the 16-row grid takes all to the form for such
bool tile_each_supports(const GroupTable& tab, int n, int k, int variant, bool* ragged)
{
    if ((variant != TILE_64x64 && variant != TILE_128x128) || tab.groups < 1 || tab.groups > GroupTable::MAX_GROUPS)
        return false;
    *ragged = false;
    for (int g = 0; g < tab.groups; ++g)
        *ragged = *ragged || tab.m[g] % 16 != 0;
    for (int g = 0; g < tab.groups; ++g) {
        GemmArgs ga{tab.a[g], tab.b[g], tab.a_scale[g], tab.b_scale[g], tab.c[g], tab.m[g], n, k, tab.lda[g]};
        if (tab.m[g] < 16 || tab.lda[g] != tab.m[g])
            return false;
        ga.m = ga.lda = tab.m[g] & ~15;  // the addresses and n
        if (!tile_supports(ga))
            return false;
    }
    return true;
}

hipError_t launch_tile_each(GroupTable& tab, int n, int k, int variant, int ksplit, float* mailbox, hipStream_t s)
{
    bool ragged;
    const int nkb = k / KBLOCK;
    if (ksplit < 1 || (ksplit - 1) * ((nkb + ksplit - 1) / ksplit) >= nkb || !tile_each_supports(tab, n, k, variant, &ragged))
        return hipErrorInvalidValue;
    return variant == TILE_64x64 ? launch_each_variant<64, 64, 2, 2, 4>(tab, ragged, n, k, ksplit, mailbox, s)
                                 : launch_each_variant<128, 128, 2, 2, 4>(tab, ragged, n, k, ksplit, mailbox, s);
}

hipError_t launch_splitk_reduce(const GemmArgs& g, int ksplit, const float* partial, hipStream_t s)
{
    size_t mn = (size_t)g.m * g.n;
    unsigned blocks = (unsigned)((mn / 4 + 255) / 256);
    launch_kernel(splitk_reduce_kernel, dim3(blocks), dim3(256), 0, s, partial, g.c, mn, ksplit);
    return hipGetLastError();
}

}  // namespace fp8gemm
