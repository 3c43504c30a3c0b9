// Decode kernel for tiny M (M <= 64) and small weights: strips of 64 columns.  Data path, mailbox and arithmetic are those
// of the wide strips (k_decode.hip); the reference has no kernel for this regime (/root/reference/mn_small.hip:16,121-125).
//
// What bounds such a launch is neither bytes nor MFMAs but a chain: the first copy's trip, the K blocks one behind the
// other, the hand-over of the K splits.  128-column strips of N = 576 are five, and in eight splits 40 workgroups:
// time stamps (24 x 576 x 7168, 7 blocks each, us since the first workgroup's start) have the last K block done at 3.9 and C
// stored at 7.0, 2.0 of it in four turns of the K loop, bound by the LDS reads of eight waves that each read all of A,
// and 3.1 in the hand-over, whose 84 KB of partial sums one CU takes in at 64 bytes per clock and then overwrites with zeros
// at the same rate, in front of C.  Against that:
//   * Strips of 64 columns: twice the workgroups, and half the partial sums for the one that adds them.
//   * K blocks are taken in pairs, one barrier for both.  Waves 0 - 3 multiply the first block of a pair and waves 4 - 7 the
//     second, each wave 16 columns: half the LDS reads of A.  The two sums of a column meet in the LDS behind the loop.
//   * The last split asks for all splits' patches together (up to eight) and the zeros go back behind C.
//   * A single row (ROW) is not spread into padded rows: its k-values lie in the K block's slab as a fragment has
//     them, 8 bytes a read.
// us, 128-column strips (64x64 tiles from 33 rows on) -> this, operands from the Infinity Cache / from HBM: 1 x 512 x 7168
// 6.38 -> 4.52 / 6.96 -> 5.73, 24 x 512 x 7168 7.12 -> 5.15 / 8.31 -> 6.51, 27 x 576 x 7168 8.81 -> 6.21 / 9.38 -> 6.73, 32 x
// 576 x 5888 7.26 -> 5.27 / 8.20 -> 6.22, 1 x 1536 x 7168 6.99 -> 5.63 / 7.27 -> 6.62, 24 x 1536 x 7168 7.90 -> 6.55, 24 x 1536 x
// 1664 4.82 -> 3.90 / 5.66 -> 4.70, 1 x 4096 x 512 3.61 -> 2.99 / 3.77 -> 4.10, 24 x 3072 x 1536 4.58 -> 4.31, 48 x 576 x 4096 6.71 ->
// 5.91 / 7.57 -> 6.75.  Where B is large the memory system decides, and 64 bytes of every k-row come slower than 128: 24 x
// 7168 x 2048 6.61 -> 6.85 / 6.89 -> 8.32, 5 x 4608 x 7168 9.42 -> 11.45 / 9.62 -> 11.81 (decode64_us).  The same pairs of
// blocks with 128-column strips, two columns to a wave: 24 x 7168 x 2048 6.69 -> 6.90, 16 x 7168 x 2048 5.69 -> 6.03; not kept.
#include "tile_common.h"

namespace fp8gemm {

namespace {

constexpr int BN = 64, RSB = 64;  // columns of a strip, LDS bytes of a k-row of B

// how the k-rows of A lie in a stage: padded, copied there row by row (M a multiple of 16); packed as in memory (of 8); padded,
// spread from the packed slab by the threads; packed and read without transposing (M = 1)
enum class Rows { GRID, PACKED, SPREAD, ROW };

// T = 16-row tiles of A
template <int T, Rows FORM>
struct Strip64 {
    static constexpr int RSA = T == 1 ? 16 : T == 2 ? 32 : 64;  // LDS bytes of a k-row of A
    static constexpr int MAT_B = KBLOCK * RSB, MAT_A = KBLOCK * RSA;
    static constexpr int SA_OFF = MAT_B + MAT_A;   // up to 64 a_scale floats
    static constexpr int SB_OFF = SA_OFF + 256;    // b_scale (every wave that brings it writes the same bytes)
    static constexpr int PACK_OFF = SB_OFF + 256;  // SPREAD: the packed slab, and 16 bytes that its last row's reads may run into
    static constexpr int STAGE = FORM == Rows::SPREAD ? (PACK_OFF + MAT_A + 16 + 511) / 512 * 512 : PACK_OFF;
    static constexpr int NS = 8 * STAGE <= 160 * 1024 ? 8 : 6;  // ring stages
    static constexpr int KEEP = (T + 1) / 2;  // row tiles that a wave ends with (of three, waves 4 - 7 one)
    static constexpr int EXCHANGE = 8 * KEEP * 1024;
    static constexpr bool APART = NS * STAGE + EXCHANGE <= 160 * 1024;  // room for the exchange behind the ring
    static constexpr int EXCHANGE_OFF = APART ? NS * STAGE : 0;
    static constexpr int LDS = NS * STAGE + (APART ? EXCHANGE : 0);
    static constexpr int A_WAVES = T > 2 ? 8 : 2 * T;   // waves that bring 1 KiB of A each
    static constexpr int COPIES = T > 2 ? 3 : 2;        // of a wave per stage: B, then A or (T > 2: and) scales
    static_assert(LDS <= 160 * 1024 && EXCHANGE <= NS * STAGE && COPIES * NS < 64, "ring");
};

constexpr unsigned PAST_L1 = 16;  // cache policy of the mailbox loads (sc1): served by the L2
constexpr unsigned long long SPIN_LIMIT = 100000000ull;  // one second of the constant 100 MHz counter (s_memrealtime)

// (the first 14 words of the arguments are in registers when a wave starts: what the copies need comes first)
template <int T, Rows FORM>
__global__ void __launch_bounds__(NTHREADS)
decode64_kernel(const uint8_t* __restrict__ b, const uint8_t* __restrict__ a, int N, int K, int M, int lda, int kb_per_split,
                int strips, const float* __restrict__ a_scale, const float* __restrict__ b_scale, uint16_t* __restrict__ c,
                float* mailbox, int ksplit, int paired)
{
    constexpr bool SPREAD = FORM == Rows::SPREAD, ROW = FORM == Rows::ROW, PACKED = FORM == Rows::PACKED;
    static_assert(!ROW || T == 1, "a single row");
    using S = Strip64<T, FORM>;
    constexpr int NS = S::NS, KEEP = S::KEEP;
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    auto lds = LDS_PTR(uint8_t, smem);
    const uint32_t lds_base = (uint32_t)(uintptr_t)lds;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = wave & 3, par = wave >> 2;  // the wave's 16 columns, and which block of a pair it multiplies

    // Workgroup ids go round the XCDs.  Paired: two strips that share B's 128-byte lines sit on one XCD.
    const int unit = blockIdx.x, split = blockIdx.y;
    const int strip = paired ? 2 * ((unit >> 4) * 8 + (unit & 7)) + ((unit >> 3) & 1) : unit;
    if (strip >= strips)
        return;
    const int n0 = strip * BN;
    const int nkb = K / KBLOCK;
    const int kb0 = split * kb_per_split;
    const int kb1 = (kb0 + kb_per_split < nkb) ? (kb0 + kb_per_split) : nkb;
    const int sn = (N + KBLOCK - 1) / KBLOCK;

    // ---- copies.  B: a wave brings rows 16 * wave + (lane >> 2), chunk position lane & 3, swizzle (r >> 2) & 3.  A: rows of 16, 32
    // or 64 bytes, swizzle 0, (r >> 3) & 1, (r >> 2) & 3; or the K block's slab, 128 * M contiguous bytes
    uint32_t voff_b, voff_a;
    {
        const int cc = (lane & 3) ^ ((lane >> 4) & 3);
        voff_b = n0 + 16 * cc < N ? (uint32_t)((16 * wave + (lane >> 2)) * N + n0 + 16 * cc) : 0x80000000u;
    }
    if (FORM == Rows::GRID) {
        constexpr int CH = S::RSA / 16;
        const int cc = T == 1 ? 0 : T == 2 ? (lane & 1) ^ ((lane >> 4) & 1) : (lane & 3) ^ ((lane >> 4) & 3);
        voff_a = 16 * cc < lda ? (uint32_t)((64 / CH * wave + lane / CH) * lda + 16 * cc) : 0x80000000u;
    } else {
        const int piece = 64 * wave + lane;
        voff_a = 16 * piece < KBLOCK * lda ? (uint32_t)(16 * piece) : 0x80000000u;
    }
    const v4i rsrc_b = make_rsrc_words(b, (uint32_t)N * (uint32_t)K), rsrc_a = make_rsrc_words(a, (uint32_t)lda * (uint32_t)K);
    const bool brings_sa = wave == (T > 2 ? 0 : 4);
    const v4i rsrc_s = brings_sa ? make_rsrc_words(a_scale, (uint32_t)nkb * (uint32_t)lda * 4u)
                                 : make_rsrc_words(b_scale, (uint32_t)nkb * (uint32_t)sn * 4u);
    const uint32_t voff_s = brings_sa ? (lane < lda ? (uint32_t)(lane * 4) : 0x80000000u)
                                      : (lane == 0 ? (uint32_t)((n0 >> 7) * 4) : 0x80000000u);
    const uint32_t step_s = (brings_sa ? (uint32_t)lda : (uint32_t)sn) * 4u;
    const uint32_t dst_s = lds_base + (brings_sa ? S::SA_OFF : S::SB_OFF);
    // SPREAD: the slab of K block kb travels with the stage two blocks before it, so that it has landed a turn before it is
    // multiplied, which is when the threads spread it
    auto issue_slab = [&](int slot, int kb) __attribute__((always_inline)) {
        if (wave < S::A_WAVES)
            lds_dma16(rsrc_a, kb < kb1 ? voff_a : 0x80000000u, lds_base + (uint32_t)(slot * S::STAGE + S::PACK_OFF + wave * 1024),
                      (uint32_t)kb * KBLOCK * (uint32_t)lda);
    };
    auto issue_stage = [&](int slot, int kb) __attribute__((always_inline)) {
        const uint32_t stage = lds_base + (uint32_t)(slot * S::STAGE);
        lds_dma16(rsrc_b, voff_b, stage + (uint32_t)(wave * 1024), (uint32_t)kb * KBLOCK * (uint32_t)N);
        if (SPREAD)
            issue_slab(slot + 2 >= NS ? slot + 2 - NS : slot + 2, kb + 2);
        else if (wave < S::A_WAVES)
            lds_dma16(rsrc_a, voff_a, stage + S::MAT_B + (uint32_t)(wave * 1024), (uint32_t)kb * KBLOCK * (uint32_t)lda);
        if (T > 2 || wave >= S::A_WAVES)
            lds_dma4(rsrc_s, voff_s, dst_s + (uint32_t)(slot * S::STAGE), (uint32_t)kb * step_s);
    };
    // SPREAD: a thread moves bytes 16 * j .. 16 * j + 15 of packed k-row r (they start at any byte: five aligned words,
    // shifted) to chunk j of the padded row, zeros where the row has ended: of both blocks of a pair, or with one or two row
    // tiles of one of them.  One whose chunk belongs to no row tile writes to the spare bytes behind the slab.
    constexpr int BLOCKS = T > 2 ? 2 : 1;
    const int sp_r = T > 2 ? (int)threadIdx.x >> 2 : ((int)threadIdx.x >> 1) & 127;
    const int sp_j = T > 2 ? (int)threadIdx.x & 3 : (int)threadIdx.x & 1;
    const uint32_t sp_stage = T > 2 ? 0u : (threadIdx.x >> 8) * (uint32_t)S::STAGE;
    const uint32_t sp_src = sp_stage + (uint32_t)(S::PACK_OFF + (sp_j < T ? (sp_r * lda + 16 * sp_j) & ~3 : 0));
    const uint32_t sp_shift = (uint32_t)((sp_r * lda) & 3);
    const uint32_t sp_dst =
        sp_stage + (uint32_t)(sp_j < T ? S::MAT_B + sp_r * S::RSA + ((T == 1 ? 0 : sp_j ^ (T == 2 ? (sp_r >> 3) & 1 : (sp_r >> 2) & 3)) << 4)
                                       : S::PACK_OFF + S::MAT_A);
    uint32_t sp_mask[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int valid = M - 16 * sp_j - 4 * i;  // bytes of word i inside the row
        sp_mask[i] = valid >= 4 ? 0xFFFFFFFFu : valid <= 0 ? 0u : (1u << (8 * valid)) - 1u;
    }
    uint32_t sp_word[BLOCKS][5];
    auto slab_read = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int v = 0; v < BLOCKS; ++v)
#pragma unroll
            for (int i = 0; i < 5; ++i)
                sp_word[v][i] = *LDS_PTR(uint32_t, lds + (slot + v) * S::STAGE + sp_src + 4 * i);
    };
    auto slab_write = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int v = 0; v < BLOCKS; ++v) {
            v4i out;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                out[i] = (int)(__builtin_amdgcn_alignbyte(sp_word[v][i + 1], sp_word[v][i], sp_shift) & sp_mask[i]);
            *LDS_PTR(v4i, lds + (slot + v) * S::STAGE + sp_dst) = out;
        }
    };
    auto wait_landed = [&](int outstanding) __attribute__((always_inline)) {  // stages whose copies may be in flight
        switch (outstanding) {
        case 0: wait_vmcnt<0>(); break;
        case 1: wait_vmcnt<S::COPIES>(); break;
        case 2: wait_vmcnt<2 * S::COPIES>(); break;
        case 3: wait_vmcnt<3 * S::COPIES>(); break;
        case 4: wait_vmcnt<4 * S::COPIES>(); break;
        case 5: wait_vmcnt<5 * S::COPIES>(); break;
        default: wait_vmcnt<6 * S::COPIES>(); break;
        }
    };
    static_assert(NS <= 8, "the wait above knows up to six stages in flight besides the pair");

    // ---- transposing reads.  Lane = 16 * g + i; read t of a K block covers k-rows 32 * t + 8 * g + (i >> 1)
    const int g4 = lane >> 4, i16 = lane & 15;
    const int r8 = 8 * g4 + (i16 >> 1);
    const uint32_t addr_b = (uint32_t)(r8 * RSB + (i16 & 1) * 8 + ((col ^ ((2 * g4 + (i16 >> 3)) & 3)) * 16));
    // PACKED: k-rows of lda bytes without a swizzle; what a read of the last row tile takes from beyond a row belongs to rows
    // of C that do not exist, as do the copies of the one row that ROW reads for lanes 1 - 15
    const int rsa = PACKED ? lda : S::RSA;
    const uint32_t addr_a = (uint32_t)S::MAT_B + (uint32_t)(ROW ? 8 * g4 : r8 * rsa + (i16 & 1) * 8);
    const int swz_a = PACKED || T == 1 ? 0 : T == 2 ? (g4 & 1) : ((2 * g4 + (i16 >> 3)) & 3);
    auto frag = [&](uint32_t addr, int step) __attribute__((always_inline)) -> v8i {
        const v2i r0 = __builtin_amdgcn_ds_read_tr8_b64_v2i32(LDS_PTR(v2i, lds + addr));
        const v2i r1 = __builtin_amdgcn_ds_read_tr8_b64_v2i32(LDS_PTR(v2i, lds + addr + step));
        const v2i r2 = __builtin_amdgcn_ds_read_tr8_b64_v2i32(LDS_PTR(v2i, lds + addr + 2 * step));
        const v2i r3 = __builtin_amdgcn_ds_read_tr8_b64_v2i32(LDS_PTR(v2i, lds + addr + 3 * step));
        return (v8i){r0.x, r0.y, r1.x, r1.y, r2.x, r2.y, r3.x, r3.y};
    };
    auto row_frag = [&](uint32_t addr) __attribute__((always_inline)) -> v8i {
        v2i r[4];
#pragma unroll
        for (int t = 0; t < 4; ++t)
            r[t] = *LDS_PTR(v2i, lds + addr + 32 * t);
        return (v8i){r[0].x, r[0].y, r[1].x, r[1].y, r[2].x, r[2].y, r[3].x, r[3].y};
    };

    v4f acc[T];
#pragma unroll
    for (int i = 0; i < T; ++i)
        acc[i] = (v4f){0.f, 0.f, 0.f, 0.f};

    // Before the first turn all slots are free (slabs, which go two slots further on, leave the last two for it), later
    // those of the pair that was multiplied last.
    constexpr int AHEAD = NS - 2, FIRST = SPREAD ? AHEAD : NS;  // stages issued before the first turn
    const int nstages = kb1 - kb0;
    if (SPREAD) {
        issue_slab(0, kb0);
        issue_slab(1, kb0 + 1);
    }
#pragma unroll
    for (int p = 0; p < FIRST; ++p)
        if (p < nstages)
            issue_stage(p, kb0 + p);
    if (SPREAD) {  // the first slabs have landed once only the stages' copies are in flight
        wait_landed(nstages < FIRST ? nstages : FIRST);
        __syncthreads();
        slab_read(0);
        slab_write(0);
    }
    int slot = 0;
    auto turn = [&](auto count, int s) __attribute__((always_inline)) {  // blocks s .. s + CNT - 1
        constexpr int CNT = decltype(count)::value;
        const int issued = s == 0 ? FIRST : s + AHEAD;
        wait_landed((nstages < issued ? nstages : issued) - s - CNT);
        __syncthreads();  // everyone's copies landed and spreads are done; the slots of the last turn are no longer read
        if (SPREAD || s > 0) {
            const int free_slot = slot == 0 ? NS - 2 : slot - 2;
#pragma unroll
            for (int p = 0; p < 2; ++p)
                if (s + AHEAD + p < nstages)
                    issue_stage(free_slot + p, kb0 + s + AHEAD + p);
        }
        const int next_slot = slot == NS - 2 ? 0 : slot + 2;
        if (SPREAD)  // also behind the last turn: nothing reads what that spreads
            slab_read(next_slot);
        const uint32_t so = (uint32_t)((slot + (CNT == 2 ? par : 0)) * S::STAGE);
        v8i fa[T];
        float sa[T];
        const v8i fb = frag(so + addr_b, 32 * RSB);
        const float sb = *LDS_PTR(float, lds + so + S::SB_OFF);
#pragma unroll
        for (int i = 0; i < T; ++i) {
            sa[i] = *LDS_PTR(float, lds + so + S::SA_OFF + (16 * i + i16) * 4);
            fa[i] = ROW ? row_frag(so + addr_a) : frag(so + addr_a + (uint32_t)((i ^ swz_a) * 16), 32 * rsa);
        }
        if (SPREAD)
            slab_write(next_slot);
        if (CNT == 2 || par == 0) {
#pragma unroll
            for (int i = 0; i < T; ++i) {
                const v4f blk = block_sum(fb, fa[i]);
                const float sc = sa[i] * sb;
                acc[i] = (v4f){fmaf(sc, blk[0], acc[i][0]), fmaf(sc, blk[1], acc[i][1]), fmaf(sc, blk[2], acc[i][2]),
                               fmaf(sc, blk[3], acc[i][3])};
            }
        }
        slot = next_slot;
    };
    int s = 0;
    for (; s + 2 <= nstages; s += 2)
        turn(std::integral_constant<int, 2>{}, s);
    if (s < nstages)
        turn(std::integral_constant<int, 1>{}, s);

    // ---- the two waves of a column add up: wave `col` ends with row tiles 0 .. KEEP-1, wave `col + 4` with the others
    auto tile = [&](int side, int p) __attribute__((always_inline)) { return acc[side * KEEP + p < T ? side * KEEP + p : 0]; };
    auto has = [&](int p) __attribute__((always_inline)) { return KEEP + p < T || par == 0; };
    if (!S::APART)
        __syncthreads();  // nobody reads the ring any more
    const uint32_t ex = (uint32_t)(S::EXCHANGE_OFF + lane * 16);
#pragma unroll
    for (int p = 0; p < KEEP; ++p)
        if (KEEP + p < T || par == 1)
            *LDS_PTR(v4f, lds + ex + (wave * KEEP + p) * 1024) = par ? tile(0, p) : tile(1, p);
    __syncthreads();
    if (T == 1 && par == 1)
        return;
    v4f own[KEEP];
#pragma unroll
    for (int p = 0; p < KEEP; ++p) {
        own[p] = (v4f){0.f, 0.f, 0.f, 0.f};
        if (has(p))
            own[p] = (par ? tile(1, p) : tile(0, p)) + *LDS_PTR(v4f, lds + ex + ((wave ^ 4) * KEEP + p) * 1024);
    }

    // a lane holds C[16 * row tile + (lane & 15)][n0 + 16 * col + 4 * (lane >> 4) + 0..3]
    const int ncol = n0 + 16 * col + 4 * g4;
    auto row_of = [&](int p) __attribute__((always_inline)) { return 16 * (par * KEEP + p) + i16; };
    auto store_c = [&](int p, v4f v) __attribute__((always_inline)) {
        if (row_of(p) < M && ncol < N) {
            uint2 pk;
            pk.x = pack_bf16x2(v[0], v[1]);
            pk.y = pack_bf16x2(v[2], v[3]);
            *reinterpret_cast<uint2*>(c + (size_t)row_of(p) * N + ncol) = pk;
        }
    };
    if (ksplit == 1) {
#pragma unroll
        for (int p = 0; p < KEEP; ++p)
            store_c(p, own[p]);
        return;
    }

    // ---- mailbox: [strip][split 0 .. ksplit-2][wave][row tile][lane] x 16 bytes, all zero between launches
    constexpr int PER_SPLIT = (T == 1 ? 4 : 8) * KEEP;  // patches of one split of a strip
    const int senders = ksplit - 1;
    const size_t first = ((size_t)strip * senders * PER_SPLIT + wave * KEEP) * 64;  // split 0
    if (split < senders) {
#pragma unroll
        for (int p = 0; p < KEEP; ++p)
            if (row_of(p) < M) {
                v4i bits = __builtin_bit_cast(v4i, own[p]);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    bits[e] = bits[e] == 0 ? (int)0x80000000 : bits[e];  // +0.0 -> -0.0: no word is zero
                reinterpret_cast<v4i*>(mailbox)[first + ((size_t)split * PER_SPLIT + p) * 64 + lane] = bits;
            }
        return;
    }
    // last split: the other splits' patches of these rows and columns, AT_ONCE splits at a time
    constexpr int AT_ONCE = KEEP == 1 ? 8 : 4;
    const __amdgpu_buffer_rsrc_t rp = make_rsrc(reinterpret_cast<const v4i*>(mailbox) + first, (uint32_t)senders * PER_SPLIT * 1024u);
    uint32_t off[KEEP];  // outside the resource, which fetches and stores nothing, where the lane's row does not exist
#pragma unroll
    for (int p = 0; p < KEEP; ++p)
        off[p] = row_of(p) < M ? (uint32_t)(p * 64 + lane) * 16u : 0x80000000u;
    auto place = [&](int z) __attribute__((always_inline)) { return (uint32_t)(z * PER_SPLIT) * 1024u; };
    const unsigned long long t_first = __builtin_amdgcn_s_memrealtime();
    bool gave_up = false;
    v4f sum[KEEP];
    for (int z0 = 0; z0 < senders; z0 += AT_ONCE) {
        v4i v[AT_ONCE][KEEP];
        for (;;) {
            asm volatile("" ::: "memory");  // the loads belong to this round of the loop
            // (a split past the last lies outside the resource too)
#pragma unroll
            for (int z = 0; z < AT_ONCE; ++z)
#pragma unroll
                for (int p = 0; p < KEEP; ++p)
                    v[z][p] = __builtin_amdgcn_raw_buffer_load_b128(rp, off[p] + place(z0 + z), 0, PAST_L1);
            bool missing = false;
#pragma unroll
            for (int z = 0; z < AT_ONCE; ++z)
#pragma unroll
                for (int p = 0; p < KEEP; ++p) {
                    const v4i w = v[z][p];
                    missing = missing | ((z0 + z < senders) & (row_of(p) < M) & ((w[0] == 0) | (w[1] == 0) | (w[2] == 0) | (w[3] == 0)));
                }
            if (__builtin_amdgcn_ballot_w64(missing) == 0)
                break;
            if (__builtin_amdgcn_s_memrealtime() - t_first > SPIN_LIMIT) {
                gave_up = true;
                break;
            }
        }
#pragma unroll
        for (int z = 0; z < AT_ONCE; ++z)
            if (z0 + z < senders)
#pragma unroll
                for (int p = 0; p < KEEP; ++p) {
                    const v4f f = __builtin_bit_cast(v4f, v[z][p]);
                    sum[p] = z0 + z == 0 ? f : sum[p] + f;
                }
    }
#pragma unroll
    for (int p = 0; p < KEEP; ++p) {
        v4f total = sum[p] + own[p];
        if (gave_up)
            total = (v4f){__builtin_nanf(""), __builtin_nanf(""), __builtin_nanf(""), __builtin_nanf("")};
        store_c(p, total);
    }
    for (int z = 0; z < senders; ++z)
#pragma unroll
        for (int p = 0; p < KEEP; ++p)
            __builtin_amdgcn_raw_buffer_store_b128((v4i){0, 0, 0, 0}, rp, off[p] + place(z), 0, 0);
}

inline int strip_count(int n) { return (n + BN - 1) / BN; }

// Neighbours on one XCD, whose L2 then has the other half of each line of B (24 x 1536 x 7168 in eight splits 7.80 -> 6.55 us,
// 7168 x 2048 in two 8.70 -> 6.95); up to 16 strips, which that would leave half of the XCDs without one, dealt out (24 x
// 576 x 7168 in 14 splits 5.99 -> 5.78).
inline bool neighbours_paired(int strips) { return strips > 16; }

}  // namespace

// us of a launch of one round, the mean of operands from the Infinity Cache and from HBM, as sums of the launch, the K blocks and
// turns one behind the other, the hand-over (its trips, eight splits each or four, and its bytes) and B's bytes.  Fitted to
// 340 random problems of 1 ... 64 rows, N = 256 ... 8192, K = 256 ... 8192, B up to 33 MB (strips of 64 columns in up to seven
// splits each, 4 % rms; of 128 in the split that decode_strip_cost picks, 5 % rms).  They are asked for larger B too: of 64 random
// problems of 33 ... 57 MB, K = 6912 ... 25216, that go to strips of 64, all are ahead from the Infinity Cache, by 22 %, and 61 from
// HBM, by 16 % on average (1 x 1488 x 24704 16.6 -> 14.6 / 16.6 -> 15.2, 55 x 4096 x 9088 16.1 -> 15.5 / 17.0 -> 17.2).
namespace {

struct Chain {
    int blocks, turns, tiles;
    double spread;  // rows that are spread
    Chain(const GemmArgs& g, int ksplit, bool row_form)
    {
        blocks = (g.k / KBLOCK + ksplit - 1) / ksplit;
        turns = (blocks + 1) / 2;
        tiles = (g.m + 15) / 16;
        spread = leading_dim(g) % 8 == 0 || (row_form && leading_dim(g) == 1) ? 0.0 : 1.0;
    }
};

double decode64_us(const GemmArgs& g, int ksplit)
{
    const Chain x(g, ksplit, true);
    double us = 2.345 + 0.218 * x.blocks + (0.084 + 0.15 * (x.tiles - 1)) * x.turns + x.spread * (0.415 + 0.053 * x.turns) +
                0.1065e-6 * g.n * g.k;
    if (ksplit > 1) {
        const int at_once = x.tiles <= 2 ? 8 : 4;
        us += 0.773 + 0.418 * ((ksplit - 1 + at_once - 1) / at_once - 1) + 0.0358 * (ksplit - 1) * x.tiles;
    }
    return us;
}

double decode128_us(const GemmArgs& g, int ksplit)
{
    const Chain x(g, ksplit, false);
    return 2.194 + (0.606 + 0.174 * (x.tiles - 1)) * x.turns + x.spread * (0.234 + 0.048 * x.turns) + 0.1263e-6 * g.n * g.k +
           (ksplit > 1 ? 0.247 + 0.1874 * (ksplit - 1) * x.tiles : 0.0);
}

}  // namespace

int decode64_ksplit(const GemmArgs& g)
{
    const int strips = strip_count(g.n), nkb = g.k / KBLOCK;
    const int per_xcd = neighbours_paired(strips) ? 2 * ((strips + 15) / 16) : (strips + 7) / 8;
    int best = 0;
    double best_us = 0.0;
    for (int ks = 1; ks <= DECODE_MAX_KSPLIT && ks <= nkb; ++ks) {
        // one round of workgroups, one to a CU; every split owns a K block
        if (per_xcd * ks > 32 || (ks - 1) * ((nkb + ks - 1) / ks) >= nkb || (ks > 1 && decode64_mailbox_bytes(g, ks) > SPLIT_MAILBOX_BYTES))
            continue;
        const double us = decode64_us(g, ks);
        if (best == 0 || us < best_us) {
            best = ks;
            best_us = us;
        }
    }
    return best;
}

// By the smaller of the two estimates, and where the reasons hold: a pair of K blocks to take, and several row tiles that eight
// waves need not all read, many splits to hand over, or a single row.  The 340 problems with the choice made so: 6.4 %
// faster than in 128-column strips throughout, up to 1.4 times (27 x 576 x 7168, 1 x 304 x 4608), 0.5 % slower at worst; each in
// the better of both 7.8 %.  One tile of 2 - 16 rows in up to four splits too: 6.7 %, 5 % slower at worst (16 x 4560 x 1536).
bool decode64_pays(const GemmArgs& g, int ksplit, int ksplit128)
{
    return ksplit > 0 && g.k > KBLOCK && (g.m > 16 || leading_dim(g) == 1 || ksplit128 >= 5) &&
           decode64_us(g, ksplit) < 0.98 * decode128_us(g, ksplit128);
}

size_t decode64_mailbox_bytes(const GemmArgs& g, int ksplit)
{
    const size_t waves = g.m <= 16 ? 4 : 8, keep = g.m <= 32 ? 1 : 2;
    return (size_t)strip_count(g.n) * (size_t)(ksplit - 1) * waves * keep * 1024;
}

hipError_t launch_decode64(const GemmArgs& g, int ksplit, float* mailbox, hipStream_t s)
{
    const int strips = strip_count(g.n), nkb = g.k / KBLOCK;
    if (!decode_strip_supports(g) || ksplit < 1 || ksplit > nkb || ksplit > DECODE_MAX_KSPLIT ||
        (ksplit > 1 && (!mailbox || decode64_mailbox_bytes(g, ksplit) > SPLIT_MAILBOX_BYTES)))
        return hipErrorInvalidValue;
    const int kb_per_split = (nkb + ksplit - 1) / ksplit;
    if ((ksplit - 1) * kb_per_split >= nkb)  // every split owns at least one K block
        return hipErrorInvalidValue;
    const bool paired = neighbours_paired(strips);
    // a multiple of 8: the splits of a strip share an XCD
    const dim3 grid(paired ? 16 * ((strips + 15) / 16) : 8 * ((strips + 7) / 8), ksplit);
    auto go = [&](auto form_c, auto tiles_c) -> hipError_t {
        constexpr Rows F = decltype(form_c)::value;
        constexpr int T = decltype(tiles_c)::value, lds = Strip64<T, F>::LDS;
        constexpr auto kern = decode64_kernel<T, F>;
        FP8GEMM_ALLOW_LDS(kern, lds);
        launch_kernel(kern, grid, dim3(NTHREADS), lds, s, g.b, g.a, g.n, g.k, g.m, leading_dim(g), kb_per_split, strips,
                           g.a_scale, g.b_scale, g.c, mailbox, ksplit, paired ? 1 : 0);
        return hipGetLastError();
    };
    auto by_tiles = [&](auto form_c) -> hipError_t {
        switch ((g.m + 15) / 16) {
        case 1: return go(form_c, std::integral_constant<int, 1>{});
        case 2: return go(form_c, std::integral_constant<int, 2>{});
        case 3: return go(form_c, std::integral_constant<int, 3>{});
        default: return go(form_c, std::integral_constant<int, 4>{});
        }
    };
    const int ld = leading_dim(g);
    if (ld == 1)
        return go(std::integral_constant<Rows, Rows::ROW>{}, std::integral_constant<int, 1>{});
    return ld % 16 == 0 ? by_tiles(std::integral_constant<Rows, Rows::GRID>{})
           : ld % 8 == 0 ? by_tiles(std::integral_constant<Rows, Rows::PACKED>{})
                         : by_tiles(std::integral_constant<Rows, Rows::SPREAD>{});
}

}  // namespace fp8gemm
