// C ABI of the library (include/fp8_block_gemm.h): argument validation, kernel dispatch,
// split-K workspace.  The dispatcher is the run-time counterpart of the reference's
// compile-time kernel choice (#include "mn_large.hip" / "mn_small.hip", check.cu:13, and the
// OPTION macro, mn_large.hip:9) and of gemmGPU's grid arithmetic (check.cu:92-114).
#include "../../include/fp8_block_gemm.h"
#include "launchers.h"

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <mutex>
#include <vector>

using namespace fp8gemm;

namespace {

constexpr int NUM_CU = 256;

// Process-wide defaults, set by fp8_block_gemm_select / _force_config / _set_persistent and read by
// the entry points without an options argument.  The _ex / _ws entry points read none of this.
std::atomic<int> g_selected{FP8GEMM_KERNEL_AUTO};
std::atomic<int> g_force_variant{-1};
std::atomic<int> g_force_ksplit{0};
std::atomic<int> g_persistent{-1};  // -1 = where it pays (decide_persistent), 0 = never, 1 = whenever possible
std::atomic<int> g_fused{-1};       // K splits added inside the GEMM kernel: -1 = by cost, 0 = never, 1 = whenever possible
thread_local const char* t_last_kernel = "none";
thread_local char t_name_buf[96];

// what decides a plan besides the shape
struct Config {
    int selected;       // FP8GEMM_KERNEL_*
    int force_variant;  // tile shape, -1 = cost model
    int force_ksplit;   // 0 = cost model
    int persistent;     // -1 / 0 / 1 as above
    // plans that add K splits inside the kernel may be chosen: the workspace starts with a zeroed header
    // and the device places workgroups on XCDs as those kernels assume (set by run())
    bool fused_ok = true;
    int fused_mode = -1;  // -1 = by cost, 0 = never, 1 = whenever fused_ok and the plan allows
    bool strips_for_tiles = true;  // 64-column strips may take the place of 64x64 tiles (strips_for_tiles below)
    bool ragged = false;  // the problem is one with its rows rounded up to 16, which tiles take as they are (off_grid_plan)
    size_t partial_room = SIZE_MAX;  // automatic plans keep no more bytes of partial sums in the workspace (fitting_plan)
};
Config global_config()
{
    Config c{g_selected.load(), g_force_variant.load(), g_force_ksplit.load(), g_persistent.load()};
    c.fused_mode = g_fused.load();
    c.fused_ok = c.fused_mode != 0;
    return c;
}
constexpr int MAX_KSPLIT = 16;

// device memory a call may use beyond its operands: fp32 partial sums of plans that split K, padded
// copies of operands off the 16-byte grid
// The first WS_HEADER bytes belong to the kernels that add their K splits themselves and are zero before
// the first call and after every call: the mailbox through which the splits of a tile or strip hand over
// their partial results.  Plans keep their data behind it.
struct Workspace {
    float* ptr;
    size_t bytes;
    bool zeroed;  // the header was zero-filled when the buffer was taken on and only this library wrote to it since
};
constexpr size_t WS_HEADER = SPLIT_MAILBOX_BYTES;
static_assert(WS_HEADER == FP8GEMM_WORKSPACE_HEADER_BYTES, "the header size is part of the ABI");
inline float* ws_data(const Workspace& w) { return w.ptr ? reinterpret_cast<float*>(reinterpret_cast<uint8_t*>(w.ptr) + WS_HEADER) : nullptr; }
inline float* ws_mailbox(const Workspace& w) { return w.ptr; }

std::mutex g_ws_mutex;
float* g_ws_own = nullptr;       // library-owned workspace
size_t g_ws_own_bytes = 0;
bool g_ws_own_captured = false;  // handed out to a call whose stream was being captured: a graph holds its address
hipStream_t g_ws_last_stream = nullptr;  // stream of the last call that was given the library-owned workspace
// Outgrown library-owned buffers.  Kernels of earlier calls may still use one: it is freed by a later
// growth once the event recorded behind its last use has completed.  One that a captured graph may hold
// (pinned) lives until fp8_block_gemm_release().
struct Retired {
    void* ptr;
    hipEvent_t done;  // nullptr when pinned
    bool pinned;
};
std::vector<Retired> g_ws_retired;
float* g_ws_user = nullptr;      // caller-supplied workspace
size_t g_ws_user_bytes = 0;
bool g_ws_user_zeroed = false;

// Size the library-owned workspace grows to when a call needs `need` bytes and `have` are there: at
// least double, so that the buffers retired on the way never add up to more than the live one.
size_t growth_target(size_t have, size_t need)
{
    if (need <= have)
        return have;
    const size_t twice = have > (SIZE_MAX >> 1) ? SIZE_MAX : 2 * have;
    return need > twice ? need : twice;
}

struct Plan {
    int family;   // FP8GEMM_KERNEL_*
    int variant;  // TileVariant for the tile families
    int ksplit;
    bool persistent = false;  // tile families, ksplit == 1: workgroups walk through the tiles
    bool padded = false;      // the plan is for the problem with m and n rounded up to 16 (run_padded)
    bool wide = false;        // decode family: 128-column strips, K splits added inside the kernel (k_decode.hip)
    bool fused = false;       // tile family, ksplit > 1: the last workgroup of a tile adds the partial tiles (no reduction launch)
    int halves = 1;           // wide decode strips: 128-column halves per strip (2 = 256-column strips, 0 = 64-column ones)
    double us = 0.0;          // the estimate that chose the plan
};

// Shapes or addresses the MFMA kernels cannot take (m or n not a multiple of 16, a base not
// 16-byte aligned) run on padded copies in the workspace: which operands are copied, and where.
struct PadLayout {
    bool a, as, b, c;
    int m16, n16;
    size_t off_a, off_as, off_b, off_c, off_partial, total;
};

inline size_t round256(size_t x) { return (x + 255) & ~(size_t)255; }
inline bool misaligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) != 0; }

// conservative = true: every operand copied (an upper bound that does not depend on addresses).
// keeps_rows = the kernels of the plan take a leading dimension for a and a_scale apart from m
// (the tile kernels and the wide decode strips): c then needs no copy on account of m.
PadLayout pad_layout(const GemmArgs& g, size_t partial_bytes, bool conservative, bool keeps_rows)
{
    PadLayout L{};
    L.m16 = (g.m + 15) & ~15;
    L.n16 = (g.n + 15) & ~15;
    const bool rm = L.m16 != g.m, rn = L.n16 != g.n;
    L.a = conservative || rm || misaligned16(g.a);
    L.as = conservative || rm || misaligned16(g.a_scale);
    L.b = conservative || rn || misaligned16(g.b);
    L.c = conservative || (rm && !keeps_rows) || rn || misaligned16(g.c);
    const size_t nkb = (size_t)g.k / 128;
    size_t off = 0;
    L.off_a = off;
    off += L.a ? round256((size_t)g.k * L.m16) : 0;
    L.off_as = off;
    off += L.as ? round256(nkb * L.m16 * sizeof(float)) : 0;
    L.off_b = off;
    off += L.b ? round256((size_t)g.k * L.n16) : 0;
    L.off_c = off;
    off += L.c ? round256((size_t)L.m16 * L.n16 * 2) : 0;
    L.off_partial = off;
    off += partial_bytes;
    L.total = off;
    return L;
}

int validate(const void* a, const void* b, const float* as, const float* bs, const void* c, int m,
             int n, int k)
{
    if (!a || !b || !as || !bs || !c)
        return FP8GEMM_E_NULLPTR;
    if (m <= 0 || n <= 0 || k <= 0 || (k % 128) != 0)
        return FP8GEMM_E_SHAPE;
    const long long lim = 0x7FFFFFFFll;
    if ((long long)m * k > lim || (long long)n * k > lim || (long long)m * n > lim)
        return FP8GEMM_E_TOOLARGE;
    return FP8GEMM_OK;
}

// The 256x256 tile, in the units of the fit below (which was made on operands in the caches and at the clock of short
// runs; 256x192 measures 1.39 us per K block where it says 1.10): full rounds and what is done with the tiles left over
// (large_tile_tail).  Measured on 8192 x 4608, 8192 x 7168 and 4096 x 4608 with K = 512 ... 7168, operands in turn: a
// round 4.0 us + 1.6 per K block, a round of halves 7.0 + 1.03, of quarters 3.7 + 0.57 (+ 2 with short K, where other
// shapes are as fast: 4322 x 4096 x 512 24.8 us against 22.9 in 128x192 tiles).  30 random shapes whose plan changed with
// this and the kernel: 26 faster, by up to 20 % (2192 x 8016 x 4864 113.2 -> 91.5 us, 6816 x 7312 x 3200 187.9 -> 156.5).
double large_tile_cost(long tiles, int k, double per_kb)
{
    const int nkb = k / 128;
    const Tail tail = large_tile_tail(tiles, k, NUM_CU);
    const long rounds = tail == Tail::NONE ? (tiles + NUM_CU - 1) / NUM_CU : tiles / NUM_CU;
    double cost = 1.79 + rounds * (4.5 + nkb * 1.335 * per_kb);
    if (tail == Tail::HALVES)
        cost += 6.0 + nkb * 0.86 * per_kb;
    else if (tail == Tail::QUARTERS)
        cost += 7.0 + nkb * 0.48 * per_kb;
    return cost;
}

// Estimated run time of a tile plan in microseconds.  The form is launch + rounds of 256
// workgroups x (pipeline fill + K blocks + store) + the split-K reduction; the constants are a
// least-squares fit to a sweep of every tile variant x ksplit over the 18 shapes of the
// reference's table (/root/reference/README.md:15-25) and the five benchmark shapes (rms
// error 10 %, the chosen plan within 6 % of the best measured one on all of them).
double tile_cost(const GemmArgs& g, int variant, int ksplit, bool fused, bool ragged)
{
    int bm, bn;
    tile_variant_dims(variant, &bm, &bn);
    const long tiles = (long)((g.m + bm - 1) / bm) * ((g.n + bn - 1) / bn);
    if (variant == TILE_256x256)
        return large_tile_cost(tiles, g.k, 1.0);
    const int nkb = g.k / 128;
    const int kbs = (nkb + ksplit - 1) / ksplit;
    const double area = (double)bm * bn / 65536.0;
    // (a single row of tiles reads every byte of B once and from HBM -- decode weights do not fit the caches --,
    // where a K block takes a quarter longer than the fit to cached operands says: without this factor
    // 48 x 7168 x 1536 stays unsplit, 9.4 us from HBM against 8.1 us with two splits; the same for two rows of
    // to four rows of 64x64 tiles over a B of 16 MB or more, which they fetch in 64-byte pieces: 128 x 4096 x 7168
    // as tile64x64_k2f 22.2 us, as tile128x128_k7 17.1 us; 176 x 4608 x 4096 as tile64x64_k1 21.2 us from HBM and
    // 12.8 us with B in the Infinity Cache, as tile128x128_k3f 16.6 and 15.9 us -- while over 1536 x 7168
    // tile64x64_k5f stays ahead, 11.9 against 12.9 us)
    const bool streams_b = g.m <= 64 || (variant == TILE_64x64 && g.m <= 256 && (long long)g.n * g.k >= 16000000ll);
    // (with the splits added inside the kernel the grid holds a multiple of 8 tiles, so that the splits of a tile
    // share an XCD: the workgroups beyond the tiles exit at once but take their turn -- 85 tiles x 3 splits are
    // 264 workgroups, and the last of them start when a CU frees up: 20.2 us against 13.9 us with two splits)
    const long items = (ksplit > 1 && fused ? (tiles + 7) / 8 * 8 : tiles) * ksplit;
    // (64x64 tiles: the fit knows the kernel before four waves read ahead and all eight hand splits over.  Fill and store
    // take 0.72 us less, and with 64 tiles or fewer a K block takes 0.285 us for 32 of them and 0.015 more for every 32
    // beyond, the hand-over starts 0.3 us earlier; with more tiles a block takes 9 % longer than the fit says, and 3.5 % with no more of
    // them over a B that streams in.  649 random
    // problems of 48 ... 4096 rows, every plan measured: the one chosen was 1.4 / 1.7 % behind the best one from the Infinity
    // Cache / HBM and is 0.7 / 0.9 %; the 110 that change are 6 and 8 % faster on average (149 x 7168 x 256 as 128x128 5.07 us,
    // now 4.32; 224 x 2336 x 4096 as 128x128 in four 14.7 / 17.0, now in three 12.1 / 15.1; 256 x 336 x 1536 unsplit 4.69 / 6.60,
    // now in three 4.49 / 5.30), at worst 368 x 1008 x 6144 as 128x128 in eight 14.7 / 16.0, now in two 14.0 / 19.4.)
    const bool small = variant == TILE_64x64;
    const bool light = small && !streams_b && tiles <= 64;
    const double of_small = !small ? 1.0 : light ? 0.838 : tiles > 64 ? 1.087 : 1.035;
    // (128x128 tiles with ragged rows, whose A comes through registers: 0.06 us more to fill than the fit says, which decides where two
    // plans are level.  Without it / with it, from the Infinity Cache and from HBM: 17 problems of 629 ... 637 x 4608 x 7168, 1891 ... 1915 x
    // 1536 x 7168 and such, unsplit / as 128x192 in two splits, 0.96 and 1.12; 11 over K = 640 and 768, unsplit / as 64x64, 1.01 and 1.10; six in
    // two splits / as 128x192 in four 0.96 and 1.07; three of 804 ... 815 x 576 x 7168 in seven splits / as 64x64 in two 1.10 and 0.88.
    // On the grid it would be wrong: 51 unsplit ones / as 128x192 in two 0.88 and 1.06 (1920 x 1536 x 7168 26.8 us / 34.4 and 36.8 / 36.9),
    // 46 / as 64x64 0.96 and 1.02.)
    // (256x192 in the persistent form: the fit knows the kernel before its barrier moved, 5 % slower)
    // (unsplit 128x128 tiles in one round: the fit knows the kernel before four waves read ahead of themselves, 10 - 15 %
    // slower from the caches, and level from HBM, where the copies bound it: they do also where a row of B starts
    // anywhere on a line of 128 bytes, so that each row of a tile is two of them, 2896 x 704 x 5760 26.4 us against 24.9 as
    // 256x128 with three splits.  At 0.94 shapes change from two or three splits of 128x192 or 256x128 tiles: 20
    // random ones with whole lines of B all faster from the caches, by 16 - 31 % (640 x 4480 x 6144 30.7 -> 23.5 us), and
    // -1 ... +22 % from HBM, 6 % on average; five without -6 ... +9 % there.  At 0.88 more change, down to -14 % from HBM.)
    const bool ahead = variant == TILE_128x128 && ksplit == 1 && g.m > 256 && tiles <= NUM_CU &&
                       leading_dim(g) % 16 == 0 && g.n % 128 == 0;
    const double per_kb = (1.19 * area + 0.267) * (variant == TILE_256x192 && ksplit == 1 && tiles > NUM_CU ? 0.95 : 1.0) *
                          (streams_b ? 1.25 : 1.0) * of_small * (ahead ? 0.94 : 1.0) +
                          (light ? 0.015 * (double)(tiles - 32) / 32.0 : 0.0);
    // (unsplit 128x192 tiles in more than one round of workgroups: the fit has them 8 % too fast against the 256-row
    // tiles -- 36 random shapes of 512 ... 8192 rows where that margin decides, before / after: the 256x256 or
    // 256x128 plan +5.6 % with B cached, +10.3 % with B from HBM on average, worst -2.3 %)
    const double in_rounds = variant == TILE_128x192 && ksplit == 1 && tiles > NUM_CU ? 1.08 : 1.0;
    double per_item = (small ? 0.23 : variant == TILE_128x128 && ragged ? 1.01 : 0.95) + 4.38 * area + kbs * per_kb * in_rounds;
    // (two 64x64 workgroups share a CU, but a single row of tiles with B from HBM is fastest with at most one
    // workgroup per CU: M = 48, 64 on 12 shapes, the split that keeps tiles x splits within 256 is the best
    // measured or within 2 % of it)
    const long rounds = (items + NUM_CU - 1) / NUM_CU;
    // (64x64 tiles over a single K block in more than one round: a round takes 1.1 to 1.6 us, the start and end of its
    // workgroups, however little they multiply; 44 problems of 276 ... 768 such tiles.  In three rounds 128x128 tiles are ahead, 4112 x
    // 640 x 128 4.6 us against 5.8, 1997 x 1536 x 128 5.4 against 6.5; in two they are level, 6342 x 224 x 128 4.8 and 4.9 us)
    if (small && rounds > 1 && per_item < 1.25)
        per_item = 1.25;
    double cost = 1.79 + rounds * per_item;
    if (ksplit > 1 && fused)  // the last split of a tile waits for the others' accumulators and reads them
        cost += (light ? 1.5 : 1.8) + 0.35 * (ksplit - 1) * (double)(bm * bn) / 4096.0;
    else if (ksplit > 1) {  // second launch + partial write and read-back
        cost += 2.86 + (double)g.m * g.n * ksplit * 8.0 / 7.38e6;
        // (a GEMM kernel shorter than a launch takes cannot hide the reduction's launch behind it: two such kernels
        // take 9 - 9.5 us back to back whatever the split, 112 x 96 x 1536 ... 256 x 256 x 7168)
        const double first = rounds * per_item;
        cost += first < 4.5 ? 4.5 - first : 0.0;
    }
    return cost;
}

// The in-kernel reduction against the reduction kernel, measured on 11 shapes x 13 split plans (all
// bit-identical): the workgroup of a tile's last split reads the other splits' accumulators at the 15-20
// bytes per clock one CU takes in, so it pays while that is little -- 64x64 tiles (16 KB per split): 2-35 %
// faster up to 8 splits; 128x128 tiles (64 KB per split): 0-45 % faster with two or three splits unless
// only a handful of workgroups run (256 x 256 x 7168: 2-6 % slower) -- and loses beyond (128x128 with six
// splits +25 %, 256x192 up to 2 x), where the reduction kernel's 256 CUs read the partials together.
bool tile_fused_pays(const GemmArgs& g, int variant, int ksplit)
{
    if (variant == TILE_64x64)
        return ksplit <= 8;
    if (variant == TILE_128x128) {
        const long tiles = (long)((g.m + 127) / 128) * ((g.n + 127) / 128);
        return ksplit <= 3 && tiles * ksplit >= 64;
    }
    return false;
}

// whether a tile plan that splits K would add its splits inside the kernel
bool tile_plan_fused(const GemmArgs& g, int variant, int ksplit, const Config& cfg)
{
    if (ksplit <= 1 || !cfg.fused_ok || cfg.fused_mode == 0 || tile_mailbox_bytes(g, variant, ksplit) > SPLIT_MAILBOX_BYTES)
        return false;
    return cfg.fused_mode == 1 || tile_fused_pays(g, variant, ksplit);
}

// Row counts off the 16-byte grid: the tiles' form that takes them as they are against the copy launch and the plain
// form.  A comes through registers in the former, 0.05 to 0.1 us more per K block, where the copies take 1.5 to 6 us: 101
// random shapes of 65 ... 4000 rows 27 % faster on average with operands from the Infinity Cache, 25 % from HBM.  The lines
// are where the two meet when a workgroup walks long (128x128: 333 x 4608 unsplit 18.9 / 23.6 / 37.6 us for 24 / 32 / 56
// blocks against 19.4 / 23.8 / 36.0; 1501 x 1536, more to copy, 37.8 against 39.3 for 56; 128x192: 397 x 7168 25.1 /
// 31.6 / 51.4 against 26.6 / 32.9 / 51.2).  256x128 tiles have no such form: no registers are left to hide a trip behind,
// and it was level at four blocks and 20 % behind at 12.
bool tile_ragged_pays(const GemmArgs& g, int variant, int ksplit)
{
    int bm, bn;
    tile_variant_dims(variant, &bm, &bn);
    const long items = (long)((g.m + bm - 1) / bm) * ((g.n + bn - 1) / bn) * ksplit;
    const long rounds = (items + NUM_CU - 1) / NUM_CU, blocks = (g.k / 128 + ksplit - 1) / ksplit;
    return rounds * blocks <= (variant == TILE_128x192 ? 40 : 56);
}

// Shapes whose best measured plan differs from the model's choice: {m, n, k, variant, ksplit}.
struct TunedShape { int m, n, k, variant, ksplit; };
constexpr TunedShape kTuned[] = {
    {1024, 512, 7168, TILE_64x64, 2},
    {1024, 576, 7168, TILE_128x128, 4},
};

// tile shapes that exist in the persistent form only (and run only when asked for by number)
inline bool persistent_only(int variant) { return variant == TILE_256x192_W4 || variant == TILE_256x256; }
// ... of which the dispatcher may pick this one by itself
inline bool persistent_only_auto(int variant) { return variant == TILE_256x256; }

// A persistent launch pays off when a CU gets more than one tile -- but for 128x128 tiles, whose plain form multiplies
// with four waves that read ahead, only while the K range is short (4992 x 1664 x 384 10.0 us persistent, 10.2 plain; 4096 x
// 4096 x 1024 26.2, 26.2; 1664 x 4864 x 1408 18.0, 16.5; 2688 x 3072 x 3840 40.7, 35.3; 1040 x 6912 x 7552 75.9, 64.2; 13
// more random shapes of K = 2176 ... 6144 all 4 - 16 % faster plain).
// For 256x192 tiles over more than eight K blocks it pays in a single round too: that kernel's barrier does not hold its
// MFMAs up (k_tile_large.hip).  Plain / persistent, us: 928 x 8640 x 2048 25.6 / 23.6, 3792 x 3072 x 3072 41.2 / 37.2, 4032 x 2640 x
// 5120 61.1 / 54.5, 3328 x 2496 x 1536 20.3 / 19.2, 2272 x 2864 x 1152 16.7 / 16.5; eight blocks 4064 x 752 x 1024 14.06 / 14.48,
// 1264 x 9536 x 1024 18.0 / 17.6, five 2288 x 1520 x 640 10.74 / 11.45.
void decide_persistent(const GemmArgs& g, Plan& p, const Config& cfg)
{
    p.persistent = false;
    const int mode = cfg.persistent;
    if (persistent_only(p.variant)) {
        p.persistent = p.ksplit == 1 && tile_persistent_supports(g, p.variant);
        return;
    }
    if (mode == 0 || p.ksplit != 1 || !tile_persistent_supports(g, p.variant))
        return;
    int bm, bn;
    tile_variant_dims(p.variant, &bm, &bn);
    const long tiles = (long)((g.m + bm - 1) / bm) * ((g.n + bn - 1) / bn);
    p.persistent = mode == 1 || (tiles > NUM_CU ? p.variant != TILE_128x128 || g.k < 1024 : p.variant == TILE_256x192 && g.k > 1024);
}

// Whether a tile plan that splits K adds the partial tiles inside the GEMM kernel (the last workgroup of
// a tile to finish) or leaves them to the reduction kernel.
void decide_fused(const GemmArgs& g, Plan& p, const Config& cfg)
{
    p.fused = tile_plan_fused(g, p.variant, p.ksplit, cfg);
}

Plan compute_plan(const GemmArgs& g, const Config& cfg);

// The plan of a problem depends on its sizes, on the low address bits of its operands and on the switches: a
// serving loop asks for the same few again and again, and working one out costs a microsecond or two of host
// time (three are looked up in a call until the workgroups' placement is known, one from then on), which is what a launch-bound decode loop runs on.  Each thread keeps the
// last plans it worked out, 64 slots indexed by a hash of the sizes.
struct PlanKey {
    int m, n, k, lda;
    uint32_t low_bits;  // 6 low address bits of a, b, a_scale, b_scale and c
    int selected, force_variant, force_ksplit, persistent, fused_mode;
    int allowed;  // bit 0: fused_ok, bit 1: strips_for_tiles, bit 2: ragged
    size_t partial_room;
    bool operator==(const PlanKey& o) const
    {
        return m == o.m && n == o.n && k == o.k && lda == o.lda && low_bits == o.low_bits && selected == o.selected &&
               force_variant == o.force_variant && force_ksplit == o.force_ksplit && persistent == o.persistent &&
               fused_mode == o.fused_mode && allowed == o.allowed && partial_room == o.partial_room;
    }
};
struct PlanSlot {
    PlanKey key;
    Plan plan;
    bool used = false;
};
Plan make_plan(const GemmArgs& g, const Config& cfg)
{
    thread_local PlanSlot slots[64];
    auto low6 = [](const void* p) { return (uint32_t)(reinterpret_cast<uintptr_t>(p) & 63); };
    const PlanKey key{g.m, g.n, g.k, g.lda,
                      low6(g.a) | low6(g.b) << 6 | low6(g.a_scale) << 12 | low6(g.b_scale) << 18 | low6(g.c) << 24,
                      cfg.selected, cfg.force_variant, cfg.force_ksplit, cfg.persistent, cfg.fused_mode,
                      (cfg.fused_ok ? 1 : 0) | (cfg.strips_for_tiles ? 2 : 0) | (cfg.ragged ? 4 : 0), cfg.partial_room};
    const uint32_t h = ((uint32_t)g.m * 2654435761u) ^ ((uint32_t)g.n * 40503u) ^ ((uint32_t)g.k * 2246822519u) ^
                       (cfg.fused_ok ? 0x9E3779B9u : 0u) ^ (cfg.partial_room != SIZE_MAX ? 0x85EBCA6Bu : 0u) ^ (cfg.ragged ? 0xC2B2AE35u : 0u);
    PlanSlot& slot = slots[(h >> 16 ^ h) & 63];
    if (slot.used && slot.key == key)
        return slot.plan;
    slot.plan = compute_plan(g, cfg);
    slot.key = key;
    slot.used = true;
    return slot.plan;
}

// Rows without 16-byte alignment under automatic dispatch: the plan of the problem padded to the grid, on copies of the
// operands that need one (their one or two extra launches cost about 5 us; the scalar kernel, one dependent load after the
// other, takes 30 us for K = 128 already) or, where only m is off the grid, without any if the plan's tiles take that.  The
// scalar kernel if padding pushes an operand past the size limit.
Plan off_grid_plan(const GemmArgs& g, Config cfg)
{
    const long long m16 = (g.m + 15) & ~15, n16 = (g.n + 15) & ~15, lim = 0x7FFFFFFFll;
    if (m16 * g.k > lim || n16 * g.k > lim || m16 * n16 > lim)
        return Plan{FP8GEMM_KERNEL_SCALAR, 0, 1};
    const uint8_t* const al8 = reinterpret_cast<const uint8_t*>(uintptr_t(4096));
    GemmArgs gp{al8, al8, reinterpret_cast<const float*>(uintptr_t(4096)), g.b_scale,
                reinterpret_cast<uint16_t*>(uintptr_t(4096)), (int)m16, (int)n16, g.k};
    cfg.ragged = tile_ragged_supports(g, TILE_128x128);
    Plan p = make_plan(gp, cfg);
    const bool tiles = p.family == FP8GEMM_KERNEL_LARGE || p.family == FP8GEMM_KERNEL_SPLITK;
    if (tiles && !p.persistent && tile_ragged_supports(g, p.variant) && tile_ragged_pays(g, p.variant, p.ksplit))
        return p;
    p.padded = p.family != FP8GEMM_KERNEL_SCALAR && p.family >= 0;
    return p;
}

// 33 ... 56 rows, multiples of 8, over weights that want five splits or more of 64x64 tiles: the 64-column strips, whose stages
// are shorter (a fragment of B is read once for all row tiles), in their own number of splits.  16 random problems, from
// the Infinity Cache / from HBM: 8 / 9 % faster on average, 4 - 16 % (48 x 1232 x 1920 6.2 -> 5.4, 48 x 1536 x 7168 9.0 -> 8.3 /
// 10.0 -> 9.4).  Left with the tiles: rows that are spread (36 x 576 x 7168 8.2 -> 8.7, 45 x 576 x 1792 5.95 -> 5.62), 57 rows and
// more (64 x 2464 x 4736 8.2 -> 9.4 / 9.5 -> 9.8, 64 x 1680 x 2560 level), fewer splits (one to three 2 - 20 % slower) and a B of
// 20 MB or more, which decides there and comes slower in pieces of 64 bytes from fewer workgroups (48 x 2400 x 9984 10.5 -> 12.4 / 12.7 ->
// 13.4, 48 x 5824 x 9088 15.8 -> 18.7 / 19.5 -> 21.1; eleven of 24 ... 53 MB 11 / 5 % slower, 55 of 1 ... 15 MB 9 / 10 % faster).
Plan strips_for_tiles(const GemmArgs& g, const Plan& tiles)
{
    if (tiles.variant != TILE_64x64 || !tiles.fused || g.m <= 32 || g.m > 56 || leading_dim(g) % 8 != 0 || tiles.ksplit < 5 ||
        (long long)g.n * g.k >= 20000000ll || !decode_strip_supports(g))
        return tiles;
    const int ks = decode64_ksplit(g);
    if (ks <= 1)
        return tiles;
    Plan strips{FP8GEMM_KERNEL_SKINNY, 0, ks};
    strips.wide = true;
    strips.halves = 0;
    return strips;
}

Plan compute_plan(const GemmArgs& g, const Config& cfg)
{
    const int selected = cfg.selected;
    Plan p{FP8GEMM_KERNEL_SCALAR, 0, 1};
    if (selected == FP8GEMM_KERNEL_SCALAR)
        return p;
    // The decode kernels (M <= 32): narrow strips (k_skinny.hip) or wide strips whose K splits are added
    // inside the kernel (k_decode.hip), whichever the cost model prefers; with the family asked for by name,
    // tile_variant 0 / 1 / 2 / 3 pins the narrow strips / the wide ones of 128, 256, 64 columns.  Under automatic dispatch the family has to hold its own
    // against the best tile plan by cost: with a long K range and many column strips 64x64 tiles with the K
    // range split are faster than the narrow kernel (measured: 12-14 us against 15-20 us for M = 16 / 32,
    // N >= 4608, K = 7168).
    Plan decode{FP8GEMM_KERNEL_SKINNY, 0, 1};
    double decode_us = -1.0;  // >= 0: the decode family is a candidate, at this cost
    const bool narrow_ok = skinny_supports(g), wide_ok = decode_strip_supports(g);
    auto has_room = [&](int ks) { return ks == 1 || (size_t)ks * g.m * g.n * sizeof(float) <= cfg.partial_room; };
    if (selected == FP8GEMM_KERNEL_SKINNY && !narrow_ok && !wide_ok) {
        p.family = -1;
        return p;
    }
    if ((narrow_ok || wide_ok) && (selected == FP8GEMM_KERNEL_SKINNY || selected == FP8GEMM_KERNEL_AUTO)) {
        const int nkb = g.k / 128;
        const bool by_name = selected == FP8GEMM_KERNEL_SKINNY;
        auto valid_split = [&](int ks) { return ks >= 1 && ks <= nkb && (ks - 1) * ((nkb + ks - 1) / ks) < nkb; };
        int forced_ks = 0;
        if (cfg.force_ksplit > 0) {  // every split has to own at least one K block
            forced_ks = cfg.force_ksplit < nkb ? cfg.force_ksplit : nkb;
            while (!valid_split(forced_ks))
                --forced_ks;
        }
        double narrow_us = 1e300, wide_us = 1e300;
        Plan narrow = decode, wide = decode;
        wide.wide = true;
        auto strips64 = [&](int ksplit) {
            Plan strips = wide;
            strips.ksplit = ksplit;
            strips.halves = 0;
            return strips;
        };
        if (by_name && cfg.force_variant == 3 && wide_ok) {  // pins the 64-column strips
            const int ks = forced_ks ? forced_ks : cfg.fused_ok ? decode64_ksplit(g) : 1;
            if (ks <= 1)
                return strips64(1);
            if (ks <= MAX_KSPLIT && cfg.fused_ok && decode_strip_can_split(g, ks, 0))
                return strips64(ks);
            p.family = -1;
            return p;
        }
        if (narrow_ok && !(by_name && cfg.force_variant >= 1)) {
            narrow.ksplit = forced_ks ? forced_ks : skinny_ksplit(g);
            if (!has_room(narrow.ksplit))
                narrow.ksplit = 1;
            narrow_us = skinny_cost(g, narrow.ksplit);
        }
        if (wide_ok && (by_name ? cfg.force_variant != 0 : cfg.force_variant < 0)) {
            // without the in-kernel reduction (no zeroed mailbox, or workgroup placement not confirmed) only
            // the unsplit form exists.  By name, tile_variant 2 pins the 256-column strips.
            // Left to the cost model, 256-column strips have to be 7 % ahead where K is split: they halve the
            // workgroups of a split and win where that saves a round (144 strips x 3 splits are 54 workgroups on
            // an XCD's 32 CUs, 72 x 3 are 27: 18432 x 7168 from HBM 28.6 against 34.6 us), and lose 15 - 40 % on
            // cfg5-sized problems.  Unsplit launches stream, and there the wider strips are ahead throughout (a
            // projection onto a vocabulary with 8 rows, 131072 x 4096: 93.3 against 101.7 us; 16 x 49152 x 4096 in
            // one round of 192 workgroups 39.0 us, against 48.4 us in 384 strips of 128 columns).
            const int hi = cfg.fused_ok ? (nkb < MAX_KSPLIT ? nkb : MAX_KSPLIT) : 1;
            for (int halves = 1; halves <= 2; ++halves) {
                if (by_name ? halves != (cfg.force_variant == 2 ? 2 : 1) : cfg.force_variant >= 0 && halves == 2)
                    continue;
                for (int ks = 1; ks <= hi; ++ks) {
                    if (!valid_split(ks) || (forced_ks && ks != forced_ks) || !decode_strip_can_split(g, ks, halves))
                        continue;
                    const double cst =
                        decode_strip_cost(g, ks, halves) * (halves == 2 && !by_name && ks > 1 ? 1.07 : 1.0);
                    if (cst < wide_us) {
                        wide_us = cst;
                        wide.ksplit = ks;
                        wide.halves = halves;
                    }
                }
            }
        }
        // Decode weights come from HBM (a model's layers do not fit the caches): there the wide strips are
        // ahead of the narrow ones and of every tile plan on all 40 shapes measured (M = 16, 32; N = 1536 ...
        // 16384; K = 1536 ... 7168: 6.0-27 us against 7.3-60 us), although the narrow kernel is 1-2 us faster
        // on short K when B happens to sit in the Infinity Cache.  They need the in-kernel reduction.
        // With more than 32 rows the 64x64 tile plans that add their K splits in the kernel are ahead of the wide
        // strips on 22 of 24 shapes (M = 48, 64; same N and K; from HBM 6.2-15 us against 7.5-16 us): the
        // four-row-tile form is there for grouped launches and runs single problems only when asked for by name.
        // ... except where N x K is large (N = 7168, K >= 4096: 12.2 - 17.4 us against 13.7 - 20.4 us).
        const long long b_bytes = (long long)g.n * g.k;
        if (!by_name && g.m > 32 && g.m % 16 == 0 && !(g.n >= 6144 && b_bytes >= 28000000ll))
            wide_us = 1e300;
        // Row counts off the 16-byte grid, which the strips take as they are: tiles that do so too over a B of up to 16 MB.
        // 66 random shapes of 33 ... 63 rows, N = 288 ... 12912, K = 256 ... 7680: 19 % faster from the Infinity Cache, 13 %
        // from HBM on average.  The line is where the gain with B in the cache and the loss from HBM, where such weights
        // are, meet.  From 12 MB on and with N in whole 128-byte lines (strips of other columns straddle two), tiles of one
        // or two splits are 15 and 7 % ahead from the cache and 7 and 8 % behind from HBM (77 and 43 shapes of 33 ... 47
        // rows; 39 x 7168 x 2048 6.6 us either way and 9.5 against 8.3 us, the worst 47 x 9216 x 1536 6.6 against 6.7 and
        // 11.1 against 8.3 us; with 49 rows and more 21 and 15 % ahead, 4 % behind and level); tiles of more splits 16 and
        // 2 % ahead.  Over 16.5 ... 23.5 MB (8 shapes) tiles are 7 - 35 % ahead from the cache and behind from HBM by 4 % on
        // average and 21 % at worst.  No tiles that need padded copies (12 shapes: 6.8 - 16.9 us against 10.8 - 23.8 us).
        if (!by_name && g.m > 32 && g.m % 16 != 0 && b_bytes < 16000000ll && cfg.force_variant < 0 &&
            cfg.force_ksplit <= 0 && cfg.fused_ok) {
            Config tiles_cfg = cfg;
            tiles_cfg.strips_for_tiles = false;  // decided below for the rows as they are
            const Plan tiles = off_grid_plan(g, tiles_cfg);
            const bool header_only = tiles.ksplit == 1 || tiles.fused;  // as the strips: no partial sums in the workspace
            if (!tiles.padded && header_only && (tiles.family == FP8GEMM_KERNEL_LARGE || tiles.family == FP8GEMM_KERNEL_SPLITK))
                return strips_for_tiles(g, tiles);
        }

        if (!by_name && cfg.force_variant < 0 && cfg.force_ksplit <= 0 && wide_us < 1e300 && cfg.fused_ok) {
            const int ks = wide.halves == 1 ? decode64_ksplit(g) : 0;
            return decode64_pays(g, ks, wide.ksplit) ? strips64(ks) : wide;
        }
        if (!by_name && !cfg.fused_ok)
            wide_us = 1e300;  // unsplit wide strips leave most CUs idle: the narrow kernel and the tile plans compete
        if (narrow_us == 1e300 && wide_us == 1e300) {
            if (by_name) {
                p.family = -1;
                return p;
            }
        } else {
            decode = wide_us < narrow_us ? wide : narrow;
            decode_us = wide_us < narrow_us ? wide_us : narrow_us;
            decode.us = decode_us;
            if (by_name || cfg.force_variant >= 0 || cfg.force_ksplit > 0 || !tile_supports(g))
                return decode;
            // one pass of one round of workgroups: nothing here is faster
            if (decode_us <= skinny_cost(g, 0))
                return decode;
        }
    }
    if (!tile_supports(g)) {
        if (selected != FP8GEMM_KERNEL_AUTO) {
            p.family = -1;
            return p;
        }
        return off_grid_plan(g, cfg);
    }
    const int fv = cfg.force_variant, fk = cfg.force_ksplit;
    const int nkb = g.k / 128;
    if (selected == FP8GEMM_KERNEL_AUTO && fv < 0 && fk <= 0)
        for (const TunedShape& t : kTuned)
            if (t.m == g.m && t.n == g.n && t.k == g.k) {
                p.family = t.ksplit > 1 ? FP8GEMM_KERNEL_SPLITK : FP8GEMM_KERNEL_LARGE;
                p.variant = t.variant;
                p.ksplit = t.ksplit;
                decide_persistent(g, p, cfg);
                decide_fused(g, p, cfg);
                p.us = tile_cost(g, p.variant, p.ksplit, p.fused, cfg.ragged);
                if (!p.fused && !has_room(p.ksplit))
                    break;
                return p;
            }
    double best = 1e300, best_256x128 = 1e300;
    int ks_256x128 = 1;
    for (int v = 0; v < TILE_VARIANT_COUNT; ++v) {
        if (fv >= 0 && v != fv)
            continue;
        if (tile_variant_name(v)[4] == '?')
            continue;
        if (persistent_only(v) && fv != v) {
            // the one-wave-per-SIMD form: only when asked for; the 256x256 tile: when its persistent form can
            // run (a ring's worth of K blocks) and the persistent kernel is not switched off
            if (!persistent_only_auto(v) || cfg.persistent == 0 || !tile_persistent_supports(g, v) ||
                selected == FP8GEMM_KERNEL_SPLITK)
                continue;
        }
        if (g.m <= 64 && fv < 0 && selected == FP8GEMM_KERNEL_AUTO && v != TILE_64x64)
            continue;  // a single row of tiles: taller tiles only multiply rows that do not exist
        for (int ks = 1; ks <= MAX_KSPLIT && ks <= nkb; ++ks) {
            if (persistent_only(v) && ks != 1)
                continue;
            if (fk > 0 && ks != (fk < nkb ? fk : nkb))
                continue;
            if (selected == FP8GEMM_KERNEL_LARGE && ks != 1)
                continue;
            if (selected == FP8GEMM_KERNEL_SPLITK && ks == 1 && nkb > 1)
                continue;
            // every split must own at least one K block
            const int kbs = (nkb + ks - 1) / ks;
            if ((ks - 1) * kbs >= nkb)
                continue;
            // a single row of tiles: the fitted constants overrate a split into short K ranges (measured for
            // M = 16 ... 64: with the reduction kernel the best split never leaves a workgroup fewer than 8 K
            // blocks; with the splits added inside the kernel, never fewer than 3)
            if (g.m <= 64 && fk <= 0 && selected == FP8GEMM_KERNEL_AUTO && ks > 1 &&
                kbs < (tile_plan_fused(g, v, ks, cfg) ? 3 : 8))
                continue;
            // 128x128 tiles that add their splits inside the kernel hand over 64 KB per split: with fewer than 8 K
            // blocks per workgroup that costs more than the split saves (27 shapes with K = 1536, 96 ... 128 tiles,
            // two splits of 6 blocks against unsplit: 10 - 28 % slower with B cached, -2 ... +15 % from HBM)
            if (v == TILE_128x128 && ks > 1 && kbs < 8 && fk <= 0 && selected == FP8GEMM_KERNEL_AUTO &&
                tile_plan_fused(g, v, ks, cfg))
                continue;
            const bool fused = tile_plan_fused(g, v, ks, cfg);
            if (!fused && !has_room(ks))
                continue;
            const double cst = tile_cost(g, v, ks, fused, cfg.ragged);
            if (cst < best) {
                best = cst;
                p.family = ks > 1 ? FP8GEMM_KERNEL_SPLITK : FP8GEMM_KERNEL_LARGE;
                p.variant = v;
                p.ksplit = ks;
            }
            if (v == TILE_256x128 && cst < best_256x128) {
                best_256x128 = cst;
                ks_256x128 = ks;
            }
        }
    }
    if (decode_us >= 0.0 && decode_us <= 0.95 * best)  // measured: at equal estimates the decode kernel is ahead
        return decode;
    if (best == 1e300) {
        p.family = -1;
        return p;
    }
    // 129 ... 1536 rows over a B of 16 MB or more with a long K: 128-row tiles read B twice as often as 256-row
    // tiles.  Where the model takes 128x128 tiles with a 256x128 plan within 12 % of them, that plan -- mostly two
    // to four splits with the reduction kernel -- measures ahead with B cached and with B from HBM: 45 random
    // shapes of up to 256 rows over 32 MB or more all faster, by 12 and 17 % on average; 56 more of up to 512 rows
    // or 18 ... 32 MB with K >= 4096: +8.3 and +6.4 % on average, worst -3.8 % (K = 3072, where an unsplit 128x128
    // plan would give way to three splits, loses 4 - 10 % and is left out); 49 of 528 ... 1536 rows: +7.4 and +6.1 %, worst
    // -3.0 %.  The same where the model takes a 128x192 plan with splits: 56 shapes, +3.6 and +7.4 %, worst -4.6 %.
    if (selected == FP8GEMM_KERNEL_AUTO && fv < 0 && fk <= 0 && (p.variant == TILE_128x128 || p.variant == TILE_128x192) && g.m > 128 && g.m <= 1536 &&
        g.k >= 4096 && (long long)g.n * g.k >= 16000000ll && best_256x128 <= 1.12 * best) {
        p.variant = TILE_256x128;
        p.ksplit = ks_256x128;
        p.family = p.ksplit > 1 ? FP8GEMM_KERNEL_SPLITK : FP8GEMM_KERNEL_LARGE;
    }
    // The same rows where the model takes the 128x192 tile: one row of 256x128 tiles streams B once where the 128x192 tile
    // the fit to cached operands prefers reads it twice.  With B from HBM -- which is what such a B is in a
    // model -- the taller tile is 2 - 13 % ahead on 22 random shapes (208 x 18816 x 3072: +12.8 %), with B in the
    // Infinity Cache -5 ... +4 %; with more rows (two to four tile rows against four to eight) the two are level.
    if (selected == FP8GEMM_KERNEL_AUTO && fv < 0 && fk <= 0 && p.variant == TILE_128x192 && p.ksplit == 1 &&
        g.m <= 256 && (long long)g.n * g.k >= 32000000ll && (g.n + 127) / 128 <= NUM_CU)
        p.variant = TILE_256x128;
    decide_persistent(g, p, cfg);
    decide_fused(g, p, cfg);
    p.us = best;
    if (persistent_only(p.variant) && !p.persistent)
        p.family = -1;
    if (cfg.strips_for_tiles && selected == FP8GEMM_KERNEL_AUTO && fv < 0 && fk <= 0)
        return strips_for_tiles(g, p);
    return p;
}

// The process-wide workspace for a call on `stream` that needs `bytes`: the caller-supplied one, else
// the library-owned one, grown on demand (growth_target).  Growing allocates, which a stream under
// capture does not allow (and which would leave the graph with a buffer it was not recorded with): such
// a call gets FP8GEMM_E_WORKSPACE, and in *at_hand what there is, and the capture stays valid.  An outgrown buffer is
// retired, not freed on the spot: kernels in flight may still use it.
int acquire_workspace(size_t bytes, hipStream_t stream, Workspace* out, size_t* at_hand = nullptr)
{
    std::lock_guard<std::mutex> lock(g_ws_mutex);
    if (at_hand)
        *at_hand = g_ws_user ? g_ws_user_bytes : g_ws_own_bytes;
    if (g_ws_user) {
        if (g_ws_user_bytes < bytes)
            return FP8GEMM_E_WORKSPACE;
        *out = Workspace{g_ws_user, g_ws_user_bytes, g_ws_user_zeroed};
        return FP8GEMM_OK;
    }
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    hipError_t e = hipStreamIsCapturing(stream, &status);
    if (e != hipSuccess)
        return (int)e;
    const bool capturing = status != hipStreamCaptureStatusNone;
    if (g_ws_own_bytes < bytes) {
        if (capturing)
            return FP8GEMM_E_WORKSPACE;
        // retired buffers whose last use has completed go back to the allocator now
        for (size_t i = 0; i < g_ws_retired.size();) {
            Retired& r = g_ws_retired[i];
            if (!r.pinned && hipEventQuery(r.done) == hipSuccess) {
                (void)hipEventDestroy(r.done);
                (void)hipFree(r.ptr);
                g_ws_retired.erase(g_ws_retired.begin() + (long)i);
            } else {
                ++i;
            }
        }
        (void)hipGetLastError();  // hipEventQuery reports "not ready" as an error
        size_t want = growth_target(g_ws_own_bytes, bytes);
        void* p = nullptr;
        e = hipMalloc(&p, want);
        if (e != hipSuccess && want > bytes) {
            (void)hipGetLastError();
            want = bytes;
            e = hipMalloc(&p, want);
        }
        if (e != hipSuccess)
            return (int)e;
        e = hipMemset(p, 0, WS_HEADER);  // the mailbox (bytes >= WS_HEADER whenever a plan needs a workspace)
        if (e != hipSuccess) {
            (void)hipFree(p);
            return (int)e;
        }
        if (g_ws_own) {
            Retired r{g_ws_own, nullptr, g_ws_own_captured};
            if (!r.pinned) {
                if (hipEventCreateWithFlags(&r.done, hipEventDisableTiming) != hipSuccess ||
                    hipEventRecord(r.done, g_ws_last_stream) != hipSuccess) {
                    (void)hipGetLastError();
                    if (r.done)
                        (void)hipEventDestroy(r.done);
                    r.done = nullptr;
                    r.pinned = true;  // no way to tell when its last use ends: kept until release
                }
            }
            g_ws_retired.push_back(r);
        }
        g_ws_own = static_cast<float*>(p);
        g_ws_own_bytes = want;
        g_ws_own_captured = false;
    }
    g_ws_own_captured = g_ws_own_captured || capturing;
    g_ws_last_stream = stream;
    *out = Workspace{g_ws_own, g_ws_own_bytes, true};
    return FP8GEMM_OK;
}

// bytes of partial sums a plan keeps behind the workspace header
size_t plan_workspace_bytes(const GemmArgs& g, const Plan& p)
{
    // splits that are added inside the kernel meet in the header
    if (p.ksplit <= 1 || (p.family == FP8GEMM_KERNEL_SKINNY && p.wide) || p.fused)
        return 0;
    return (size_t)p.ksplit * g.m * g.n * sizeof(float);
}
// whether a plan uses the header although it keeps nothing behind it
inline bool plan_uses_header(const Plan& p) { return p.ksplit > 1 && ((p.family == FP8GEMM_KERNEL_SKINNY && p.wide) || p.fused); }
// a workspace that holds `data` bytes of a plan: nothing, or the header and the data
inline size_t with_header(size_t data, bool header_alone = false) { return data || header_alone ? data + WS_HEADER : 0; }

void plan_name(const Plan& p, char* out, size_t cap)
{
    const char* pre = p.padded ? "padded_" : "";
    if (p.family == FP8GEMM_KERNEL_SCALAR)
        snprintf(out, cap, "scalar");
    else if (p.family == FP8GEMM_KERNEL_SKINNY)
        snprintf(out, cap, p.wide ? (p.halves == 2 ? "%sdecode256_k%d" : p.halves == 0 ? "%sdecode64_k%d" : "%sdecode128_k%d") : "%sskinny_k%d", pre, p.ksplit);
    else
        snprintf(out, cap, "%s%s_k%d%s", pre, tile_variant_name(p.variant), p.ksplit,
                 p.persistent ? "_persistent" : (p.fused ? "f" : ""));
}

// The thread's last launch by name; a plan's is put together when somebody asks (0.06 us of a call).
thread_local Plan t_last_plan;
thread_local bool t_plan_unnamed = false;  // t_last_plan is newer than t_last_kernel
const char* last_kernel_name()
{
    if (t_plan_unnamed) {
        plan_name(t_last_plan, t_name_buf, sizeof(t_name_buf));
        t_last_kernel = t_name_buf;
        t_plan_unnamed = false;
    }
    return t_last_kernel;
}

// the kernels of a plan on operands they can take; `partial` holds plan_workspace_bytes, `w` is the
// workspace whose zeroed header the plans use that add their K splits inside the kernel
hipError_t launch_plan(const GemmArgs& g, const Plan& p, float* partial, const Workspace& w, hipStream_t stream)
{
    switch (p.family) {
    case FP8GEMM_KERNEL_SCALAR:
        return launch_scalar(g, stream);
    case FP8GEMM_KERNEL_SKINNY:
        if (p.wide)
            return launch_decode_strips(g, p.ksplit, p.halves, ws_mailbox(w), stream);
        return launch_skinny(g, p.ksplit, partial, stream);
    default: {
        if (p.persistent)
            return launch_tile_persistent(g, p.variant, NUM_CU, stream);
        hipError_t e = launch_tile(g, p.variant, p.ksplit, partial, p.fused ? ws_mailbox(w) : nullptr, stream);
        if (e == hipSuccess && p.ksplit > 1 && !p.fused)
            e = launch_splitk_reduce(g, p.ksplit, partial, stream);
        return e;
    }
    }
}

// pad what needs padding into the workspace, run the plan there, copy C's corner out
// bytes run_padded needs for this call (depends on which operands are off the grid)
size_t padded_bytes(const GemmArgs& g, const Plan& p)
{
    GemmArgs gp = g;
    gp.m = (g.m + 15) & ~15;
    gp.n = (g.n + 15) & ~15;
    const bool keeps_rows = p.family == FP8GEMM_KERNEL_LARGE || p.family == FP8GEMM_KERNEL_SPLITK ||
                            (p.family == FP8GEMM_KERNEL_SKINNY && p.wide);
    return with_header(pad_layout(g, plan_workspace_bytes(gp, p), false, keeps_rows).total, plan_uses_header(p));
}

int run_padded(const GemmArgs& g, const Plan& p, const Workspace& w, hipStream_t stream)
{
    GemmArgs gp = g;
    const int m16 = (g.m + 15) & ~15;
    gp.m = m16;
    gp.n = (g.n + 15) & ~15;
    const bool keeps_rows = p.family == FP8GEMM_KERNEL_LARGE || p.family == FP8GEMM_KERNEL_SPLITK ||
                            (p.family == FP8GEMM_KERNEL_SKINNY && p.wide);
    const PadLayout L = pad_layout(g, plan_workspace_bytes(gp, p), false, keeps_rows);
    if (!L.c) {  // c is written in place: its m rows, while a and a_scale have m16 per k-row
        gp.m = g.m;
        gp.lda = m16;
    }
    if (!w.ptr || w.bytes < with_header(L.total))
        return FP8GEMM_E_WORKSPACE;
    uint8_t* base = reinterpret_cast<uint8_t*>(ws_data(w));
    const int nkb = g.k / 128;
    // every operand that needs a padded copy, in one launch
    PadJobs<PAD_JOBS_SINGLE> jobs;
    jobs.base = base;
    if (L.a) {
        jobs.add(g.a, L.off_a, g.k, g.m, m16);
        gp.a = base + L.off_a;
    }
    if (L.as) {
        jobs.add(g.a_scale, L.off_as, nkb, (size_t)g.m * 4, (size_t)m16 * 4);
        gp.a_scale = reinterpret_cast<float*>(base + L.off_as);
    }
    if (L.b) {
        jobs.add(g.b, L.off_b, g.k, g.n, gp.n);
        gp.b = base + L.off_b;
    }
    hipError_t e = launch_pad(jobs, stream);
    if (L.c)
        gp.c = reinterpret_cast<uint16_t*>(base + L.off_c);
    if (e == hipSuccess)
        e = launch_plan(gp, p, reinterpret_cast<float*>(base + L.off_partial), w, stream);
    if (e == hipSuccess && L.c)
        e = launch_crop_bf16(gp.c, g.c, g.m, g.n, gp.n, stream);
    return (int)e;
}

// bytes of workspace that a call needs under a plan
size_t call_bytes(const GemmArgs& g, const Plan& p)
{
    return p.padded ? padded_bytes(g, p) : with_header(plan_workspace_bytes(g, p), plan_uses_header(p));
}

// The plan of a call whose workspace of `at_hand` bytes is too small for `p`, automatic dispatch's choice: the cheapest one
// whose partial sums find room in it, if that is next to as fast; else p, which the caller is told to bring a workspace
// for.  Which of two plans level with each other the estimates prefer thus does not decide whether a call runs at all (639 x
// 4608 x 7168: 128x192 tiles in two splits, 38 MiB, or 128x128 unsplit and no workspace).  The line: a new fit of the estimates
// had taken the plan that ran without a workspace, or within the fixed array, from 470 of 54 000 problems (the projections of
// the table with 16 ... 3199 rows, and random ones); all have one back from 1.08 on, all but three from 1.05 on.  Further up, calls would run that much slower where a workspace helps.
constexpr double FITTING_PLAN_WITHIN = 1.10;
Plan fitting_plan(const GemmArgs& g, const Plan& p, Config cfg, size_t at_hand)
{
    if (p.family < 0 || cfg.selected != FP8GEMM_KERNEL_AUTO || cfg.force_variant >= 0 || cfg.force_ksplit > 0 || cfg.fused_mode == 1)
        return p;
    GemmArgs gp = g;
    if (p.padded) {
        gp.m = (g.m + 15) & ~15;
        gp.n = (g.n + 15) & ~15;
    }
    const size_t partial = plan_workspace_bytes(gp, p), rest = call_bytes(g, p) - partial;
    for (;; cfg.fused_ok = false) {  // (splits added inside the kernel need the header)
        for (const size_t taken : {WS_HEADER, rest}) {  // room beside no copies, which p may need and another plan not, and beside p's
            cfg.partial_room = at_hand > taken ? at_hand - taken : 0;
            const Plan fit = make_plan(g, cfg);
            if (fit.family >= 0 && call_bytes(g, fit) <= at_hand && fit.us <= FITTING_PLAN_WITHIN * p.us)
                return fit;
        }
        if (!cfg.fused_ok)
            return p;
    }
}

// Whether plans that add their K splits inside the kernel may run for a call on `stream`: the device
// must place workgroups on XCDs as those kernels assume.  The first call on a device finds out with a
// probe grid that it waits for; while `stream` is being captured nothing is probed and an unknown
// placement counts as "no".
bool placement_ok(hipStream_t stream)
{
    int known = xcd_placement_confirmed(false);
    if (known >= 0)
        return known == 1;
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &status) != hipSuccess || status != hipStreamCaptureStatusNone)
        return false;
    return xcd_placement_confirmed(true) == 1;
}

// One GEMM.  explicit_ws = the caller's per-call workspace (its bytes may be 0 / its pointer NULL when the
// plan needs none); nullptr = the process-wide workspace.
int run(const void* a, const void* b, const float* as, const float* bs, void* c, int m, int n, int k,
        hipStream_t stream, Config cfg, const Workspace* explicit_ws)
{
    int v = validate(a, b, as, bs, c, m, n, k);
    if (v != FP8GEMM_OK)
        return v;
    GemmArgs g{static_cast<const uint8_t*>(a), static_cast<const uint8_t*>(b), as, bs,
               static_cast<uint16_t*>(c), m, n, k};
    // in-kernel K-split reduction: a zeroed header (every process-wide workspace has one; a per-call
    // one when the caller says so) and a confirmed workgroup placement
    cfg.fused_ok = cfg.fused_ok && (!explicit_ws || explicit_ws->zeroed);
    if (cfg.fused_ok && xcd_placement_confirmed(false) != 1) {  // not known yet, or not as they assume
        Config probe = cfg;
        probe.fused_ok = false;
        const Plan with = make_plan(g, cfg), without = make_plan(g, probe);
        const bool differs = with.family != without.family || with.ksplit != without.ksplit ||
                             with.wide != without.wide || with.fused != without.fused || with.halves != without.halves;
        if (differs && !placement_ok(stream))
            cfg.fused_ok = false;
    }
    Plan p = make_plan(g, cfg);
    if (p.family < 0)
        return FP8GEMM_E_KERNEL;
    Workspace w{nullptr, 0, false};
    bool fitted = false;
    for (int attempt = 0;; ++attempt) {
        const size_t need = call_bytes(g, p);
        int rc = FP8GEMM_OK;
        size_t at_hand = 0;
        if (need) {
            if (explicit_ws) {
                if (!explicit_ws->ptr || explicit_ws->bytes < need ||
                    (reinterpret_cast<uintptr_t>(explicit_ws->ptr) % 256) != 0)
                    rc = FP8GEMM_E_WORKSPACE;
                else
                    w = *explicit_ws;
                at_hand = explicit_ws->ptr && (reinterpret_cast<uintptr_t>(explicit_ws->ptr) % 256) == 0 ? explicit_ws->bytes : 0;
            } else {
                rc = acquire_workspace(need, stream, &w, &at_hand);
            }
        }
        if (rc == FP8GEMM_OK)
            break;
        // A plan that adds its K splits inside the kernel needs the header; when the workspace at hand cannot
        // hold it (a small caller-owned buffer, or none while the stream is being captured) the plan without
        // it may still run -- cfg1-like shapes then need no workspace at all.  Not when that form was asked for.  Then one
        // that finds room (fitting_plan).
        if (rc != FP8GEMM_E_WORKSPACE || fitted)
            return rc;
        if (attempt == 0 && cfg.fused_ok && cfg.fused_mode != 1 && plan_uses_header(p)) {
            cfg.fused_ok = false;
            p = make_plan(g, cfg);
        } else {
            cfg.fused_ok = cfg.fused_ok && placement_ok(stream);  // (not asked where p needs no more than the plan without it)
            p = fitting_plan(g, p, cfg, at_hand);
            if (call_bytes(g, p) > at_hand)
                return rc;
            fitted = true;
        }
        if (p.family < 0)
            return FP8GEMM_E_WORKSPACE;
    }
    const int rc = p.padded ? run_padded(g, p, w, stream) : (int)launch_plan(g, p, ws_data(w), w, stream);
    if (rc == FP8GEMM_OK) {
        t_last_plan = p;
        t_plan_unnamed = true;
    }
    return rc;
}

// ---- the entry point that allocates nothing: its workspace is this array, part of the library's device
// image (every GPU the library runs on holds its own copy, at its own address, until the process
// ends).  In host code the array's name is only a handle for hipGetSymbolAddress: the device address is
// looked up once per device, with that device current, and everything else uses that pointer.
static __device__ __align__(256) unsigned char scratch[FP8GEMM_NOALLOC_MAX_BYTES];

constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[MAX_DEVICES] = {};

int scratch_for_current_device(void** out)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess)
        return (int)e;
    if (dev < 0 || dev >= MAX_DEVICES)
        return (int)hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess)
            return (int)e;
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return FP8GEMM_OK;
}

// the tiles of a grouped launch: every group starts a tile row of its own
long grouped_tiles(const GroupTable& tab, int n, int variant)
{
    int bm, bn;
    tile_variant_dims(variant, &bm, &bn);
    long rows = 0;
    for (int g = 0; g < tab.groups; ++g)
        rows += (tab.m[g] + bm - 1) / bm;
    return rows * ((n + bn - 1) / bn);
}

// Estimated run time of a grouped tile launch in microseconds: tile_cost's form -- launch + rounds of 256
// workgroups x (fill + K blocks + store) -- on the launch's own tile count, with a K block priced for operands
// that come from HBM: every group brings its own B, and a tile row of a group reads all of it, so the launch
// moves more bytes per flop than the single problems tile_cost was fitted on, the more the smaller the tile.
// Factors on the K block from 25 launches (1 ... 64 groups of 65 ... 3000 rows, N = 1536 ... 7168, K = 2048 and
// 7168, every tile shape pinned): 1.2 for 256x256, 1.43 for 256x192, 1.5 for 256x128, 1.7 for 128x192 and 128x128; the
// first two have since got 5 % faster, which is in the factors and not in these figures --
// e.g. 8 groups of 300 ... 3000 rows, 4608 x 7168: 498 / 610 / 680 / 775 / 893 us estimated for 256x256 / 256x192 /
// 256x128 / 128x192 / 128x128, 515 / 615 / 727 / 875 / 1042 us measured; 4 groups of 65 ... 256 rows, 7168 x 2048:
// 35 / 34 / 26 / 46 / 37 us estimated, 32 / 33 / 25 / 42 / 36 us measured.
double grouped_tile_cost(const GroupTable& tab, int n, int k, int variant)
{
    int bm, bn;
    tile_variant_dims(variant, &bm, &bn);
    const double area = (double)bm * bn / 65536.0;
    if (variant == TILE_256x256)
        return large_tile_cost(grouped_tiles(tab, n, variant), k, 1.2);
    const long tiles = grouped_tiles(tab, n, variant);
    // 128x256 tiles where they are no more than tiles of 256x256 would be, which is where no group has more than 128 rows: half
    // of A's slots go to a third stage, more of B is on its way (19 launches of up to 128 rows a group 0.2 - 15 % ahead of 256x256,
    // 10 % on average).  Where they are more it is open, 15 of 25 with 1.08 to 1.65 times as many behind by up to 50 %.
    if (variant == TILE_128x256) {
        const int nkb = k / 128;
        if (nkb < 3 || tiles != grouped_tiles(tab, n, TILE_256x256))
            return 1e300;
        const bool tail = large_tile_tail(tiles, k, NUM_CU) != Tail::NONE;
        const long whole = tail ? tiles / NUM_CU : (tiles + NUM_CU - 1) / NUM_CU;
        return 1.79 + (double)whole * 0.89 * (4.5 + nkb * 1.6) + (tail ? 3.0 + nkb * 0.7 : 0.0);
    }
    // (256x192 tiles in a single round, where 256x256 tiles are fewer still: 18 of 20 random launches are 1 - 13 % faster in
    // the smaller ones and two 1 % slower, 384 - 624 rows, 4960 x 1664, 140 or 182 tiles, 25.3 / 22.3 us, 16 of 96 - 656, 1232 x
    // 1792, 28.3 / 24.9, six of 80 - 336, 4608 x 7168, 93.1 / 88.3; and fewer of them are too few for one launch, below)
    const double from_hbm = variant == TILE_256x192 ? (tiles <= NUM_CU ? 1.32 : 1.43) : bm == 256 ? 1.5 : 1.7;
    const double per_kb = (1.19 * area + 0.267) * from_hbm;
    const double per_item = 0.95 + 4.38 * area + (k / 128) * per_kb;
    const long rounds = (tiles + NUM_CU - 1) / NUM_CU;
    return 1.79 + rounds * per_item;
}

// tile shape for a grouped launch: the cheapest by grouped_tile_cost among the shapes that have a grouped form
// (no K split); -1 when none can take the table
int grouped_variant(const GroupTable& tab, int n, int k, const Config& cfg)
{
    long long m_total = 0;
    for (int g = 0; g < tab.groups; ++g)
        m_total += tab.m[g];
    if (m_total > 0x7FFFFFFFll)
        return -1;
    int best_v = -1;
    double best = 1e300;
    const int fv = cfg.force_variant;
    for (int v = 0; v <= TILE_128x256; ++v) {
        if ((fv >= 0 && v != fv) || !tile_grouped_supports(tab, n, k, v))
            continue;
        if (fv < 0 && persistent_only(v) && !persistent_only_auto(v))
            continue;
        const double cst = grouped_tile_cost(tab, n, k, v);
        if (cst < best) {
            best = cst;
            best_v = v;
        }
    }
    return best_v;
}

// the workspace of a call: the caller's per-call one, else the process-wide one
int workspace_for(size_t need, hipStream_t stream, const Workspace* explicit_ws, Workspace* out)
{
    *out = Workspace{nullptr, 0, false};
    if (!need)
        return FP8GEMM_OK;
    if (explicit_ws) {
        if (!explicit_ws->ptr || explicit_ws->bytes < need || (reinterpret_cast<uintptr_t>(explicit_ws->ptr) % 256) != 0)
            return FP8GEMM_E_WORKSPACE;
        *out = *explicit_ws;
        return FP8GEMM_OK;
    }
    return acquire_workspace(need, stream, out);
}

constexpr int GROUPED_NOT_APPLICABLE = -1000;

// A grouped launch of the persistent kernels that leaves a third of the CUs without a tile while each tile walks a long K
// range is not made: single problems split K (one group of 200 x 4096 x 7168: 19 us against 52 us, two: 42 against 56 us;
// four groups of 1536 x 7168: level; with K = 2048 one group 13.4 against 15.6 us, two 26 against 19 us).
bool grouped_leaves_cus_idle(const GroupTable& tab, int n, int k, int variant)
{
    return tab.groups <= 8 && k >= 2048 && grouped_tiles(tab, n, variant) < 160;
}

// What the persistent kernels take for a grouped launch of tall groups: their cheapest shape, and the copies of A into
// padded rows; no end where they would not run it.
double grouped_persistent_cost(const GroupTable& tab, int n, int k)
{
    double best = 1e300;
    int variant = -1;
    for (int v = 0; v <= TILE_128x256; ++v) {
        if (v == TILE_64x64 || (persistent_only(v) && !persistent_only_auto(v)))
            continue;
        const double cost = grouped_tile_cost(tab, n, k, v);
        if (cost < best)
            best = cost, variant = v;
    }
    if (grouped_leaves_cus_idle(tab, n, k, variant))
        return 1e300;
    double copied = 0;
    for (int g = 0; g < tab.groups; ++g)
        copied += tab.m[g] % 16 != 0 ? 2.0 * tab.m[g] * k : 0.0;
    return best + (copied > 0 ? 2.9 + copied / 4.5e6 : 0.0);
}

// What a tile of 64x64 or 128x128 per workgroup takes, us: launch, rounds of 256 workgroups (two small ones share a CU, so a
// round begun is not a whole one) x (start and store + K blocks), the hand-over of K splits, and the operands' way.  Fitted
// to 784 plans of 220 random grouped launches (2 - 64 groups of 65 - 2048 rows, 256 ... 8192 x 256 ... 7168, three quarters
// off the row grid, three sets of operands in turn), which it reproduces within 8.5 % (standard deviation).
double grouped_each_cost(const GroupTable& tab, int n, int k, int variant, int ksplit, bool ragged)
{
    const bool small = variant == TILE_64x64;
    const long tiles = grouped_tiles(tab, n, variant);
    const long items = (ksplit > 1 ? (tiles + 7) / 8 * 8 : tiles) * ksplit, rounds = (items + NUM_CU - 1) / NUM_CU;
    const int blocks = (k / 128 + ksplit - 1) / ksplit;
    double m = 0;
    for (int g = 0; g < tab.groups; ++g)
        m += tab.m[g];
    const double megabytes = (m * k + (double)tab.groups * n * k + 2.0 * m * n) * 1e-6;
    const double handed = ksplit - 1;
    if (small) {
        const double turns = rounds > 1 ? 0.66 * (double)rounds + 0.34 * (double)items / NUM_CU : 1.0;
        return 2.8 + turns * (0.93 + blocks * (ragged ? 0.4 : 0.35)) + (ksplit > 1 ? 0.57 + 0.4 * handed : 0.0) + 0.02 * megabytes;
    }
    return 1.4 + (double)rounds * (3.3 + blocks * (ragged ? 0.6 : 0.42) * (n % 128 ? 1.06 : 1.0)) +
           (ksplit > 1 ? 1.0 + 1.67 * handed : 0.0) + 0.11 * megabytes;
}

struct EachPlan { int variant; int ksplit; double cost; };
EachPlan grouped_each_plan(const GroupTable& tab, int n, int k, const Config& cfg, bool can_split, bool ragged)
{
    const int nkb = k / 128;
    EachPlan best{-1, 1, 1e300};
    for (const int v : {TILE_64x64, TILE_128x128}) {
        if (cfg.force_variant >= 0 && v != cfg.force_variant)
            continue;
        const size_t mail = (size_t)grouped_tiles(tab, n, v) * (v == TILE_64x64 ? 1 : 4) * 16384;
        for (int ks = 1; ks <= (v == TILE_64x64 ? 8 : 3); ++ks) {
            if (cfg.force_ksplit > 0 && can_split && ks != cfg.force_ksplit)
                continue;
            // (off the row grid, where A comes through registers, not over a hundred K blocks for a CU: six groups of 3741 rows,
            // 1536 x 7168, 79.7 us with copies and 256x128 tiles, 91.3 with 128x128; 35 of 27064, 576 x 7168, 243 / 246)
            const long items = grouped_tiles(tab, n, v) * ks;
            if (ragged && cfg.force_variant < 0 && (items + NUM_CU - 1) / NUM_CU * ((nkb + ks - 1) / ks) > 100)
                continue;
            if (ks > 1 && (!can_split || (ks - 1) * ((nkb + ks - 1) / ks) >= nkb || mail * (ks - 1) > SPLIT_MAILBOX_BYTES))
                continue;
            const double cost = grouped_each_cost(tab, n, k, v, ks, ragged);
            if (cost < best.cost)
                best = EachPlan{v, ks, cost};
        }
    }
    return best;
}

// Tall groups with a tile of 64x64 or 128x128 per workgroup (launch_tile_each): A's rows as they are, K split where the
// tiles are few.  Against the persistent kernels behind copies of A into padded rows, or the groups one by one, where the
// estimates have it ahead: the 220 launches above 21 % faster in the geometric mean, none slower by more than 1 % (three groups
// of 705 rows, 448 x 5632, one by one 27.0 us, now 14.0; 31 of 65 - 180, 576 x 7168, 72.9 / 34.1; four of 4608 x 2304 59.6 / 26.3;
// 14 of 528 x 640 14.9 / 9.5).  N < 256 is not measured and stays.  A pinned shape comes here with persistent = 0.
int run_grouped_each(GroupTable tab, int n, int k, hipStream_t s, const Config& cfg, const Workspace* explicit_ws)
{
    const bool pinned = cfg.force_variant >= 0;
    bool ragged;
    if (n < 256 || cfg.persistent == 1 || (pinned ? cfg.persistent != 0 : cfg.force_ksplit > 0) ||
        !tile_each_supports(tab, n, k, pinned ? cfg.force_variant : TILE_64x64, &ragged))
        return GROUPED_NOT_APPLICABLE;
    const double other = pinned ? 1e300 : grouped_persistent_cost(tab, n, k);
    const bool one_by_one = !pinned && other == 1e300;  // there, single problems may split K with the reduction kernel
    bool can_split = cfg.fused_ok && cfg.fused_mode != 0 && (!explicit_ws || explicit_ws->zeroed);
    // Splits meet in the workspace, and calls that share the process-wide one must not overlap on two streams.  Groups that
    // need none of it otherwise -- on the row grid in one launch, or each by itself in an unsplit plan -- stay without.
    if (!explicit_ws && !pinned && can_split) {
        bool shares = ragged && !one_by_one;
        for (int g = 0; g < tab.groups && one_by_one && !shares; ++g) {
            const GemmArgs ga{tab.a[g], tab.b[g], tab.a_scale[g], tab.b_scale[g], tab.c[g], tab.m[g], n, k, tab.lda[g]};
            shares = call_bytes(ga, make_plan(ga, cfg)) > 0;
        }
        can_split = shares;
    }
    EachPlan p{-1, 1, 1e300};
    Workspace w{nullptr, 0, false};
    for (;; can_split = false) {
        p = grouped_each_plan(tab, n, k, cfg, can_split, ragged);
        if (p.variant < 0 || p.cost >= other || (one_by_one && !can_split))
            return GROUPED_NOT_APPLICABLE;
        if (p.ksplit == 1)
            break;
        if (!placement_ok(s))
            continue;
        const int rc = workspace_for(with_header(0, true), s, explicit_ws, &w);
        if (rc == FP8GEMM_OK)
            break;
        if (rc != FP8GEMM_E_WORKSPACE)  // an error of the runtime's, as from a single problem
            return rc;
    }
    const hipError_t e = launch_tile_each(tab, n, k, p.variant, p.ksplit, p.ksplit > 1 ? ws_mailbox(w) : nullptr, s);
    if (e == hipSuccess) {
        snprintf(t_name_buf, sizeof(t_name_buf), "%s_k%d%s_grouped%d", tile_variant_name(p.variant), p.ksplit,
                 p.ksplit > 1 ? "f" : "", tab.groups);
        t_last_kernel = t_name_buf;
        t_plan_unnamed = false;
    }
    return (int)e;
}

// One grouped launch for the problems of `tab` (same n and k): the decode kernel when every group has at
// most 64 rows (decode = true), else a tile kernel (run_grouped_each, or the persistent one).  For the latter, groups off the 16-byte grid (n, or for the
// tile kernel m, not a multiple of 16; an operand off a 16-byte boundary) run on zero-padded copies in the
// workspace: one launch for those of a and a_scale, one each for b and c where they need it.  Returns GROUPED_NOT_APPLICABLE when it cannot run (the caller
// then takes the groups one by one).
int run_grouped_table(const GroupTable& tab, int n, int k, bool decode, hipStream_t s, const Config& cfg,
                      const Workspace* explicit_ws)
{
    if (!decode) {
        const int rc = run_grouped_each(tab, n, k, s, cfg, explicit_ws);
        if (rc != GROUPED_NOT_APPLICABLE)
            return rc;
    }
    const long long lim = 0x7FFFFFFFll;
    const int n16 = (n + 15) & ~15;
    const size_t nkb = (size_t)k / 128;
    bool pad_a = false, pad_b = n16 != n, pad_c = n16 != n;
    // The decode kernel takes row counts off the 16-byte grid as they are (it spreads A's packed slabs in the
    // LDS) and 4-byte aligned scales: measured on 2 to 64 groups of 1 - 64 rows, N = 1536 ... 7168, K = 2048 and
    // 7168, level with the padded copies (one more launch, then the plain kernel) or up to 20 % ahead.  Launches
    // large enough for the streaming form, which wants rows on the grid, are the exception: 9 % for one copy launch.
    const bool streams = decode && decode_grouped_streams(tab.groups, n16);
    for (int g = 0; g < tab.groups; ++g) {
        pad_a = pad_a || misaligned16(tab.a[g]) || (tab.m[g] % 16 != 0 && (!decode || streams)) ||
                (!decode && misaligned16(tab.a_scale[g]));
        pad_b = pad_b || misaligned16(tab.b[g]);
        pad_c = pad_c || misaligned16(tab.c[g]);
    }
    const bool padded = pad_a || pad_b || pad_c;
    size_t off_a[GroupTable::MAX_GROUPS], off_as[GroupTable::MAX_GROUPS], off_b[GroupTable::MAX_GROUPS],
        off_c[GroupTable::MAX_GROUPS];
    size_t off = 0;
    if (padded)
        for (int g = 0; g < tab.groups; ++g) {
            const long long m16 = (tab.m[g] + 15) & ~15;
            if (m16 * k > lim || (long long)n16 * k > lim || m16 * n16 > lim)
                return GROUPED_NOT_APPLICABLE;
            off_a[g] = off;
            off += round256((size_t)k * m16);
            off_as[g] = off;
            off += round256(nkb * m16 * sizeof(float));
            off_b[g] = off;
            off += pad_b ? round256((size_t)k * n16) : 0;
            off_c[g] = off;
            off += pad_c ? round256((size_t)m16 * n16 * 2) : 0;
        }
    // the problems as the GEMM kernel sees them (addresses in the workspace are filled in below): c in place
    // keeps its m rows, a and a_scale have m16 per k-row
    GroupTable pt = tab;
    if (padded)
        for (int g = 0; g < tab.groups; ++g) {
            const int m16 = (tab.m[g] + 15) & ~15;
            pt.m[g] = pad_c ? m16 : tab.m[g];
            pt.lda[g] = m16;
        }
    // decode kernel: K split by cost (it needs the zeroed mailbox and the XCD placement); tile kernel: none
    int ksplit = 1;
    int variant = -1;
    if (decode) {
        // placeholder addresses that pass the alignment checks while the real ones are not known yet
        GroupTable probe = pt;
        if (padded)
            for (int g = 0; g < tab.groups; ++g) {
                probe.a[g] = reinterpret_cast<const uint8_t*>(uintptr_t(4096));
                probe.a_scale[g] = reinterpret_cast<const float*>(uintptr_t(4096));
                if (pad_b)
                    probe.b[g] = reinterpret_cast<const uint8_t*>(uintptr_t(4096));
                if (pad_c)
                    probe.c[g] = reinterpret_cast<uint16_t*>(uintptr_t(4096));
            }
        if (!decode_grouped_supports(probe, n16, k))
            return GROUPED_NOT_APPLICABLE;
        bool fused_ok = cfg.fused_ok && (!explicit_ws || explicit_ws->zeroed);
        if (fused_ok && decode_grouped_ksplit(pt, n16, k, true) > 1)
            fused_ok = placement_ok(s);
        ksplit = cfg.force_ksplit > 0 && fused_ok ? cfg.force_ksplit : decode_grouped_ksplit(pt, n16, k, fused_ok);
        const int nkb_i = k / 128;
        while (ksplit > 1 && (ksplit > nkb_i || (ksplit - 1) * ((nkb_i + ksplit - 1) / ksplit) >= nkb_i))
            --ksplit;
        if (decode_grouped_mailbox_bytes(pt, n16, ksplit) > SPLIT_MAILBOX_BYTES)
            ksplit = 1;
    }
    Workspace w;
    const int wrc = workspace_for(with_header(off, ksplit > 1), s, explicit_ws, &w);
    if (wrc == FP8GEMM_E_WORKSPACE)
        return GROUPED_NOT_APPLICABLE;  // a workspace sized for single problems: one by one
    if (wrc != FP8GEMM_OK)
        return wrc;
    uint8_t* base = reinterpret_cast<uint8_t*>(ws_data(w));
    PadJobs<PAD_JOBS_GROUPED> jobs;
    CropTable tc;
    jobs.base = base;
    tc.groups = tab.groups, tc.n = n, tc.ld_src = n16;
    if (padded)
        for (int g = 0; g < tab.groups; ++g) {
            const int m = tab.m[g], m16 = (m + 15) & ~15;
            // a group that lies on the grid by itself stays where it is
            if (m16 != m || misaligned16(tab.a[g]) || misaligned16(tab.a_scale[g])) {
                jobs.add(tab.a[g], off_a[g], k, m, m16);
                jobs.add(tab.a_scale[g], off_as[g], nkb, (size_t)m * 4, (size_t)m16 * 4);
                pt.a[g] = base + off_a[g];
                pt.a_scale[g] = reinterpret_cast<const float*>(base + off_as[g]);
            }
            pt.b[g] = pad_b ? base + off_b[g] : tab.b[g];
            pt.c[g] = pad_c ? reinterpret_cast<uint16_t*>(base + off_c[g]) : tab.c[g];
            tc.src[g] = base + off_c[g], tc.dst[g] = tab.c[g], tc.m[g] = m;
        }
    if (!decode) {
        variant = grouped_variant(pt, n16, k, cfg);
        if (variant < 0)
            return GROUPED_NOT_APPLICABLE;
        if (cfg.force_variant < 0 && grouped_leaves_cus_idle(pt, n16, k, variant))
            return GROUPED_NOT_APPLICABLE;
    }
    hipError_t e = hipSuccess;
    if (padded) {
        e = launch_pad(jobs, s);
        if (e == hipSuccess && pad_b) {
            jobs.count = 0;
            for (int g = 0; g < tab.groups; ++g)
                jobs.add(tab.b[g], off_b[g], k, n, n16);
            e = launch_pad(jobs, s);
        }
    }
    if (e == hipSuccess)
        e = decode ? launch_decode_grouped(pt, n16, k, ksplit, ws_mailbox(w), s)
                   : launch_tile_grouped(pt, n16, k, variant, NUM_CU, s);
    if (e == hipSuccess && pad_c)
        e = launch_crop_bf16_batched(tc, s);
    if (e == hipSuccess) {
        if (decode)
            snprintf(t_name_buf, sizeof(t_name_buf), "%sdecode128_k%d_grouped%d", padded ? "padded_" : "", ksplit, tab.groups);
        else
            snprintf(t_name_buf, sizeof(t_name_buf), "%s%s_k1_grouped%d", padded ? "padded_" : "", tile_variant_name(variant),
                     tab.groups);
        t_last_kernel = t_name_buf;
        t_plan_unnamed = false;
    }
    return (int)e;
}

// nullptr = automatic dispatch; rc = FP8GEMM_OK when the options are usable
Config config_from_options(const fp8gemm_options* opt, int* rc)
{
    *rc = FP8GEMM_OK;
    if (!opt)
        return Config{FP8GEMM_KERNEL_AUTO, -1, 0, -1};
    if (opt->kernel < FP8GEMM_KERNEL_AUTO || opt->kernel > FP8GEMM_KERNEL_SKINNY ||
        opt->tile_variant >= TILE_VARIANT_COUNT || opt->ksplit < 0 || opt->ksplit > MAX_KSPLIT ||
        opt->persistent < -1 || opt->persistent > 1 || (opt->flags & ~FP8GEMM_FLAG_WORKSPACE_ZEROED) != 0)
        *rc = FP8GEMM_E_KERNEL;
    return Config{opt->kernel, opt->tile_variant < 0 ? -1 : opt->tile_variant, opt->ksplit, opt->persistent};
}

// aligned = the plan for 16-byte aligned operands; otherwise the larger of that and what the padded
// plan needs when every operand has to be copied
size_t workspace_bytes_for(int m, int n, int k, const Config& cfg_in, bool any_alignment)
{
    if (m <= 0 || n <= 0 || k <= 0 || (k % 128) != 0)
        return 0;
    const uintptr_t al = 4096;
    GemmArgs g{reinterpret_cast<const uint8_t*>(al), reinterpret_cast<const uint8_t*>(al),
               reinterpret_cast<const float*>(al), nullptr, reinterpret_cast<uint16_t*>(al), m, n, k};
    GemmArgs gp = g;
    gp.m = (m + 15) & ~15;
    gp.n = (n + 15) & ~15;
    size_t need = 0;
    // the larger need of the plans a call may settle on: with the K splits added inside the kernel, and
    // -- when the device turns out not to place workgroups as that needs -- with the reduction kernel
    for (int fused = 0; fused < 2; ++fused) {
        Config cfg = cfg_in;
        if (!fused)
            cfg.fused_ok = false;
        const Plan p = make_plan(g, cfg);
        size_t one = 0;
        if (p.family >= 0)
            one = with_header(p.padded ? pad_layout(g, plan_workspace_bytes(gp, p), true, false).total
                                       : plan_workspace_bytes(g, p), plan_uses_header(p));
        if (any_alignment && !(p.family >= 0 && p.padded)) {
            // the same shape with an operand off a 16-byte boundary: the plan of the padded shape on copies
            const long long lim = 0x7FFFFFFFll;
            if ((long long)gp.m * k <= lim && (long long)gp.n * k <= lim && (long long)gp.m * gp.n <= lim &&
                cfg.selected != FP8GEMM_KERNEL_SCALAR) {
                const Plan pp = make_plan(gp, cfg);
                if (pp.family >= 0 && pp.family != FP8GEMM_KERNEL_SCALAR) {
                    const size_t all = with_header(pad_layout(g, plan_workspace_bytes(gp, pp), true, false).total,
                                                   plan_uses_header(pp));
                    one = all > one ? all : one;
                }
            }
        }
        need = one > need ? one : need;
    }
    return need;
}

}  // namespace

extern "C" {

int fp8_block_gemm(const void* a, const void* b, const float* a_scale, const float* b_scale, void* c,
                   int m, int n, int k)
{
    return run(a, b, a_scale, b_scale, c, m, n, k, nullptr, global_config(), nullptr);
}

int fp8_block_gemm_stream(const void* a, const void* b, const float* a_scale, const float* b_scale,
                          void* c, int m, int n, int k, void* stream)
{
    return run(a, b, a_scale, b_scale, c, m, n, k, static_cast<hipStream_t>(stream), global_config(), nullptr);
}

int fp8_block_gemm_ex(const void* a, const void* b, const float* a_scale, const float* b_scale, void* c,
                      int m, int n, int k, const fp8gemm_options* options, void* workspace,
                      size_t workspace_bytes, void* stream)
{
    int rc;
    const Config cfg = config_from_options(options, &rc);
    if (rc != FP8GEMM_OK)
        return rc;
    const bool zeroed = options && (options->flags & FP8GEMM_FLAG_WORKSPACE_ZEROED) != 0;
    const Workspace w{static_cast<float*>(workspace), workspace ? workspace_bytes : 0, zeroed};
    return run(a, b, a_scale, b_scale, c, m, n, k, static_cast<hipStream_t>(stream), cfg, &w);
}

int fp8_block_gemm_ws(const void* a, const void* b, const float* a_scale, const float* b_scale, void* c,
                      int m, int n, int k, void* workspace, size_t workspace_bytes, void* stream)
{
    return fp8_block_gemm_ex(a, b, a_scale, b_scale, c, m, n, k, nullptr, workspace, workspace_bytes, stream);
}

int fp8_block_gemm_noalloc(const void* a, const void* b, const float* a_scale, const float* b_scale, void* c,
                           int m, int n, int k, void* stream)
{
    // arguments first (no device call), then the plan's need against the fixed size: a plan that does
    // not fit is refused here, with the code a too small workspace always gets
    const int v = validate(a, b, a_scale, b_scale, c, m, n, k);
    if (v != FP8GEMM_OK)
        return v;
    const Config cfg = global_config();
    const GemmArgs g{static_cast<const uint8_t*>(a), static_cast<const uint8_t*>(b), a_scale, b_scale,
                     static_cast<uint16_t*>(c), m, n, k};
    // the largest need among the plans run() may settle on (with and without the in-kernel reduction)
    size_t need = 0;
    for (int fused = 0; fused < 2; ++fused) {
        Config probe = cfg;
        probe.fused_ok = fused != 0;
        Plan p = make_plan(g, probe);
        if (p.family < 0)
            return FP8GEMM_E_KERNEL;
        if (call_bytes(g, p) > (size_t)FP8GEMM_NOALLOC_MAX_BYTES)
            p = fitting_plan(g, p, probe, FP8GEMM_NOALLOC_MAX_BYTES);
        const size_t bytes = call_bytes(g, p);
        need = bytes > need ? bytes : need;
    }
    if (need > (size_t)FP8GEMM_NOALLOC_MAX_BYTES)
        return FP8GEMM_E_WORKSPACE;
    void* ptr = nullptr;
    const int rc = scratch_for_current_device(&ptr);
    if (rc != FP8GEMM_OK)
        return rc;
    // the array starts out zero and every kernel that uses the header leaves it zero
    const Workspace w{static_cast<float*>(ptr), (size_t)FP8GEMM_NOALLOC_MAX_BYTES, true};
    return run(a, b, a_scale, b_scale, c, m, n, k, static_cast<hipStream_t>(stream), cfg, &w);
}

int fp8_block_gemm_scalar(const void* a, const void* b, const float* a_scale, const float* b_scale,
                          void* c, int m, int n, int k, void* stream)
{
    return run(a, b, a_scale, b_scale, c, m, n, k, static_cast<hipStream_t>(stream),
               Config{FP8GEMM_KERNEL_SCALAR, -1, 0, -1}, nullptr);
}

int fp8_block_gemm_select(int kernel_id)
{
    if (kernel_id < FP8GEMM_KERNEL_AUTO || kernel_id > FP8GEMM_KERNEL_SKINNY)
        return FP8GEMM_E_KERNEL;
    g_selected.store(kernel_id);
    return FP8GEMM_OK;
}

int fp8_block_gemm_force_config(int tile_variant, int ksplit)
{
    if (tile_variant >= TILE_VARIANT_COUNT || ksplit < 0 || ksplit > MAX_KSPLIT)
        return FP8GEMM_E_KERNEL;
    g_force_variant.store(tile_variant < 0 ? -1 : tile_variant);
    g_force_ksplit.store(ksplit);
    return FP8GEMM_OK;
}

// Grouped GEMM behind both entry points.  explicit_ws = the caller's per-call workspace, nullptr = the
// process-wide one.
static int run_grouped(int groups, const void* const* a, const void* const* b, const float* const* a_scale,
                       const float* const* b_scale, void* const* c, const int* m, int n, int k, hipStream_t s,
                       const Config& cfg, const Workspace* explicit_ws)
{
    if (groups < 0)
        return FP8GEMM_E_SHAPE;
    if (groups == 0)
        return FP8GEMM_OK;
    if (!a || !b || !a_scale || !b_scale || !c || !m)
        return FP8GEMM_E_NULLPTR;
    // Groups of at most 64 rows (an MoE layer in a decode step) go to the decode kernel, which streams
    // every group's B once in whole lines; taller groups to the tile kernels.  A pinned tile
    // shape sends everything to the tile kernel.
    // A few small groups beside many taller ones ride along in the tile launch: their tiles fill its last round,
    // which costs less than a launch of their own (15 small + 49 tall groups, N = 2048, K = 7168: 258 us against
    // 281 us; 32 + 32: 284 against 257 us) -- unless that would put an on-grid tile launch on padded copies.
    bool small_to_tiles = cfg.force_variant >= 0;
    if (!small_to_tiles) {
        int small_n = 0, tall_n = 0;
        bool small_ragged = false, tall_ragged = false;
        for (int g = 0; g < groups; ++g) {
            if (m[g] <= 0)
                continue;
            (m[g] <= 64 ? small_n : tall_n) += 1;
            (m[g] <= 64 ? small_ragged : tall_ragged) |= m[g] % 16 != 0;
        }
        small_to_tiles = small_n > 0 && 3 * small_n <= tall_n && (!small_ragged || tall_ragged);
    }
    auto is_small = [&](int g) { return m[g] <= 64 && !small_to_tiles; };
    // every problem is validated before anything is launched
    long long m_total = 0;
    int count[2] = {0, 0};  // small, tall
    for (int g = 0; g < groups; ++g) {
        if (m[g] < 0)
            return FP8GEMM_E_SHAPE;
        if (m[g] == 0)
            continue;
        const int v = validate(a[g], b[g], a_scale[g], b_scale[g], c[g], m[g], n, k);
        if (v != FP8GEMM_OK)
            return v;
        m_total += m[g];
        ++count[is_small(g) ? 0 : 1];
    }
    if (count[0] + count[1] == 0)
        return FP8GEMM_OK;
    if (count[0] + count[1] == 1 && cfg.force_variant < 0)  // one problem: the dispatcher for single problems
        for (int g = 0; g < groups; ++g)
            if (m[g] > 0)
                return run(a[g], b[g], a_scale[g], b_scale[g], c[g], m[g], n, k, s, cfg, explicit_ws);
    static_assert(GroupTable::MAX_GROUPS == FP8GEMM_MAX_GROUPS, "table size mirrors the ABI constant");
    if (cfg.selected == FP8GEMM_KERNEL_AUTO && m_total <= 0x7FFFFFFFll) {
        // One launch holds MAX_GROUPS problems (the table travels in the kernel arguments): more of a kind run
        // as the fewest launches that hold them, of equal size, one after the other on the stream.
        int rc = FP8GEMM_OK;
        char first_name[sizeof(t_name_buf)] = "";
        for (int kind = 0; kind < 2 && rc == FP8GEMM_OK; ++kind) {
            if (count[kind] == 0)
                continue;
            const int launches = (count[kind] + GroupTable::MAX_GROUPS - 1) / GroupTable::MAX_GROUPS;
            const int per_launch = (count[kind] + launches - 1) / launches;
            GroupTable tab;
            tab.groups = 0;
            int seen = 0;
            for (int g = 0; g < groups && rc == FP8GEMM_OK; ++g) {
                if (m[g] == 0 || is_small(g) != (kind == 0))
                    continue;
                const int t = tab.groups++;
                tab.a[t] = static_cast<const uint8_t*>(a[g]);
                tab.b[t] = static_cast<const uint8_t*>(b[g]);
                tab.a_scale[t] = a_scale[g];
                tab.b_scale[t] = b_scale[g];
                tab.c[t] = static_cast<uint16_t*>(c[g]);
                tab.m[t] = m[g];
                tab.lda[t] = m[g];
                ++seen;
                if (tab.groups == per_launch || seen == count[kind]) {
                    rc = run_grouped_table(tab, n, k, kind == 0, s, cfg, explicit_ws);
                    if (rc == GROUPED_NOT_APPLICABLE) {  // these groups one by one
                        rc = FP8GEMM_OK;
                        for (int t = 0; t < tab.groups && rc == FP8GEMM_OK; ++t)
                            rc = run(tab.a[t], tab.b[t], tab.a_scale[t], tab.b_scale[t], tab.c[t], tab.m[t], n, k, s, cfg,
                                     explicit_ws);
                    }
                    tab.groups = 0;
                }
            }
            if (rc != FP8GEMM_OK)
                break;
            (void)last_kernel_name();  // into t_name_buf
            if (launches > 1) {  // the last launch's name and how many there were
                char many[sizeof(t_name_buf)];
                snprintf(many, sizeof(many), "%.88sx%d", t_name_buf, launches);
                snprintf(t_name_buf, sizeof(t_name_buf), "%s", many);
            }
            if (kind == 0 && count[1] > 0)
                snprintf(first_name, sizeof(first_name), "%s", t_name_buf);
            if (kind == 1 && first_name[0]) {  // both kernels ran: name both
                char both[sizeof(t_name_buf)];
                snprintf(both, sizeof(both), "%.46s+%.46s", first_name, t_name_buf);
                snprintf(t_name_buf, sizeof(t_name_buf), "%s", both);
            }
        }
        return rc;
    }
    for (int g = 0; g < groups; ++g) {
        if (m[g] == 0)
            continue;
        const int rc = run(a[g], b[g], a_scale[g], b_scale[g], c[g], m[g], n, k, s, cfg, explicit_ws);
        if (rc != FP8GEMM_OK)
            return rc;
    }
    return FP8GEMM_OK;
}

int fp8_block_gemm_grouped(int groups, const void* const* a, const void* const* b,
                           const float* const* a_scale, const float* const* b_scale,
                           void* const* c, const int* m, int n, int k, void* stream)
{
    return run_grouped(groups, a, b, a_scale, b_scale, c, m, n, k, static_cast<hipStream_t>(stream), global_config(),
                       nullptr);
}

int fp8_block_gemm_grouped_ex(int groups, const void* const* a, const void* const* b, const float* const* a_scale,
                              const float* const* b_scale, void* const* c, const int* m, int n, int k,
                              const fp8gemm_options* options, void* workspace, size_t workspace_bytes, void* stream)
{
    int rc;
    const Config cfg = config_from_options(options, &rc);
    if (rc != FP8GEMM_OK)
        return rc;
    const bool zeroed = options && (options->flags & FP8GEMM_FLAG_WORKSPACE_ZEROED) != 0;
    const Workspace w{static_cast<float*>(workspace), workspace ? workspace_bytes : 0, zeroed};
    return run_grouped(groups, a, b, a_scale, b_scale, c, m, n, k, static_cast<hipStream_t>(stream), cfg, &w);
}

int fp8_block_gemm_set_fused_reduction(int mode)
{
    if (mode < -1 || mode > 1)
        return FP8GEMM_E_KERNEL;
    g_fused.store(mode);
    return FP8GEMM_OK;
}

int fp8_block_gemm_set_persistent(int mode)
{
    if (mode < -1 || mode > 1)
        return FP8GEMM_E_KERNEL;
    g_persistent.store(mode);
    return FP8GEMM_OK;
}

const char* fp8_block_gemm_last_kernel(void) { return last_kernel_name(); }

int fp8_block_gemm_plan(int m, int n, int k, char* name, size_t cap)
{
    if (!name || cap == 0)
        return FP8GEMM_E_NULLPTR;
    if (m <= 0 || n <= 0 || k <= 0 || (k % 128) != 0)
        return FP8GEMM_E_SHAPE;
    // aligned dummy addresses: only their alignment is inspected
    GemmArgs g{reinterpret_cast<const uint8_t*>(uintptr_t(4096)), reinterpret_cast<const uint8_t*>(uintptr_t(4096)),
               reinterpret_cast<const float*>(uintptr_t(4096)), nullptr, reinterpret_cast<uint16_t*>(uintptr_t(4096)),
               m, n, k};
    Plan p = make_plan(g, global_config());
    if (p.family < 0)
        return FP8GEMM_E_KERNEL;
    plan_name(p, name, cap);
    return FP8GEMM_OK;
}

size_t fp8_block_gemm_workspace_bytes(int m, int n, int k)
{
    return workspace_bytes_for(m, n, k, global_config(), false);
}

size_t fp8_block_gemm_workspace_bytes_ex(int m, int n, int k, const fp8gemm_options* options, int any_alignment)
{
    int rc;
    const Config cfg = config_from_options(options, &rc);
    if (rc != FP8GEMM_OK)
        return 0;
    return workspace_bytes_for(m, n, k, cfg, any_alignment != 0);
}

static size_t grouped_bytes(int groups, const int* m, int n, int k, const Config& cfg)
{
    if (groups <= 0 || !m || n <= 0 || k <= 0 || (k % 128) != 0)
        return 0;
    // a grouped launch on padded copies takes every group's copies at once (the decode kernel's splits meet
    // in the header); one by one the largest single need would do
    const int n16 = (n + 15) & ~15;
    const size_t nkb = (size_t)k / 128;
    size_t total = 0, small_groups = 0;
    for (int g = 0; g < groups; ++g) {
        if (m[g] <= 0)
            continue;
        const size_t m16 = ((size_t)m[g] + 15) & ~(size_t)15;
        total += round256((size_t)k * m16) + round256(nkb * m16 * sizeof(float)) + round256((size_t)k * n16) +
                 round256(m16 * n16 * 2);
        small_groups += m[g] <= 64 ? 1 : 0;
    }
    total = with_header(total, small_groups > 0);
    for (int g = 0; g < groups; ++g) {
        if (m[g] <= 0)
            continue;
        const size_t single = workspace_bytes_for(m[g], n, k, cfg, true);
        total = total > single ? total : single;
    }
    return total;
}

size_t fp8_block_gemm_grouped_workspace_bytes(int groups, const int* m, int n, int k)
{
    return grouped_bytes(groups, m, n, k, global_config());
}

size_t fp8_block_gemm_grouped_workspace_bytes_ex(int groups, const int* m, int n, int k, const fp8gemm_options* options)
{
    int rc;
    const Config cfg = config_from_options(options, &rc);
    return rc == FP8GEMM_OK ? grouped_bytes(groups, m, n, k, cfg) : 0;
}

int fp8_block_gemm_set_workspace(void* device_ptr, size_t bytes)
{
    if (device_ptr && (reinterpret_cast<uintptr_t>(device_ptr) % 256) != 0)
        return FP8GEMM_E_WORKSPACE;
    // the header at its start is zero-filled here (the call waits for that fill); a buffer too
    // small to hold it can serve no plan anyway
    bool zeroed = false;
    if (device_ptr && bytes >= WS_HEADER) {
        const hipError_t e = hipMemset(device_ptr, 0, WS_HEADER);
        if (e != hipSuccess)
            return (int)e;
        zeroed = true;
    }
    std::lock_guard<std::mutex> lock(g_ws_mutex);
    g_ws_user = static_cast<float*>(device_ptr);
    g_ws_user_bytes = device_ptr ? bytes : 0;
    g_ws_user_zeroed = zeroed;
    return FP8GEMM_OK;
}

int fp8_block_gemm_release(void)
{
    const hipError_t staging = release_host_staging();
    std::lock_guard<std::mutex> lock(g_ws_mutex);
    if (!g_ws_own && g_ws_retired.empty())
        return (int)staging;
    hipError_t e = hipDeviceSynchronize();  // kernels of earlier calls may still use the buffers
    if (e != hipSuccess)
        return (int)e;
    hipError_t first = staging;
    for (Retired& r : g_ws_retired) {
        if (r.done)
            (void)hipEventDestroy(r.done);
        e = hipFree(r.ptr);
        first = first == hipSuccess ? e : first;
    }
    g_ws_retired.clear();
    g_ws_own_captured = false;
    if (g_ws_own) {
        e = hipFree(g_ws_own);
        first = first == hipSuccess ? e : first;
        g_ws_own = nullptr;
        g_ws_own_bytes = 0;
    }
    return (int)first;
}

int fp8_convert_f32_to_e4m3fn(const float* in, void* out, size_t count, void* stream)
{
    if (count == 0)
        return FP8GEMM_OK;
    if (!in || !out)
        return FP8GEMM_E_NULLPTR;
    if (reinterpret_cast<uintptr_t>(in) % 16 != 0 || reinterpret_cast<uintptr_t>(out) % 4 != 0)
        return FP8GEMM_E_ALIGN;  // the kernel reads four floats and writes four codes at a time
    return (int)launch_convert(in, static_cast<uint8_t*>(out), count, static_cast<hipStream_t>(stream));
}

static int quantize_entry(const void* x, int x_dtype, void* q, float* scale, int rows, int k,
                          void* stream, bool block128)
{
    if (!x || !q || !scale)
        return FP8GEMM_E_NULLPTR;
    if (rows <= 0 || k <= 0 || (k % 128) != 0)
        return FP8GEMM_E_SHAPE;
    if ((long long)rows * k > 0x7FFFFFFFll)
        return FP8GEMM_E_TOOLARGE;
    if (x_dtype != FP8GEMM_DTYPE_BF16 && x_dtype != FP8GEMM_DTYPE_F32 && x_dtype != FP8GEMM_DTYPE_BF16_F32MATH)
        return FP8GEMM_E_DTYPE;
    if (reinterpret_cast<uintptr_t>(x) % 16 != 0)
        return FP8GEMM_E_ALIGN;
    static_assert(QUANT_SOURCE_BF16 == FP8GEMM_DTYPE_BF16 && QUANT_SOURCE_F32 == FP8GEMM_DTYPE_F32 &&
                      QUANT_SOURCE_BF16_F32MATH == FP8GEMM_DTYPE_BF16_F32MATH,
                  "launcher enum mirrors the ABI constants");
    return (int)launch_quantize(x, static_cast<QuantSource>(x_dtype), static_cast<uint8_t*>(q), scale, rows,
                                k, block128, static_cast<hipStream_t>(stream));
}

int fp8_quantize_a_1x128(const void* x, int x_dtype, void* a, float* a_scale, int m, int k,
                         void* stream)
{
    return quantize_entry(x, x_dtype, a, a_scale, m, k, stream, false);
}

int fp8_quantize_b_128x128(const void* x, int x_dtype, void* b, float* b_scale, int n, int k,
                           void* stream)
{
    return quantize_entry(x, x_dtype, b, b_scale, n, k, stream, true);
}

const char* fp8_block_gemm_error_string(int code)
{
    switch (code) {
    case FP8GEMM_OK: return "success";
    case FP8GEMM_E_NULLPTR: return "a required pointer is NULL";
    case FP8GEMM_E_SHAPE: return "m, n, k must be positive and k a multiple of 128";
    case FP8GEMM_E_KERNEL: return "unknown kernel id or kernel not applicable to this shape";
    case FP8GEMM_E_WORKSPACE: return "workspace missing, too small or misaligned (or it would have to grow under stream capture)";
    case FP8GEMM_E_TOOLARGE: return "operand exceeds 2^31-1 elements";
    case FP8GEMM_E_DTYPE: return "unknown source element type";
    case FP8GEMM_E_ALIGN: return "pointer alignment: 16 bytes for a source, 4 for the converter's output";
    default: break;
    }
    if (code > 0)
        return hipGetErrorString(static_cast<hipError_t>(code));
    return "unknown error code";
}

size_t fp8_block_gemm_workspace_growth(size_t have, size_t need) { return growth_target(have, need); }

int fp8_block_gemm_abi_version(void) { return 5; }

}  // extern "C"
