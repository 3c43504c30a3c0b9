// Internal (C++) launch functions behind the C ABI in include/fp8_block_gemm.h.
// Each returns a hipError_t; none synchronises.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <atomic>

namespace fp8gemm {

struct GemmArgs {
    const uint8_t* a;
    const uint8_t* b;
    const float* a_scale;
    const float* b_scale;
    uint16_t* c;
    int m, n, k;
    // elements between consecutive k-rows of a and of a_scale; 0 = m (the layout of the ABI).
    // Only the tile kernels take another value (padded copies whose c keeps m rows).
    int lda = 0;
};
inline int leading_dim(const GemmArgs& g) { return g.lda ? g.lda : g.m; }

// Kernels with more than 64 KiB of dynamic LDS need the attribute raised before their first launch
// on a device.  Once per kernel and device (a bit per device in a word of each kernel's own) instead of
// once per launch: the runtime call costs as much as a short kernel takes.
template <auto KERNEL>
hipError_t allow_lds(int bytes)
{
    static std::atomic<uint64_t> done{0};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess)
        return e;
    const uint64_t bit = 1ull << (dev & 63);
    if (done.load(std::memory_order_acquire) & bit)
        return hipSuccess;
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(KERNEL), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e == hipSuccess)
        done.fetch_or(bit, std::memory_order_release);
    return e;
}
// A kernel as an argument of a generic lambda: kernels with the same parameters have one type, so the function
// pointer itself would leave them one instantiation, and one word of allow_lds, between them.
template <auto KERNEL>
struct Kernel {
    static constexpr auto value = KERNEL;
};
#define FP8GEMM_ALLOW_LDS(kern, bytes)                                                                       \
    do {                                                                                                     \
        const hipError_t e_ = allow_lds<kern>(bytes);                                                        \
        if (e_ != hipSuccess)                                                                                \
            return e_;                                                                                       \
    } while (0)

// A launch by the kernel's own argument list.  The triple-chevron form, and the macro that stands for it, hand the launch shape to
// the runtime and fetch it back in the kernel's stub: 0.1 us more on the host of the 2.3 us that a launch takes there (calls back to back
// from Python, with the plan looked up once and named when asked for: 16 x 128 x 128 3.14 -> 2.95 us, quantiser 2.77 -> 2.70).
template <class... P, class... A>
void launch_kernel(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t s, A... args)
{
    [&](P... p) {
        void* list[] = {const_cast<void*>(static_cast<const void*>(&p))...};
        (void)hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, list, lds, s);
    }(args...);
}

// one thread per C element (check.cu:30-49)
hipError_t launch_scalar(const GemmArgs& g, hipStream_t s);

// The mailbox: device memory that only the kernels that add their K splits themselves write, all zero
// before a launch and all zero again after it; the splits of a tile or strip hand their partial results
// over through it.
constexpr size_t SPLIT_MAILBOX_BYTES = (size_t)16 << 20;

// MFMA tile kernel family.  `variant` picks the workgroup tile; ksplit > 1 writes fp32
// partial sums to `partial` ([ksplit][m][n]) instead of c.  With mailbox == nullptr it must be followed
// by launch_splitk_reduce; with a mailbox (SPLIT_MAILBOX_BYTES) the workgroup of a tile's last split
// adds the other splits' accumulators itself and writes c, with the same arithmetic, and `partial` is
// not used.  The latter needs xcd_placement_confirmed() and tile_mailbox_bytes() <= SPLIT_MAILBOX_BYTES.
enum TileVariant { TILE_256x192 = 0, TILE_256x128 = 1, TILE_128x128 = 2, TILE_128x192 = 3,
                   TILE_64x64 = 4, TILE_256x192_W4 = 5, TILE_256x256 = 6, TILE_VARIANT_COUNT,
                   TILE_128x256 = TILE_VARIANT_COUNT };  // grouped launches only, not to be asked for by number
bool tile_supports(const GemmArgs& g);
// row counts off the 16-byte grid, taken as they are (launch_tile, plain form)
bool tile_ragged_supports(const GemmArgs& g, int variant);
const char* tile_variant_name(int variant);
void tile_variant_dims(int variant, int* bm, int* bn);
size_t tile_mailbox_bytes(const GemmArgs& g, int variant, int ksplit);
hipError_t launch_tile(const GemmArgs& g, int variant, int ksplit, float* partial, float* mailbox,
                       hipStream_t s);
// Persistent form (ksplit = 1 only): `workgroups` (a multiple of 8) workgroups walk through
// all tiles, the copies of a tile's first K blocks overlap the previous tile's epilogue.
bool tile_persistent_supports(const GemmArgs& g, int variant);
hipError_t launch_tile_persistent(const GemmArgs& g, int variant, int workgroups, hipStream_t s);
// Grouped form: several problems with the same n and k and their own m in one persistent launch
// (the table travels by value in the kernel arguments; tile_start is filled by the launcher).
struct GroupTable {
    static constexpr int MAX_GROUPS = 64;
    const uint8_t* a[MAX_GROUPS];
    const uint8_t* b[MAX_GROUPS];
    const float* a_scale[MAX_GROUPS];
    const float* b_scale[MAX_GROUPS];
    uint16_t* c[MAX_GROUPS];
    int m[MAX_GROUPS];
    int lda[MAX_GROUPS];  // as GemmArgs::lda, but always filled in
    int tile_start[MAX_GROUPS + 1];
    int groups;
};
bool tile_grouped_supports(const GroupTable& tab, int n, int k, int variant);
hipError_t launch_tile_grouped(GroupTable& tab, int n, int k, int variant, int workgroups, hipStream_t s);
// The same problems with a tile of 64x64 or 128x128 per workgroup, rows off the 16-row grid as they are (`ragged`), their K
// splits added inside the kernel: mailbox = SPLIT_MAILBOX_BYTES as above, not used with ksplit 1.  lda has to be m.
bool tile_each_supports(const GroupTable& tab, int n, int k, int variant, bool* ragged);
hipError_t launch_tile_each(GroupTable& tab, int n, int k, int variant, int ksplit, float* mailbox, hipStream_t s);
// ... of the two large tiles, 256x192 and 256x256 (called by the two functions above, which check the arguments)
// The tiles of a last round of 256x256 that would leave half the workgroups or more without one are cut into halves
// (256x128) or quarters (128x128), one for each workgroup.
enum class Tail { NONE, HALVES, QUARTERS };
Tail large_tile_tail(long tiles, int k, int workgroups);
hipError_t launch_tile_large(const GemmArgs& g, int variant, int workgroups, hipStream_t s);
hipError_t launch_tile_large_grouped(GroupTable& tab, int n, int k, int variant, int workgroups, hipStream_t s);
hipError_t launch_splitk_reduce(const GemmArgs& g, int ksplit, const float* partial, hipStream_t s);

// tiny-M streaming kernel (decode shapes)
bool skinny_supports(const GemmArgs& g);
int skinny_ksplit(const GemmArgs& g);
double skinny_cost(const GemmArgs& g, int ksplit);
hipError_t launch_skinny(const GemmArgs& g, int ksplit, float* partial, hipStream_t s);

// wide-strip decode kernel (M <= 64): 128-column strips, the K splits of a strip added inside the
// kernel.  `mailbox` = SPLIT_MAILBOX_BYTES as above.  ksplit > 1 needs xcd_placement_confirmed() and
// decode_strip_can_split.
constexpr int DECODE_MAX_KSPLIT = 16;
bool decode_strip_supports(const GemmArgs& g);
// halves = 128-column halves of a strip: 1, or 2 (256-column strips: 256 contiguous bytes of every k-row of B), or 0: strips
// of 64 columns (k_decode64.hip)
size_t decode_strip_mailbox_bytes(const GemmArgs& g, int ksplit, int halves = 1);
bool decode_strip_can_split(const GemmArgs& g, int ksplit, int halves = 1);
double decode_strip_cost(const GemmArgs& g, int ksplit, int halves = 1);
hipError_t launch_decode_strips(const GemmArgs& g, int ksplit, int halves, float* mailbox, hipStream_t s);
// ... in strips of 64 columns (called by the functions above for halves = 0)
size_t decode64_mailbox_bytes(const GemmArgs& g, int ksplit);
int decode64_ksplit(const GemmArgs& g);  // the split that it would run with; 0: more strips than the device holds at once
bool decode64_pays(const GemmArgs& g, int ksplit, int ksplit128);  // against 128-column strips in ksplit128 splits
hipError_t launch_decode64(const GemmArgs& g, int ksplit, float* mailbox, hipStream_t s);
// The same kernel on several problems with common n and k and their own m <= 64 (multiples of 16), whose
// strips form one list of work items; tile_start of the table is not used.
bool decode_grouped_supports(const GroupTable& tab, int n, int k);
int decode_grouped_ksplit(const GroupTable& tab, int n, int k, bool fused_ok);
size_t decode_grouped_mailbox_bytes(const GroupTable& tab, int n, int ksplit);
bool decode_grouped_streams(int groups, int n);  // the launch takes the streaming form (rows on the 16-byte grid, no K split)
hipError_t launch_decode_grouped(const GroupTable& tab, int n, int k, int ksplit, float* mailbox, hipStream_t s);
// 1 = workgroups whose linear ids agree modulo 8 share an XCD on the current device (looked at once
// per device with a probe grid, which the first call waits for: not under stream capture),
// 0 = they do not, or it could not be looked at; -1 = not looked at yet and may_probe is false
int xcd_placement_confirmed(bool may_probe);

// Padding copies of a call (bytes of a and b, fp32 values of a_scale taken as bytes), all in one launch: rows of ld_src
// bytes copied into rows of 16 * chunks >= ld_src bytes, the rest zero.  The destinations are given as distances
// from `base` (16-byte aligned) in steps of 256 bytes, which lets the jobs of a full grouped launch travel by value in the kernel arguments.
constexpr int PAD_JOBS_SINGLE = 3, PAD_JOBS_GROUPED = 128;
template <int MAX>
struct PadJobs {
    const void* src[MAX];
    uint8_t* base;
    uint32_t dst256[MAX];  // distance of the destination from base in units of 256 bytes
    uint32_t rows[MAX], ld_src[MAX], chunks[MAX];
    uint32_t first_block[MAX];  // filled in by the launcher
    int count = 0;
    // offset (from base) is a multiple of 256
    void add(const void* from, size_t offset, size_t n_rows, size_t row_bytes, size_t padded_bytes)
    {
        src[count] = from;
        dst256[count] = (uint32_t)(offset / 256);
        rows[count] = (uint32_t)n_rows;
        ld_src[count] = (uint32_t)row_bytes;
        chunks[count] = (uint32_t)(padded_bytes / 16);
        ++count;
    }
};
template <int MAX>
hipError_t launch_pad(PadJobs<MAX>& jobs, hipStream_t s);
// Cropping: the m x n corner of a bf16 matrix with ld_src elements per row copied into a dense one; batched: for
// several matrices in one launch
hipError_t launch_crop_bf16(const uint16_t* src, uint16_t* dst, int m, int n, int ld_src, hipStream_t s);
struct CropTable {
    static constexpr int MAX_GROUPS = 64;
    const void* src[MAX_GROUPS];
    void* dst[MAX_GROUPS];
    int m[MAX_GROUPS];
    int n, ld_src;
    int groups;
};
hipError_t launch_crop_bf16_batched(const CropTable& tab, hipStream_t s);

// fp32 -> e4m3fn (check.cu:17-22)
hipError_t launch_convert(const float* in, uint8_t* out, size_t count, hipStream_t s);

// 1 x 128 (block128 = false) or 128 x 128 quantiser of a row-major [rows][k] matrix into the
// GEMM's column-major fp8 layout and scale layout (quantize.py:16-67)
// source: element type of x and the arithmetic (values of FP8GEMM_DTYPE_*)
enum QuantSource { QUANT_SOURCE_BF16 = 0, QUANT_SOURCE_F32 = 1, QUANT_SOURCE_BF16_F32MATH = 2 };
hipError_t launch_quantize(const void* x, QuantSource source, uint8_t* q, float* scale_out, int rows,
                           int k, bool block128, hipStream_t s);

// host_gemm.hip: the pinned staging buffer kept between calls of fp8_gemm_host, back to the system
hipError_t release_host_staging();

}  // namespace fp8gemm
