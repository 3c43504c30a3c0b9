// Host-buffer launcher: the counterpart of gemmGPU (/root/reference/check.cu:51-130,
// /root/reference/sgemm.cu:24-191): fp32 values in host memory in, bf16 in host memory out, with every
// HIP return code checked instead of discarded.
//
// What bounds it is the way from pageable memory to the device.  Uploaded as they are, the fp32 values cross the
// link at four times the size that the GEMM reads, through the runtime's own staging of pageable memory.  Here a few
// host threads round the values to e4m3fn (bit for bit what k_convert.hip does) on their way into a pinned staging
// buffer, which the values would have to be copied into anyway, and the staged bytes are uploaded while later ones are
// converted; device memory is one allocation, made meanwhile.  1024 x 1536 x 7168 (73 MB of fp32 values): 4460 us with
// fp32 uploads and a buffer per operand, 1660 us with conversion into staging memory pinned by each call, 1400 us with the
// staging buffer kept; of these, by time stamps, 130 start the threads, 640 to 840 convert and upload (the values are read
// from memory at 110 GB/s), 210 are the GEMM and the way back.
#include "../../include/fp8_block_gemm.h"
#include "launchers.h"

#include <algorithm>
#include <atomic>
#include <cfenv>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <thread>
#if defined(__x86_64__)
#include <cpuid.h>
#endif

namespace {

struct DeviceBuf {
    void* p = nullptr;
    ~DeviceBuf()
    {
        if (p)
            (void)hipFree(p);
    }
    hipError_t alloc(size_t bytes) { return hipMalloc(&p, bytes ? bytes : 1); }
};

constexpr size_t SCALES_STAGED = (size_t)1 << 20;  // bytes of scales that go through the staging buffer

// Staging memory of a call.  Pinned if the system grants it, pageable otherwise: the copies below are right either way.
// Pinning costs as much as converting into it (16 MiB: 0.5 to 1.2 ms), so one buffer of at most STAGING_MAX is kept
// between calls, for whichever call asks first, and given back by fp8_block_gemm_release; calls that overlap with its
// user pin their own.
constexpr size_t STAGING_MAX = (size_t)32 << 20;
std::mutex g_staging_mutex;
void* g_staging = nullptr;  // the kept buffer while no call uses it
size_t g_staging_bytes = 0;

struct StagingBuf {
    uint8_t* p = nullptr;
    size_t bytes = 0;
    bool pinned = false;
    ~StagingBuf()
    {
        if (!pinned) {
            std::free(p);
            return;
        }
        void* drop = p;
        if (bytes <= STAGING_MAX) {  // the larger of the two is kept
            std::lock_guard<std::mutex> lock(g_staging_mutex);
            if (bytes > g_staging_bytes) {
                drop = g_staging;
                g_staging = p;
                g_staging_bytes = bytes;
            }
        }
        if (drop)
            (void)hipHostFree(drop);
    }
    bool alloc(size_t need)
    {
        {
            std::lock_guard<std::mutex> lock(g_staging_mutex);
            if (g_staging && g_staging_bytes >= need) {
                p = static_cast<uint8_t*>(g_staging);
                bytes = g_staging_bytes;
                pinned = true;
                g_staging = nullptr;
                g_staging_bytes = 0;
                return true;
            }
        }
        void* q = nullptr;
        if (hipHostMalloc(&q, need, hipHostMallocPortable) == hipSuccess) {
            pinned = true;
        } else {
            (void)hipGetLastError();
            q = std::malloc(need);
        }
        p = static_cast<uint8_t*>(q);
        bytes = need;
        return p != nullptr;
    }
};

// fp32 -> e4m3fn, nearest even, beyond +-448 saturated, NaN kept.  Normal results: the upper bits of the fp32 word,
// rounded by adding half a unit (less one, plus the bit that stays last), with the exponent's bias moved from 127 to 7.
// Below 2^-6 the code counts steps of 2^-9: adding 2^14 rounds to that step in hardware (NearestEven below).
inline uint32_t e4m3fn_code(float x)
{
    uint32_t u;
    std::memcpy(&u, &x, 4);
    const uint32_t au = u & 0x7FFFFFFFu;
    const uint32_t normal = ((au + 0x7FFFFu + ((au >> 20) & 1u)) >> 20) - (120u << 3);
    float ax;
    std::memcpy(&ax, &au, 4);
    const float stepped = ax + 16384.0f;
    uint32_t su;
    std::memcpy(&su, &stepped, 4);
    uint32_t code = au < 0x3C800000u ? (su & 0xFFu) : normal;  // 2^-6
    code = au >= 0x43E00000u ? 0x7Eu : code;                   // 448
    code = au > 0x7F800000u ? 0x7Fu : code;
    return code | ((u >> 24) & 0x80u);
}

// The arithmetic above rounds to nearest and raises no exception whatever the caller's floating-point environment (which
// threads inherit) asks for, and leaves that environment as it was.
struct NearestEven {
    std::fenv_t caller;
    NearestEven()
    {
        std::feholdexcept(&caller);
        std::fesetround(FE_TONEAREST);
    }
    ~NearestEven() { std::fesetenv(&caller); }
};

#if defined(__x86_64__)
// The values are asked for past L2 and L3, which the caller's other data need: the call on 1024 x 1536 x 7168 takes 1.40 ms
// instead of 1.65.
__attribute__((target("avx2"), noinline)) void convert_avx2(const float* __restrict__ in, uint8_t* __restrict__ out, size_t count)
{
    constexpr size_t LINE = 16, AHEAD = 32 * LINE;
    size_t i = 0;
    for (; i + LINE <= count; i += LINE) {
        __builtin_prefetch(in + std::min(i + AHEAD, count - 1), 0, 0);
        for (size_t j = 0; j < LINE; ++j)
            out[i + j] = (uint8_t)e4m3fn_code(in[i + j]);
    }
    for (; i < count; ++i)
        out[i] = (uint8_t)e4m3fn_code(in[i]);
}

// (__builtin_cpu_supports answers from the compiler runtime's table, which does not hold this one everywhere)
bool has_clflushopt()
{
    uint32_t a, b, c, d;
    return __get_cpuid_count(7, 0, &a, &b, &c, &d) != 0 && ((b >> 23) & 1u) != 0;
}

// Every line of in[0 .. count) out of all caches, to memory if it is dirty.
__attribute__((target("clflushopt"))) void evict_lines(const float* in, size_t count)
{
    const uintptr_t end = reinterpret_cast<uintptr_t>(in + count);
    for (uintptr_t line = reinterpret_cast<uintptr_t>(in) & ~(uintptr_t)63; line < end; line += 64)
        __builtin_ia32_clflushopt(reinterpret_cast<const void*>(line));
}
#endif

__attribute__((noinline)) void convert_plain(const float* __restrict__ in, uint8_t* __restrict__ out, size_t count)
{
    for (size_t i = 0; i < count; ++i)
        out[i] = (uint8_t)e4m3fn_code(in[i]);
}

void convert_host(const float* in, uint8_t* out, size_t count)
{
    const NearestEven environment;  // (the converters are not inlined: nothing of theirs moves out of its span)
#if defined(__x86_64__)
    if (__builtin_cpu_supports("avx2"))
        return convert_avx2(in, out, count);
#endif
    convert_plain(in, out, count);
}

// Values that the workers have read leave the caches.  Left in those of the cores that converted them, they make the
// caller's next write to that memory wait for those cores, line by line, which can cost more than the workers save.  In ms,
// with the values read and rewritten in place before each call, write / call / both: 300 x 2048 x 2048 with fp32 uploads
// 0.25 / 0.90 / 1.16, with workers 0.9 ... 1.7 / 0.48 / 1.4 ... 2.3, this way 0.46 / 0.53 / 1.0; 1024 x 1536 x 7168 1.8 / 4.5 /
// 6.4, 2.3 ... 5.9 / 1.6 / 3.7 ... 7.6, 1.9 / 1.6 / 3.4; 4096 x 4608 x 7168 6.5 / 12.4 / 19, 7.5 ... 11.5 / 4.7 / 12.1 ... 16.7,
// 6.5 / 5.3 / 11.9.  Written by a plain copy, which does not read, or into new memory, level with the workers alone (both
// together 1.13, 4.0 and 12.8 against 1.12, 4.0 and 12.4; fp32 uploads 1.7, 7.0 and 21).  Each piece's lines right behind
// its conversion instead of all of them behind the last one: 0.1 to 0.2 ms more on the first two.  On a processor without
// the instruction the lines stay.
void give_back(const float* in, size_t count)
{
#if defined(__x86_64__)
    static const bool can = has_clflushopt();
    if (can)
        evict_lines(in, count);
#else
    (void)in, (void)count;
#endif
}

// A and B as one run of pieces, a ring of SLOTS of which is staged at a time.  Workers take pieces in order, main
// uploads them in order and hands slots back once their upload has completed.
struct Pipeline {
    static constexpr size_t PIECE = 128 * 1024;  // elements: 24 us of conversion, small enough to share out evenly
    static constexpr size_t SLOTS = 248;         // 31 MiB: with the scales at most STAGING_MAX
    static constexpr int MAX_WORKERS = 8;        // 4, 8, 16 threads convert 73 MB in 0.87, 0.54, 0.61 ms
    // Fewer pieces than this the caller converts alone.  Call, and call with the values rewritten in place before it:
    // 100 x 512 x 1024 (5 pieces) 0.19 and 0.22 ms against 0.27 and 0.32 with a worker, 128 x 1024 x 1024 (9) 0.30 and
    // 0.36 against 0.23 and 0.36 with two, 300 x 2048 x 2048 (37) 1.07 and 1.32 against 0.53 and 1.0 with eight.
    static constexpr size_t MIN_PIECES = 8;

    const float* src[2];
    size_t count[2], pieces[2];
    size_t total;  // pieces of both
    size_t slots;  // of the ring that this call needs
    uint8_t* staging = nullptr;
    std::atomic<size_t> next{0}, freed{0}, returned{0};
    std::atomic<bool> abort{false};
    std::atomic<size_t> ready[SLOTS];  // number of the last piece converted into the slot, plus one

    Pipeline(const float* a, size_t na, const float* b, size_t nb)
        : src{a, b}, count{na, nb}, pieces{(na + PIECE - 1) / PIECE, (nb + PIECE - 1) / PIECE}
    {
        total = pieces[0] + pieces[1];
        slots = std::min(total, SLOTS);
        for (auto& r : ready)
            r.store(0, std::memory_order_relaxed);
    }

    // matrix, first element and number of elements of a piece
    void piece(size_t p, int& which, size_t& first, size_t& n) const
    {
        which = p < pieces[0] ? 0 : 1;
        first = (p - (which ? pieces[0] : 0)) * PIECE;
        n = std::min(PIECE, count[which] - first);
    }

    void convert(size_t p)
    {
        int which;
        size_t first, n;
        piece(p, which, first, n);
        convert_host(src[which] + first, staging + (p % slots) * PIECE, n);
        ready[p % slots].store(p + 1, std::memory_order_release);
    }

    void work()
    {
        for (;;) {
            const size_t p = next.fetch_add(1, std::memory_order_relaxed);
            if (p >= total)
                break;
            while (p >= freed.load(std::memory_order_acquire) + slots) {
                if (abort.load(std::memory_order_relaxed))
                    return;
                std::this_thread::yield();
            }
            convert(p);
        }
        // the lines back to the caller, while main is busy with the last uploads, the GEMM and c
        while (!abort.load(std::memory_order_relaxed)) {
            const size_t p = returned.fetch_add(1, std::memory_order_relaxed);
            if (p >= total)
                return;
            int which;
            size_t first, n;
            piece(p, which, first, n);
            give_back(src[which] + first, n);
        }
    }

    bool is_ready(size_t p) const { return ready[p % slots].load(std::memory_order_acquire) == p + 1; }

    // main: everything to dst[0] and dst[1] on the null stream; the last copies may be in flight on return
    hipError_t upload(void* const dst[2], bool have_workers)
    {
        size_t p = 0;
        while (p < total) {
            // half of the ring back at a time: the other half is what the workers fill meanwhile
            if (total > slots && p - freed.load(std::memory_order_relaxed) >= slots / 2) {
                const hipError_t e = hipStreamSynchronize(nullptr);
                if (e != hipSuccess)
                    return e;
                freed.store(p, std::memory_order_release);
            }
            if (!have_workers)
                convert(p);
            while (!is_ready(p))
                std::this_thread::yield();
            // as many pieces as lie behind one another, converted, in the same matrix: a copy costs about 9 us
            int which;
            size_t first, n;
            piece(p, which, first, n);
            size_t end = p + 1, bytes = n;
            const size_t stop = std::min(which ? total : pieces[0], p + (slots - p % slots));
            while (have_workers && end < stop && end - p < slots / 4 && is_ready(end)) {
                int w;
                size_t f, more;
                piece(end, w, f, more);
                bytes += more;
                ++end;
            }
            const hipError_t e = hipMemcpyAsync(static_cast<uint8_t*>(dst[which]) + first, staging + (p % slots) * PIECE,
                                                bytes, hipMemcpyHostToDevice, nullptr);
            if (e != hipSuccess)
                return e;
            p = end;
        }
        return hipSuccess;
    }
};

// The worker threads of one call: joined whatever way the call ends.
struct Workers {
    Pipeline& pipe;
    std::thread thread[Pipeline::MAX_WORKERS];
    int count = 0;

    explicit Workers(Pipeline& p) : pipe(p) {}
    ~Workers()
    {
        pipe.abort.store(true, std::memory_order_relaxed);
        join();
    }
    void start()
    {
        const int cpus = (int)std::thread::hardware_concurrency();
        const int want = pipe.total < Pipeline::MIN_PIECES
                             ? 0
                             : std::min({Pipeline::MAX_WORKERS, cpus - 1, (int)std::min<size_t>(pipe.total / 4, 64)});
        try {
            for (; count < want; ++count)
                thread[count] = std::thread([this] { pipe.work(); });
        } catch (...) {  // no more threads to be had: those that run, or the caller alone, do it all
        }
    }
    void join()
    {
        for (int i = 0; i < count; ++i)
            if (thread[i].joinable())
                thread[i].join();
    }
};

// c through the staging buffer, in two halves that take turns: one is copied out of while the other fills
hipError_t download(unsigned short* c, const void* d_c, size_t bytes, uint8_t* staging, size_t staging_bytes)
{
    const size_t half = std::min<size_t>(staging_bytes / 2, 1 << 20);
    uint8_t* out = reinterpret_cast<uint8_t*>(c);
    size_t done = 0, n = 0;
    for (size_t at = 0, turn = 0; done < bytes; ++turn) {
        const size_t coming = std::min(half, bytes - at);
        if (coming) {
            const hipError_t e = hipMemcpyAsync(staging + (turn & 1) * half, static_cast<const uint8_t*>(d_c) + at, coming,
                                                hipMemcpyDeviceToHost, nullptr);
            if (e != hipSuccess)
                return e;
        }
        if (n)
            std::memcpy(out + done, staging + ((turn & 1) ^ 1) * half, n);
        done += n;
        n = coming;
        at += coming;
        const hipError_t e = hipStreamSynchronize(nullptr);
        if (e != hipSuccess)
            return e;
    }
    return hipSuccess;
}

size_t padded(size_t bytes) { return (bytes + 255) / 256 * 256; }

}  // namespace

// the kept staging buffer back to the system (fp8_block_gemm_release)
hipError_t fp8gemm::release_host_staging()
{
    void* drop;
    {
        std::lock_guard<std::mutex> lock(g_staging_mutex);
        drop = g_staging;
        g_staging = nullptr;
        g_staging_bytes = 0;
    }
    return drop ? hipHostFree(drop) : hipSuccess;
}

extern "C" int fp8_gemm_host(unsigned short* c, const float* a, const float* b, const float* a_scale,
                             const float* b_scale, size_t m, size_t n, size_t k, int option)
{
    if (!c || !a || !b || !a_scale || !b_scale)
        return FP8GEMM_E_NULLPTR;
    if (m == 0 || n == 0 || k == 0 || k % 128 != 0)
        return FP8GEMM_E_SHAPE;
    if (m * k > 0x7FFFFFFFull || n * k > 0x7FFFFFFFull || m * n > 0x7FFFFFFFull)
        return FP8GEMM_E_TOOLARGE;
    // per-call options and a workspace of this call's own: no process-wide switch is touched
    fp8gemm_options opt{FP8GEMM_KERNEL_AUTO, -1, 0, -1, 0};
    if (option == 2)
        opt.kernel = FP8GEMM_KERNEL_SCALAR;
    else if (option >= 100 && option <= 100 + FP8GEMM_KERNEL_SKINNY)
        opt.kernel = option - 100;
    else if (option != 0 && option != 1)
        return FP8GEMM_E_KERNEL;
    const size_t nkb = k / 128, sn = (n + 127) / 128;
    const size_t ws_bytes = fp8_block_gemm_workspace_bytes_ex((int)m, (int)n, (int)k, &opt, 0);
    hipError_t e;
#define TRY(x)                 \
    do {                       \
        e = (x);               \
        if (e != hipSuccess)   \
            return (int)e;     \
    } while (0)
    StagingBuf staging;
    DeviceBuf device;
    Pipeline pipe(a, m * k, b, n * k);
    // behind the ring the scales, if they are small: a pageable copy of 200 KB takes up to 0.15 ms
    const size_t ring_bytes = pipe.slots * Pipeline::PIECE;  // two pieces at least
    const size_t scale_bytes = padded(nkb * m * 4) + nkb * sn * 4;
    const bool stage_scales = scale_bytes <= SCALES_STAGED;
    if (!staging.alloc(ring_bytes + (stage_scales ? scale_bytes : 0)))
        return (int)hipErrorOutOfMemory;
    pipe.staging = staging.p;
    {
        Workers workers(pipe);
        workers.start();
        const size_t o_b = padded(m * k), o_as = o_b + padded(n * k), o_bs = o_as + padded(nkb * m * 4),
                     o_c = o_bs + padded(nkb * sn * 4), o_ws = o_c + padded(m * n * 2);
        TRY(device.alloc(o_ws + ws_bytes));
        uint8_t* const d = static_cast<uint8_t*>(device.p);
        if (stage_scales) {  // laid out as on the device: one copy
            std::memcpy(staging.p + ring_bytes, a_scale, nkb * m * 4);
            std::memcpy(staging.p + ring_bytes + (o_bs - o_as), b_scale, nkb * sn * 4);
            TRY(hipMemcpyAsync(d + o_as, staging.p + ring_bytes, scale_bytes, hipMemcpyHostToDevice, nullptr));
        } else {
            TRY(hipMemcpy(d + o_as, a_scale, nkb * m * 4, hipMemcpyHostToDevice));
            TRY(hipMemcpy(d + o_bs, b_scale, nkb * sn * 4, hipMemcpyHostToDevice));
        }
        void* const dst[2] = {d, d + o_b};
        TRY(pipe.upload(dst, workers.count > 0));  // every value has been converted: the staging buffer is main's again
        const int rc = fp8_block_gemm_ex(d, d + o_b, reinterpret_cast<const float*>(d + o_as),
                                         reinterpret_cast<const float*>(d + o_bs), d + o_c, (int)m, (int)n, (int)k, &opt,
                                         ws_bytes ? d + o_ws : nullptr, ws_bytes, nullptr);
        if (rc != 0)
            return rc;
        TRY(download(c, d + o_c, m * n * 2, staging.p, ring_bytes));  // blocking: also the sync
        workers.join();
    }
#undef TRY
    return FP8GEMM_OK;
}
