/* A program that carries its own stand-ins for the HIP runtime's calls (the library's references resolve to them first),
 * takes the decode kernels' entry points through many shapes without a device and prints what the launches asked for:
 * "kernels K raised R again A missing M" -- kernels launched with more than 64 KiB of dynamic LDS, kernels whose limit was
 * raised, times it was raised again for one, launches above their kernel's limit.
 * With arguments "rows n k split groups [tile]" (split 0 = automatic; groups 0 = a single problem, by the decode kernels if
 * split; tile = a tile variant) only that call, and the mangled names of the kernels that it launches.
 * With arguments "no-memory groups rows n k" only a grouped call in the process-wide workspace, which cannot be allocated: the
 * names of the kernels that it launches and "code C". */
#include <stddef.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "../include/fp8_block_gemm.h"

typedef struct { uint32_t x, y, z; } dim3;
static struct { dim3 grid, block; size_t lds; void *stream; } cfg;

enum { MAX_KERNELS = 1024 };
static struct { const void *kernel; int raised, times, large; } seen[MAX_KERNELS];
static int kernels, missing, say_names;
static struct { const void *kernel; const char *name; } known[8192];
static int registered;

void __hipRegisterFunction(void **modules, const void *kernel, char *a, const char *name, unsigned b, void *c, void *d, void *e,
                           void *f, int *g)
{
    (void)modules, (void)a, (void)b, (void)c, (void)d, (void)e, (void)f, (void)g;
    if (registered == 8192)
        abort();
    known[registered].kernel = kernel;
    known[registered++].name = name;
}

static int number_of(const void *kernel)
{
    int i = 0;
    while (i < kernels && seen[i].kernel != kernel)
        ++i;
    if (i == MAX_KERNELS)
        abort();
    if (i == kernels)
        seen[kernels++].kernel = kernel;
    return i;
}

int hipFuncSetAttribute(const void *kernel, int attribute, int value)
{
    const int i = number_of(kernel);
    (void)attribute;
    seen[i].raised = value;
    ++seen[i].times;
    return 0;
}
int hipLaunchKernel(const void *kernel, dim3 grid, dim3 block, void **args, size_t lds, void *stream)
{
    (void)grid, (void)block, (void)args, (void)stream;
    for (int i = 0; say_names && i < registered; ++i)
        if (known[i].kernel == kernel)
            printf("%s\n", known[i].name);
    if (lds > 64 * 1024) {
        const int i = number_of(kernel);
        seen[i].large = 1;
        missing += (size_t)seen[i].raised < lds;
    }
    return 0;
}
int __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, void *stream)
{
    cfg.grid = grid, cfg.block = block, cfg.lds = lds, cfg.stream = stream;
    return 0;
}
int __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, void **stream)
{
    *grid = cfg.grid, *block = cfg.block, *lds = cfg.lds, *stream = cfg.stream;
    return 0;
}
int hipGetDevice(int *device) { *device = 0; return 0; }
static int last_error;
int hipGetLastError(void)
{
    const int e = last_error;
    last_error = 0;
    return e;
}
int hipMalloc(void **out, size_t bytes)
{
    (void)out, (void)bytes;
    return last_error = 2; /* out of memory */
}
int hipStreamIsCapturing(void *stream, int *status) { (void)stream; *status = 0; return 0; }
int hipGetSymbolAddress(void **address, const void *symbol) { (void)symbol; *address = (void *)4096; return 0; }
/* what the look at the placement of workgroups reads back: eight XCDs in turn */
int hipMemcpy(void *to, const void *from, size_t bytes, int kind)
{
    (void)from, (void)kind;
    for (size_t i = 0; i < bytes / 4; ++i)
        ((uint32_t *)to)[i] = i % 8;
    return 0;
}

/* never read: nothing is launched */
static void *const p = (void *)(uintptr_t)(1 << 20), *const odd = (void *)(uintptr_t)((1 << 20) + 8);

/* groups problems of m rows each; c = not on a 16-byte boundary if odd_c, the first one with other rows if first > 0 */
static int grouped(int groups, int m, int first, int n, int k, int split, int odd_c)
{
    const void *ptr[64];
    void *out[64];
    int rows[64];
    for (int g = 0; g < groups; ++g) {
        ptr[g] = p;
        out[g] = odd_c ? odd : p;
        rows[g] = first > 0 && g == 0 ? first : m;
    }
    const fp8gemm_options opt = {FP8GEMM_KERNEL_AUTO, -1, split, -1, FP8GEMM_FLAG_WORKSPACE_ZEROED};
    return fp8_block_gemm_grouped_ex(groups, ptr, ptr, (const float *const *)ptr, (const float *const *)ptr, out, rows, n, k, &opt,
                                     p, (size_t)1 << 36, 0);
}

static int one_call(int words, char **word)
{
    const int m = atoi(word[1]), n = atoi(word[2]), k = atoi(word[3]), split = atoi(word[4]), groups = atoi(word[5]);
    const int tile = words > 6 ? atoi(word[6]) : -1;
    const fp8gemm_options opt = {split && tile < 0 ? FP8GEMM_KERNEL_SKINNY : FP8GEMM_KERNEL_AUTO, tile >= 0 ? tile : split ? 1 : -1,
                                 split, -1, FP8GEMM_FLAG_WORKSPACE_ZEROED};
    /* the first call looks at the placement of workgroups */
    fp8_block_gemm_ex(p, p, p, p, p, 32, 7168, 2048, 0, p, (size_t)1 << 32, 0);
    grouped(2, 16, 0, 7168, 2048, 2, 0);
    say_names = 1;
    return groups ? grouped(groups, m, 0, n, k, split, 0)
                  : fp8_block_gemm_ex(p, p, p, p, p, m, n, k, &opt, p, (size_t)1 << 32, 0);
}

static int no_memory(char **word)
{
    const int groups = atoi(word[2]), m = atoi(word[3]), n = atoi(word[4]), k = atoi(word[5]);
    const void *ptr[64];
    int rows[64];
    grouped(2, 16, 0, 7168, 2048, 2, 0); /* looks at the placement of workgroups */
    for (int g = 0; g < groups; ++g)
        ptr[g] = p, rows[g] = m;
    say_names = 1;
    const int rc = fp8_block_gemm_grouped(groups, ptr, ptr, (const float *const *)ptr, (const float *const *)ptr, (void *const *)ptr,
                                          rows, n, k, 0);
    printf("code %d\n", rc);
    return 0;
}

int main(int argc, char **argv)
{
    if (argc == 6 && !strcmp(argv[1], "no-memory"))
        return no_memory(argv);
    if (argc >= 6)
        return one_call(argc, argv);
    const int rows[] = {1, 8, 15, 16, 24, 31, 32, 40, 47, 48, 56, 63, 64};
    const int ns[] = {128, 1536, 4608, 7152, 7168, 16384, 28672, 33024, 49152, 65536, 65664, 131072};
    const int ks[] = {128, 384, 512, 1024, 2048, 4096, 7168, 8192};
    const int nrows = sizeof(rows) / sizeof(rows[0]), nns = sizeof(ns) / sizeof(ns[0]), nks = sizeof(ks) / sizeof(ks[0]);
    long calls = 0;
    for (int i = 0; i < nrows; ++i)
        for (int j = 0; j < nns; ++j)
            for (int l = 0; l < nks; ++l) {
                for (int variant = 1; variant <= 2; ++variant)
                    for (int split = 1; split <= 8; ++split)
                        for (int c = 0; c < 2; ++c) {
                            const fp8gemm_options opt = {FP8GEMM_KERNEL_SKINNY, variant, split, -1, FP8GEMM_FLAG_WORKSPACE_ZEROED};
                            calls += fp8_block_gemm_ex(p, p, p, p, c ? odd : p, rows[i], ns[j], ks[l], &opt, p, (size_t)1 << 32, 0) == 0;
                        }
                for (int groups = 2; groups <= 64; groups *= 2)
                    for (int split = 0; split <= 4; split += 4)
                        for (int ragged = 0; ragged < 2; ++ragged)
                            for (int c = 0; c < 2; ++c)
                                calls += grouped(groups, (rows[i] + 15) / 16 * 16, ragged ? (rows[i] > 1 ? rows[i] - 1 : 1) : 0, ns[j],
                                                 ks[l], split, c) == 0;
            }
    int large = 0, raised = 0, again = 0;
    for (int i = 0; i < kernels; ++i) {
        large += seen[i].large;
        raised += seen[i].times > 0;
        again += seen[i].times > 1 ? seen[i].times - 1 : 0;
    }
    printf("calls %ld kernels %d raised %d again %d missing %d\n", calls, large, raised, again, missing);
    return 0;
}
