/*
 * A stand-in libamdhip64.so.7 for CPU tests of libr9vx's launch plans: a
 * device of 256 compute units on which every launch succeeds and runs
 * nothing.  recorded(i, ...) gives the i-th launch's kernel name, grid and
 * block, in launch order.  Launches past HIP's limits (2^32 threads in a
 * dimension, 65535 workgroups in y and z) fail as there.
 */
#include <stddef.h>
#include <stdint.h>
#include <string.h>

typedef int hipError_t;
typedef void *hipStream_t;
typedef struct {
    uint32_t x, y, z;
} dim3;

#define INVALID_CONFIGURATION 9
#define MAX_KERNELS 4096
#define MAX_LAUNCHES 4096

static struct {
    const void *host;
    const char *name;
} kernels[MAX_KERNELS];
static struct {
    const char *name;
    dim3 g, b;
} launches[MAX_LAUNCHES];
static int n_kernels, n_launches;
static hipError_t last_error;
static void *modules[4];
static dim3 push_g, push_b;

int recorded(int i, const char **name, uint32_t *grid, uint32_t *block) {
    if (i < 0 || i >= n_launches) return 0;
    *name = launches[i].name;
    memcpy(grid, &launches[i].g, sizeof(dim3));
    memcpy(block, &launches[i].b, sizeof(dim3));
    return 1;
}
void record_clear(void) { n_launches = 0; }

void **__hipRegisterFatBinary(const void *data) {
    (void)data;
    return modules;
}
void __hipUnregisterFatBinary(void **m) { (void)m; }
void __hipRegisterFunction(void **m, const void *host, char *dev, const char *name, unsigned limit, void *tid,
                           void *bid, void *bdim, void *gdim, int *wsize) {
    (void)m, (void)dev, (void)limit, (void)tid, (void)bid, (void)bdim, (void)gdim, (void)wsize;
    if (n_kernels < MAX_KERNELS) kernels[n_kernels].host = host, kernels[n_kernels++].name = name;
}
void __hipRegisterVar(void **m, void *var, char *hvar, char *dvar, int ext, size_t size, int constant,
                      int global) {
    (void)m, (void)var, (void)hvar, (void)dvar, (void)ext, (void)size, (void)constant, (void)global;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t shmem, hipStream_t s) {
    (void)shmem, (void)s;
    push_g = g, push_b = b;
    return 0;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *shmem, hipStream_t *s) {
    *g = push_g, *b = push_b, *shmem = 0, *s = 0;
    return 0;
}
static int too_many(uint32_t g, uint32_t b) { return g == 0 || (uint64_t)g * b > 0xFFFFFFFFull; }
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t shmem, hipStream_t s) {
    const char *name = "?";
    (void)args, (void)shmem, (void)s;
    if (too_many(g.x, b.x) || too_many(g.y, b.y) || too_many(g.z, b.z) || g.y > 65535 || g.z > 65535)
        return last_error = INVALID_CONFIGURATION;
    for (int i = 0; i < n_kernels; ++i)
        if (kernels[i].host == f) name = kernels[i].name;
    if (n_launches < MAX_LAUNCHES) {
        launches[n_launches].name = name;
        launches[n_launches].g = g;
        launches[n_launches++].b = b;
    }
    return 0;
}
hipError_t hipGetDevice(int *dev) {
    *dev = 0;
    return 0;
}
hipError_t hipDeviceGetAttribute(int *v, int attr, int dev) {
    (void)attr, (void)dev;
    *v = 256;
    return 0;
}
hipError_t hipGetLastError(void) {
    hipError_t e = last_error;
    last_error = 0;
    return e;
}
const char *hipGetErrorString(hipError_t e) { return e == INVALID_CONFIGURATION ? "hipErrorInvalidConfiguration" : "?"; }
hipError_t hipGetSymbolAddress(void **p, const void *sym) {
    *p = (void *)sym;
    return 0;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, int kind, hipStream_t st) {
    (void)d, (void)s, (void)n, (void)kind, (void)st;
    return 0;
}
hipError_t hipMemcpy2DAsync(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, int kind,
                            hipStream_t st) {
    (void)d, (void)dp, (void)s, (void)sp, (void)w, (void)h, (void)kind, (void)st;
    return 0;
}
hipError_t hipMemcpyFromSymbolAsync(void *d, const void *sym, size_t n, size_t off, int kind, hipStream_t st) {
    (void)d, (void)sym, (void)n, (void)off, (void)kind, (void)st;
    return 0;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    (void)s;
    return 0;
}
