/* A HIP runtime that runs nothing, for CPU tests of the library's host side:
 * it hands out host memory, fails an allocation on request, and keeps the
 * names of the kernels launched, with one 32-bit argument of a chosen kernel.
 * Loaded (RTLD_GLOBAL) before libqrhip.so, it takes the place of
 * libamdhip64's functions of the same names. */
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

enum { kMaxLaunch = 4096, kMaxKernel = 4096 };
static struct { const void *host; const char *name; } kernels[kMaxKernel];
static int nkernels;
static struct { const char *name; uint32_t arg, blocks; size_t shmem; } launches[kMaxLaunch];
static int nlaunches;
static const char *watch_name = "";
static int watch_arg;
static long malloc_left = -1;   /* allocations that succeed yet; -1: all */
static uint64_t malloc_bytes;   /* of hipMalloc, in all */
static int graphs_made, capturing, syncs_in_capture;

int stub_launches(void) { return nlaunches; }
const char *stub_name(int i) { return launches[i].name; }
uint32_t stub_arg(int i) { return launches[i].arg; }
uint32_t stub_blocks(int i) { return launches[i].blocks; }
uint32_t stub_shmem(int i) { return (uint32_t)launches[i].shmem; }
void stub_reset(void) { nlaunches = 0; malloc_bytes = 0; }
void stub_watch(const char *name, int arg) { watch_name = strdup(name); watch_arg = arg; }
void stub_fail_malloc_after(long n) { malloc_left = n; }
uint64_t stub_malloc_bytes(void) { return malloc_bytes; }
int stub_graphs_made(void) { return graphs_made; }
void stub_capture(int on) { capturing = on; }
int stub_syncs_in_capture(void) { return syncs_in_capture; }

typedef struct { uint32_t x, y, z; } dim3;

void **__hipRegisterFatBinary(const void *d) { (void)d; static void *h; return &h; }
void __hipUnregisterFatBinary(void **h) { (void)h; }
void __hipRegisterFunction(void **h, const void *host, char *device, const char *name, unsigned limit, void *tid,
                           void *bid, dim3 *block, dim3 *grid, int *w) {
    (void)h; (void)device; (void)limit; (void)tid; (void)bid; (void)block; (void)grid; (void)w;
    if (nkernels < kMaxKernel) {
        kernels[nkernels].host = host;
        kernels[nkernels++].name = strdup(name);
    }
}
void __hipRegisterVar(void **h, void *var, char *host, char *device, int ext, size_t size, int constant, int global) {
    (void)h; (void)var; (void)host; (void)device; (void)ext; (void)size; (void)constant; (void)global;
}
static dim3 cfg_grid, cfg_block;
static size_t cfg_shmem;
static void *cfg_stream;
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, void *st) {
    cfg_grid = g; cfg_block = b; cfg_shmem = s; cfg_stream = st;
    return 0;
}
int __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *s, void **st) {
    *g = cfg_grid; *b = cfg_block; *s = cfg_shmem; *st = cfg_stream;
    return 0;
}
int hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t shmem, void *stream) {
    (void)block; (void)stream;
    if (nlaunches == kMaxLaunch) return 1;
    const char *name = "";
    for (int i = 0; i < nkernels; ++i)
        if (kernels[i].host == f) name = kernels[i].name;
    launches[nlaunches].name = name;
    launches[nlaunches].blocks = grid.x;
    launches[nlaunches].shmem = shmem;
    launches[nlaunches].arg = 0;
    if (*watch_name && strstr(name, watch_name)) memcpy(&launches[nlaunches].arg, args[watch_arg], 4);
    ++nlaunches;
    return 0;
}

static int take(void **p, size_t n) {
    *p = NULL;
    if (malloc_left == 0) return 2; /* hipErrorOutOfMemory */
    if (malloc_left > 0) --malloc_left;
    *p = malloc(n ? n : 1);
    return *p ? 0 : 2;
}
int hipMalloc(void **p, size_t n) {
    if (capturing) ++syncs_in_capture;
    const int rc = take(p, n);
    if (!rc) malloc_bytes += n;
    return rc;
}
int hipFree(void *p) { free(p); return 0; }
int hipMallocAsync(void **p, size_t n, void *s) { (void)s; return take(p, n); }
int hipMallocFromPoolAsync(void **p, size_t n, void *pool, void *s) { (void)pool; (void)s; return take(p, n); }
int hipFreeAsync(void *p, void *s) { (void)s; free(p); return 0; }
int hipHostMalloc(void **p, size_t n, unsigned f) { (void)f; return take(p, n); }
int hipHostFree(void *p) { free(p); return 0; }
int hipMemPoolCreate(void **p, const void *props) { (void)props; static int pool; *p = &pool; return 0; }
int hipMemPoolSetAttribute(void *p, int a, void *v) { (void)p; (void)a; (void)v; return 0; }
int hipMemcpy(void *d, const void *s, size_t n, int kind) {
    (void)kind;
    if (capturing) ++syncs_in_capture;
    if (n) memcpy(d, s, n);
    return 0;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *st) {
    (void)d; (void)s; (void)n; (void)kind; (void)st;
    return 0;
}
int hipMemsetAsync(void *d, int v, size_t n, void *st) { (void)d; (void)v; (void)n; (void)st; return 0; }
int hipGetSymbolAddress(void **p, const void *s) { (void)s; static double scratch[1 << 19]; *p = scratch; return 0; }

int hipGetDevice(int *d) { *d = 0; return 0; }
int hipSetDevice(int d) { (void)d; return 0; }
int hipDeviceGetAttribute(int *v, int a, int d) { (void)a; (void)d; *v = 256; return 0; }
int hipGetDevicePropertiesR0600(void *p, int d) { (void)p; (void)d; return 1; }
int hipDeviceSynchronize(void) { return 0; }
int hipFuncSetAttribute(const void *f, int a, int v) { (void)f; (void)a; (void)v; return 0; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int b, size_t s) {
    (void)f; (void)b; (void)s; *n = 1; return 0;
}
const char *hipGetErrorString(int e) { return e == 2 ? "out of memory" : e ? "error" : "no error"; }
int hipGetLastError(void) { return 0; }

static int handle;
int hipStreamCreateWithFlags(void **s, unsigned f) { (void)f; *s = &handle; return 0; }
int hipStreamDestroy(void *s) { (void)s; return 0; }
int hipStreamSynchronize(void *s) { (void)s; return 0; }
int hipStreamWaitEvent(void *s, void *e, unsigned f) { (void)s; (void)e; (void)f; return 0; }
int hipStreamIsCapturing(void *s, int *status) { (void)s; *status = capturing; return 0; }
int hipGetStreamDeviceId(void *s) { (void)s; return 0; }
int hipEventCreate(void **e) { *e = &handle; return 0; }
int hipEventCreateWithFlags(void **e, unsigned f) { (void)f; *e = &handle; return 0; }
int hipEventDestroy(void *e) { (void)e; return 0; }
int hipEventRecord(void *e, void *s) { (void)e; (void)s; return 0; }
int hipEventSynchronize(void *e) { (void)e; return 0; }
int hipEventElapsedTime(float *ms, void *a, void *b) { (void)a; (void)b; *ms = 1.0f; return 0; }
int hipStreamBeginCapture(void *s, int mode) { (void)s; (void)mode; return 0; }
int hipStreamEndCapture(void *s, void **g) { (void)s; *g = &handle; return 0; }
int hipGraphInstantiate(void **x, void *g, void **n, char *log, size_t len) {
    (void)g; (void)n; (void)log; (void)len;
    ++graphs_made;
    *x = &handle;
    return 0;
}
int hipGraphLaunch(void *x, void *s) { (void)x; (void)s; return 0; }
int hipGraphDestroy(void *g) { (void)g; return 0; }
int hipGraphExecDestroy(void *x) { (void)x; return 0; }
