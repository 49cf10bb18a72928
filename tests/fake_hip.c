/* A HIP runtime that runs nothing, for CPU tests of the library's host code:
 * memory is the process's own, and a kernel launch calls a hook with the
 * kernel's name, its workgroups and its arguments.  Loaded with global
 * symbols before libcvl_hip.so, whose calls then bind to it. */
#include <stddef.h>
#include <stdlib.h>
#include <string.h>

typedef struct { unsigned x, y, z; } dim3;
typedef void (*hook_t)(const char *name, unsigned workgroups, void **args);

enum { kKernels = 1 << 16, kAllocs = 1 << 10 };
static struct { const void *fn; const char *name; } kernels[kKernels];
static int nkernels;
static struct { char *p; size_t bytes; int device; } allocs[kAllocs];
static int nallocs, device;
static hook_t hook;
static struct { dim3 grid, block; size_t shmem; void *stream; } pending;

void fake_set_hook(hook_t h) { hook = h; }
void fake_set_device(int d) { device = d; }
/* The device whose hipMalloc returned the memory at p, -1 for none. */
int fake_device_of(const void *p) {
    for (int i = 0; i < nallocs; i++)
        if ((char *)p >= allocs[i].p && (char *)p < allocs[i].p + allocs[i].bytes) return allocs[i].device;
    return -1;
}

void **__hipRegisterFatBinary(const void *data) { static void *module; (void)data; return &module; }
void __hipUnregisterFatBinary(void **m) { (void)m; }
void __hipRegisterFunction(void **m, const void *fn, char *device_fn, const char *name, unsigned limit, void *tid,
                           void *bid, void *block, void *grid, int *size) {
    (void)m; (void)device_fn; (void)limit; (void)tid; (void)bid; (void)block; (void)grid; (void)size;
    if (nkernels < kKernels) { kernels[nkernels].fn = fn; kernels[nkernels++].name = name; }
}
void __hipRegisterVar(void **m, void *var, char *host, const char *dev, int ext, size_t size, int c, int g) {
    (void)m; (void)var; (void)host; (void)dev; (void)ext; (void)size; (void)c; (void)g;
}
int __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shmem, void *stream) {
    pending.grid = grid; pending.block = block; pending.shmem = shmem; pending.stream = stream;
    return 0;
}
int __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shmem, void **stream) {
    *grid = pending.grid; *block = pending.block; *shmem = pending.shmem; *stream = pending.stream;
    return 0;
}
int hipLaunchKernel(const void *fn, dim3 grid, dim3 block, void **args, size_t shmem, void *stream) {
    (void)block; (void)shmem; (void)stream;
    const char *name = "";
    for (int i = 0; i < nkernels; i++)
        if (kernels[i].fn == fn) { name = kernels[i].name; break; }
    if (hook) hook(name, grid.x, args);
    return 0;
}

int hipGetDevice(int *d) { *d = device; return 0; }
int hipSetDevice(int d) { device = d; return 0; }
int hipGetLastError(void) { return 0; }
const char *hipGetErrorString(int e) { (void)e; return "fake"; }
int hipMalloc(void **p, size_t bytes) {
    *p = aligned_alloc(256, (bytes + 255) / 256 * 256);
    if (!*p || nallocs == kAllocs) return 2;
    allocs[nallocs].p = *p; allocs[nallocs].bytes = bytes; allocs[nallocs++].device = device;
    return 0;
}
int hipHostMalloc(void **p, size_t bytes, unsigned flags) {
    (void)flags;
    *p = calloc(1, bytes);
    return *p ? 0 : 2;
}
int hipHostGetDevicePointer(void **d, void *h, unsigned flags) { (void)flags; *d = h; return 0; }
int hipMemset(void *p, int v, size_t bytes) { memset(p, v, bytes); return 0; }
int hipMemsetAsync(void *p, int v, size_t bytes, void *stream) { (void)p; (void)v; (void)bytes; (void)stream; return 0; }
int hipMemcpyAsync(void *d, const void *s, size_t bytes, int kind, void *stream) {
    (void)d; (void)s; (void)bytes; (void)kind; (void)stream;
    return 0;
}
int hipStreamSynchronize(void *stream) { (void)stream; return 0; }
int hipDeviceGetAttribute(int *v, int attr, int d) { (void)attr; (void)d; *v = 256; return 0; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *v, const void *f, int threads, size_t shmem) {
    (void)f; (void)threads; (void)shmem;
    *v = 2;
    return 0;
}
