/*
 * hip_stand_in.c -- the HIP entry points that libktm.so imports, on the host:
 * device memory is host memory under a limit, and kernel launches are written
 * down (kernel name, grid, workgroup, dynamic LDS) instead of run.  Loaded
 * with RTLD_GLOBAL before the library, it takes the runtime's place, so that
 * tests without a GPU can see which kernel a call launches, what it allocates
 * and what it does when an allocation fails.
 */
#include <hip/hip_runtime_api.h>

#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#define MAX_KERNELS 4096
#define MAX_BLOCKS 4096
#define MAX_RECORDS 65536

static struct { const void *host; const char *name; } kernels[MAX_KERNELS];
static int nkernels;
static struct { void *p; size_t bytes; } blocks[MAX_BLOCKS];
static size_t live, limit = SIZE_MAX, symbol_bytes = (size_t)256 << 20;
static struct { const char *name; uint32_t grid[3], block[3]; size_t lds; } launches[MAX_RECORDS];
static size_t allocations[MAX_RECORDS];
static int nlaunches, nallocations;
static struct { dim3 grid, block; size_t lds; hipStream_t s; } pushed;
static hipError_t last;

/* ---- what the tests ask ---- */
void standin_limit(size_t bytes) { limit = bytes; }
size_t standin_live(void) { return live; }
void standin_clear(void) { nlaunches = nallocations = 0; }
int standin_launches(void) { return nlaunches; }
int standin_allocations(void) { return nallocations; }
size_t standin_allocation(int i) { return allocations[i]; }
const char *standin_launch(int i, uint32_t *dims)
{
    memcpy(dims, launches[i].grid, 12);
    memcpy(dims + 3, launches[i].block, 12);
    dims[6] = (uint32_t)launches[i].lds;
    return launches[i].name;
}

/* ---- the code objects ---- */
void **__hipRegisterFatBinary(const void *data) { (void)data; return (void **)&kernels; }
void __hipUnregisterFatBinary(void **m) { (void)m; }
void __hipRegisterFunction(void **m, const void *host, char *dev, const char *name, unsigned threads,
                           void *a, void *b, void *c, void *d, int *e)
{
    (void)m; (void)dev; (void)threads; (void)a; (void)b; (void)c; (void)d; (void)e;
    if (nkernels < MAX_KERNELS) {
        kernels[nkernels].host = host;
        kernels[nkernels++].name = name;
    }
}
void __hipRegisterVar(void **m, void *v, char *host, char *dev, int ext, size_t n, int con, int global)
{
    (void)m; (void)v; (void)host; (void)dev; (void)ext; (void)n; (void)con; (void)global;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s)
{
    pushed.grid = grid; pushed.block = block; pushed.lds = lds; pushed.s = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *s)
{
    *grid = pushed.grid; *block = pushed.block; *lds = pushed.lds; *s = pushed.s;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t lds, hipStream_t s)
{
    (void)args; (void)s;
    const char *name = "?";
    for (int i = 0; i < nkernels; ++i)
        if (kernels[i].host == f) name = kernels[i].name;
    if (nlaunches < MAX_RECORDS) {
        const uint32_t g[3] = {grid.x, grid.y, grid.z}, b[3] = {block.x, block.y, block.z};
        launches[nlaunches].name = name;
        memcpy(launches[nlaunches].grid, g, sizeof g);
        memcpy(launches[nlaunches].block, b, sizeof b);
        launches[nlaunches++].lds = lds;
    }
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *f, hipFuncAttribute a, int v)
{
    (void)f; (void)a; (void)v;
    return hipSuccess;
}

/* ---- memory ---- */
hipError_t hipMalloc(void **p, size_t bytes)
{
    *p = NULL;
    if (bytes > limit || live > limit - bytes) return last = hipErrorOutOfMemory;
    for (int i = 0; i < MAX_BLOCKS; ++i) {
        if (blocks[i].p) continue;
        if (!(*p = calloc(1, bytes ? bytes : 1))) return last = hipErrorOutOfMemory;
        blocks[i].p = *p;
        blocks[i].bytes = bytes;
        live += bytes;
        if (nallocations < MAX_RECORDS) allocations[nallocations++] = bytes;
        return hipSuccess;
    }
    return last = hipErrorOutOfMemory;
}
hipError_t hipFree(void *p)
{
    if (!p) return hipSuccess;
    for (int i = 0; i < MAX_BLOCKS; ++i) {
        if (blocks[i].p != p) continue;
        live -= blocks[i].bytes;
        blocks[i].p = NULL;
        free(p);
        return hipSuccess;
    }
    return last = hipErrorInvalidValue;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned flags)
{
    (void)flags;
    return (*p = malloc(bytes ? bytes : 1)) ? hipSuccess : (last = hipErrorOutOfMemory);
}
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k)
{
    (void)k;
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st)
{
    (void)st;
    return hipMemcpy(d, s, n, k);
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t s)
{
    (void)s;
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *symbol)
{
    static void *space;
    (void)symbol;
    if (!space) space = calloc(1, symbol_bytes);
    return (*p = space) ? hipSuccess : (last = hipErrorOutOfMemory);
}

/* ---- device, streams, events ---- */
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int d) { return d ? (last = hipErrorInvalidDevice) : hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
int hipGetStreamDeviceId(hipStream_t s) { (void)s; return 0; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int d)   /* the R0600 form */
{
    (void)d;
    memset(p, 0, sizeof *p);
    strcpy(p->gcnArchName, "gfx950");
    p->warpSize = 64;
    p->multiProcessorCount = 256;
    p->maxThreadsPerBlock = 1024;
    p->sharedMemPerBlock = 160 * 1024;
    return hipSuccess;
}
hipError_t hipGetLastError(void)
{
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipStreamCreate(hipStream_t *s) { return (*s = malloc(1)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipStreamDestroy(hipStream_t s) { free(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned f) { (void)s; (void)e; (void)f; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return (*e = malloc(1)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { (void)e; (void)s; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) { (void)a; (void)b; *ms = 0.0f; return hipSuccess; }
