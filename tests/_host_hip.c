/* A HIP runtime without a GPU, for tests of the library's host code: device
 * memory is address space that is never backed until it is copied to, kernel
 * launches are reported to a callback and do nothing, and every operation put
 * on a stream counts as in flight until something waits. */
#define _GNU_SOURCE
#include <stdint.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>

typedef struct {
    uint32_t x, y, z;
} dim3_t;
typedef int err_t;
enum { OK = 0, OOM = 2, UNSUPPORTED = 801 };

/* ---- the test's side ---- */
typedef void (*launch_fn)(const char* name, uint32_t grid, uint32_t block, void** args);
static launch_fn on_launch;
static int mallocs, fail_from = -1; /* allocations so far; the first one that fails */
static uint64_t live, limit = ~0ull; /* bytes allocated, and how many may be */
static uint64_t said_free = 288ull << 30; /* what hipMemGetInfo says */
static int in_flight;                /* operations nothing has waited for */

void host_hip_on_launch(launch_fn f) { on_launch = f; }
void host_hip_fail_from(int n) { fail_from = n < 0 ? -1 : mallocs + n; }
void host_hip_limit(uint64_t bytes) { limit = bytes; }
void host_hip_say_free(uint64_t bytes) { said_free = bytes; }
uint64_t host_hip_live(void) { return live; }
int host_hip_mallocs(void) { return mallocs; }
int host_hip_in_flight(void) { return in_flight; }

enum { MAXBLOCKS = 4096 };
static struct {
    char* p;
    size_t n;
} blocks[MAXBLOCKS];

/* bytes of an allocation behind address p (0: not device memory) */
uint64_t host_hip_room(uintptr_t p)
{
    for (int i = 0; i < MAXBLOCKS; ++i)
        if (blocks[i].p && p >= (uintptr_t)blocks[i].p && p < (uintptr_t)blocks[i].p + blocks[i].n)
            return (uintptr_t)blocks[i].p + blocks[i].n - p;
    return 0;
}

/* ---- memory ---- */
err_t hipMalloc(void** p, size_t n)
{
    const int k = mallocs++;
    if ((fail_from >= 0 && k >= fail_from) || n > limit || live > limit - n) return OOM;
    int i = 0;
    while (i < MAXBLOCKS && blocks[i].p) ++i;
    void* m = i < MAXBLOCKS ? mmap(0, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0)
                            : MAP_FAILED;
    if (m == MAP_FAILED) return OOM;
    blocks[i].p = m;
    blocks[i].n = n;
    live += n;
    *p = m;
    return OK;
}
err_t hipFree(void* p)
{
    for (int i = 0; i < MAXBLOCKS; ++i)
        if (p && blocks[i].p == p) {
            munmap(p, blocks[i].n);
            live -= blocks[i].n;
            blocks[i].p = 0;
        }
    return OK;
}
err_t hipHostMalloc(void** p, size_t n, unsigned flags) { return (*p = calloc(1, n)) ? OK : OOM; }
err_t hipHostFree(void* p) { free(p); return OK; }
err_t hipMemGetInfo(size_t* fr, size_t* total)
{
    *total = 288ull << 30;
    *fr = said_free;
    return OK;
}
static void copy(void* dst, const void* src, size_t n, int kind)
{
    /* device memory that nothing was copied to reads as zeros */
    if (kind != 3) memcpy(dst, src, n);
}
err_t hipMemcpy(void* dst, const void* src, size_t n, int kind) { copy(dst, src, n, kind); in_flight = 0; return OK; }
err_t hipMemcpyAsync(void* dst, const void* src, size_t n, int kind, void* s)
{
    copy(dst, src, n, kind);
    ++in_flight;
    return OK;
}
err_t hipGetSymbolAddress(void** p, const void* sym) { return UNSUPPORTED; }

/* ---- streams, events, graphs ---- */
err_t hipDeviceSynchronize(void) { in_flight = 0; return OK; }
err_t hipStreamSynchronize(void* s) { in_flight = 0; return OK; }
err_t hipEventSynchronize(void* e) { return OK; }
err_t hipStreamCreateWithFlags(void** s, unsigned f) { *s = malloc(1); return OK; }
err_t hipStreamDestroy(void* s) { free(s); return OK; }
err_t hipStreamWaitEvent(void* s, void* e, unsigned f) { return OK; }
err_t hipEventCreate(void** e) { *e = malloc(1); return OK; }
err_t hipEventCreateWithFlags(void** e, unsigned f) { return hipEventCreate(e); }
err_t hipEventDestroy(void* e) { free(e); return OK; }
err_t hipEventRecord(void* e, void* s) { return OK; }
err_t hipEventElapsedTime(float* ms, void* a, void* b) { *ms = 1.0f; return OK; }
err_t hipStreamBeginCapture(void* s, int mode) { return UNSUPPORTED; }
err_t hipStreamEndCapture(void* s, void** g) { return UNSUPPORTED; }
err_t hipGraphInstantiate(void** e, void* g, void* n, char* log, size_t size) { return UNSUPPORTED; }
err_t hipGraphLaunch(void* e, void* s) { return UNSUPPORTED; }
err_t hipGraphDestroy(void* g) { return OK; }
err_t hipGraphExecDestroy(void* e) { return OK; }

/* ---- device and errors ---- */
err_t hipGetDevice(int* d) { *d = 0; return OK; }
err_t hipSetDevice(int d) { return OK; }
err_t hipGetLastError(void) { return OK; }
const char* hipGetErrorString(err_t e) { return e == OOM ? "out of memory" : "not supported"; }

/* ---- kernels ---- */
enum { MAXKERNELS = 1 << 15 };
static struct {
    const void* f;
    const char* name;
} kernels[MAXKERNELS];
static int nkernels;
static struct {
    dim3_t grid, block;
    size_t lds;
    void* s;
} call;

void** __hipRegisterFatBinary(const void* data)
{
    static void* module;
    return &module;
}
void __hipUnregisterFatBinary(void** m) {}
void __hipRegisterFunction(void** m, const void* f, char* dev, const char* name, unsigned limit_, void* a, void* b,
                           void* c, void* d, int* e)
{
    if (nkernels < MAXKERNELS) {
        kernels[nkernels].f = f;
        kernels[nkernels++].name = name;
    }
}
void __hipRegisterVar(void** m, void* v, char* dev, const char* name, int ext, size_t n, int c, int g) {}
err_t __hipPushCallConfiguration(dim3_t grid, dim3_t block, size_t lds, void* s)
{
    call.grid = grid;
    call.block = block;
    call.lds = lds;
    call.s = s;
    return OK;
}
err_t __hipPopCallConfiguration(dim3_t* grid, dim3_t* block, size_t* lds, void** s)
{
    *grid = call.grid;
    *block = call.block;
    *lds = call.lds;
    *s = call.s;
    return OK;
}
err_t hipLaunchKernel(const void* f, dim3_t grid, dim3_t block, void** args, size_t lds, void* s)
{
    ++in_flight;
    for (int i = 0; i < nkernels; ++i)
        if (kernels[i].f == f) {
            if (on_launch) on_launch(kernels[i].name, grid.x, block.x, args);
            return OK;
        }
    return UNSUPPORTED;
}
