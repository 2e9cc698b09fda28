/* A HIP runtime without a device, for tests of the library's host code on the CPU: memory is host
 * memory, copies copy, kernels are written down by name and not run.  Which call fails, and with
 * what, is set by the test.  Built with the soname of the HIP runtime and loaded before the library
 * (host_hip.py), so that it serves the library's calls in that process. */
#include <hip/hip_runtime_api.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>

enum { MAX_FUNCTIONS = 4096, MAX_LAUNCHES = 1 << 16, MAX_BLOCKS = 1 << 14 };
static struct { const void *fn; const char *name; } functions[MAX_FUNCTIONS];
static int n_functions;
static const char *launches[MAX_LAUNCHES];
static dim3 grids[MAX_LAUNCHES];
static int n_launches;
static struct { void *p; size_t bytes; } blocks[MAX_BLOCKS];
static int n_blocks, n_pinned, blocks_per_cu = 1;
static size_t allocated, malloc_limit = (size_t)-1;
static char failing[64];
static hipError_t last_error;
static struct { dim3 grid, block; size_t lds; hipStream_t stream; } config;

/* ---- what a test sets and reads ---- */
void host_hip_malloc_limit(size_t bytes) { malloc_limit = bytes; } /* larger requests fail */
void host_hip_fail_kernel(const char *part) { strncpy(failing, part, sizeof(failing) - 1); }
void host_hip_clear(void) { n_launches = 0; }
int host_hip_launches(void) { return n_launches; }
const char *host_hip_launch(int i) { return launches[i]; }
unsigned host_hip_workgroups(int i) { return grids[i].x * grids[i].y * grids[i].z; }
void host_hip_blocks_per_cu(int n) { blocks_per_cu = n; } /* of every kernel; asked for once per kernel and size of LDS */
size_t host_hip_allocated(void) { return allocated; }
int host_hip_pinned(void) { return n_pinned; } /* requests for pinned memory so far */

static hipError_t done(hipError_t e) {
    if (e != hipSuccess) last_error = e;
    return e;
}

/* ---- registration and launches ---- */
void **__hipRegisterFatBinary(const void *data) { static void *h; h = (void *)data; return &h; }
void __hipUnregisterFatBinary(void **m) { (void)m; }
void __hipRegisterFunction(void **m, const void *host, char *dev, const char *name, unsigned limit,
                           void *tid, void *bid, void *bdim, void *gdim, int *ws) {
    (void)m; (void)dev; (void)limit; (void)tid; (void)bid; (void)bdim; (void)gdim; (void)ws;
    if (n_functions == MAX_FUNCTIONS) abort();
    functions[n_functions].fn = host;
    functions[n_functions++].name = name;
}
void __hipRegisterVar(void **m, void *var, char *host, char *dev, int ext, size_t size, int c, int global) {
    (void)m; (void)var; (void)host; (void)dev; (void)ext; (void)size; (void)c; (void)global;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s) {
    config.grid = grid; config.block = block; config.lds = lds; config.stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *s) {
    *grid = config.grid; *block = config.block; *lds = config.lds; *s = config.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *fn, dim3 grid, dim3 block, void **args, size_t lds, hipStream_t s) {
    (void)args; (void)s;
    const char *name = "?";
    for (int i = 0; i < n_functions; ++i)
        if (functions[i].fn == fn) name = functions[i].name;
    if (failing[0] && strstr(name, failing)) return done(hipErrorLaunchFailure);
    if (!grid.x || !grid.y || !grid.z || !block.x || block.x * block.y * block.z > 1024 || lds > 160 * 1024)
        return done(hipErrorInvalidConfiguration);
    if (n_launches < MAX_LAUNCHES) {
        launches[n_launches] = name;
        grids[n_launches++] = grid;
    }
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *f, hipFuncAttribute a, int v) { (void)f; (void)a; (void)v; return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int threads, size_t lds) {
    (void)f; (void)threads; (void)lds;
    *n = blocks_per_cu;
    return hipSuccess;
}
hipError_t hipGetLastError(void) { hipError_t e = last_error; last_error = hipSuccess; return e; }
const char *hipGetErrorString(hipError_t e) {
    return e == hipErrorOutOfMemory ? "out of memory" : e == hipErrorLaunchFailure ? "launch failure" : "error";
}

/* ---- memory (address space only until it is touched) ---- */
static hipError_t give(void **p, size_t bytes) {
    if (bytes > malloc_limit || n_blocks == MAX_BLOCKS) return done(hipErrorOutOfMemory);
    void *m = mmap(NULL, bytes ? bytes : 1, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (m == MAP_FAILED) return done(hipErrorOutOfMemory);
    blocks[n_blocks].p = m;
    blocks[n_blocks++].bytes = bytes ? bytes : 1;
    *p = m;
    return hipSuccess;
}
static size_t take(void *p) {
    for (int i = 0; i < n_blocks; ++i)
        if (blocks[i].p == p) {
            const size_t bytes = blocks[i].bytes;
            munmap(p, bytes);
            blocks[i] = blocks[--n_blocks];
            return bytes;
        }
    if (p) abort(); /* freed twice, or never allocated */
    return 0;
}
hipError_t hipMalloc(void **p, size_t bytes) {
    const hipError_t e = give(p, bytes);
    if (e == hipSuccess) allocated += bytes ? bytes : 1;
    return e;
}
hipError_t hipFree(void *p) { allocated -= take(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned flags) { (void)flags; ++n_pinned; return give(p, bytes); }
hipError_t hipHostFree(void *p) { take(p); return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) {
    (void)k;
    if (n <= (size_t)64 << 20) memcpy(d, s, n); /* (what is larger is never looked at) */
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st) {
    (void)st;
    return hipMemcpy(d, s, n, k);
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t s) {
    (void)s;
    if (v || n <= (size_t)64 << 20) memset(d, v, n); /* (blocks are zero to begin with) */
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *symbol) {
    (void)symbol;
    static char array[4 << 20];
    *p = array;
    return hipSuccess;
}

/* ---- device, streams, events, graphs ---- */
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int d) { (void)d; return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int d) { /* (a macro of the header names the version) */
    (void)d;
    memset(p, 0, sizeof(*p));
    strcpy(p->name, "no device");
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned f) { (void)f; *s = (hipStream_t)&config; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode m) { (void)s; (void)m; return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g) { (void)s; *g = (hipGraph_t)&config; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, hipGraphNode_t *n, char *log, size_t size) {
    (void)g; (void)n; (void)log; (void)size;
    *e = (hipGraphExec_t)&config;
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t s) { (void)e; (void)s; return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { (void)g; return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { (void)e; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)&config; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { (void)e; (void)s; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) { (void)a; (void)b; *ms = 1.f; return hipSuccess; }
