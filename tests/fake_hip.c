/* fake_hip.c -- stands in for the HIP runtime in a process without a GPU: loaded
 * before libwtc.so with its symbols global, it answers the library's runtime
 * calls itself.  "Device" memory is host memory, copies are made at once, and a
 * kernel does not run: its name is put on a list.  So a test sees what the host
 * code would allocate, copy and launch, and the host code's results are zero. */
#include <stdlib.h>
#include <string.h>

#include <hip/hip_runtime_api.h>

#define MAXK 4096
#define MAXL (1 << 16)
static struct { const void *fn; const char *name; } kernels[MAXK];
static int n_kernels;
static const char *launched[MAXL];
static int n_launched;
static unsigned long long allocs, copies;

int fake_launches(void) { return n_launched; }
const char *fake_launch(int i) { return launched[i]; }
unsigned long long fake_allocs(void) { return allocs; }
unsigned long long fake_copies(void) { return copies; }
void fake_reset(void) {
    n_launched = 0;
    allocs = copies = 0;
}

void **__hipRegisterFatBinary(const void *data) {
    static void *handle;
    (void)data;
    return &handle;
}
void __hipUnregisterFatBinary(void **m) { (void)m; }
void __hipRegisterFunction(void **m, const void *fn, char *dev, const char *name, unsigned limit, void *tid, void *bid,
                           void *bdim, void *gdim, int *wsize) {
    (void)m, (void)dev, (void)limit, (void)tid, (void)bid, (void)bdim, (void)gdim, (void)wsize;
    if (n_kernels < MAXK) kernels[n_kernels].fn = fn, kernels[n_kernels++].name = name;
}
void __hipRegisterVar(void **m, void *var, char *host, char *dev, int ext, size_t size, int constant, int global) {
    (void)m, (void)var, (void)host, (void)dev, (void)ext, (void)size, (void)constant, (void)global;
}
static __thread struct { dim3 g, b; size_t shm; hipStream_t st; } conf;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t shm, hipStream_t st) {
    conf.g = g, conf.b = b, conf.shm = shm, conf.st = st;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *shm, hipStream_t *st) {
    *g = conf.g, *b = conf.b, *shm = conf.shm, *st = conf.st;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *fn, dim3 g, dim3 b, void **args, size_t shm, hipStream_t st) {
    const char *name = "?";
    (void)g, (void)b, (void)args, (void)shm, (void)st;
    for (int i = 0; i < n_kernels; i++)
        if (kernels[i].fn == fn) name = kernels[i].name;
    if (n_launched < MAXL) launched[n_launched++] = name;
    return hipSuccess;
}

hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int d) { return d ? hipErrorInvalidDevice : hipSuccess; }
int hipGetStreamDeviceId(hipStream_t st) { return (void)st, 0; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int d) {
    (void)d;
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 163840;
    return hipSuccess;
}
#undef hipGetDeviceProperties
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int d) {
    (void)d;
    memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    p->sharedMemPerBlock = 163840;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *fn, hipFuncAttribute a, int v) { return (void)fn, (void)a, (void)v, hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *fn, int threads, size_t shm) {
    (void)fn, (void)threads, (void)shm;
    return *n = 2, hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *sym) { return (void)sym, *p = calloc(1, 4096), hipSuccess; }

hipError_t hipMalloc(void **p, size_t bytes) {
    allocs += bytes;
    return (*p = malloc(bytes)) ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void *p) { return free(p), hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned flags) {
    (void)flags;
    return (*p = calloc(1, bytes)) ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) { return free(p), hipSuccess; }
hipError_t hipMemcpy(void *dst, const void *src, size_t bytes, hipMemcpyKind k) {
    (void)k;
    copies += bytes;
    return memcpy(dst, src, bytes), hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes, hipMemcpyKind k, hipStream_t st) {
    return (void)st, hipMemcpy(dst, src, bytes, k);
}
hipError_t hipMemsetAsync(void *p, int v, size_t bytes, hipStream_t st) { return (void)st, memset(p, v, bytes), hipSuccess; }

static int handle;
hipError_t hipStreamCreateWithFlags(hipStream_t *st, unsigned f) { return (void)f, *st = (hipStream_t)&handle, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t st) { return (void)st, hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t st) { return (void)st, hipSuccess; }
hipError_t hipStreamQuery(hipStream_t st) { return (void)st, hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t st, hipEvent_t e, unsigned f) { return (void)st, (void)e, (void)f, hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return *e = (hipEvent_t)&handle, hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned f) { return (void)f, hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return (void)e, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t st) { return (void)e, (void)st, hipSuccess; }
hipError_t hipEventQuery(hipEvent_t e) { return (void)e, hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { return (void)e, hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) { return (void)a, (void)b, *ms = 0, hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t st, hipStreamCaptureMode m) { return (void)st, (void)m, hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t st, hipGraph_t *g) { return (void)st, *g = (hipGraph_t)&handle, hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, hipGraphNode_t *n, char *log, size_t size) {
    return (void)g, (void)n, (void)log, (void)size, *e = (hipGraphExec_t)&handle, hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t st) { return (void)e, (void)st, hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { return (void)g, hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { return (void)e, hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "error"; }
