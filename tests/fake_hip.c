/* A HIP runtime for tests on the CPU: device memory is addresses that nothing
 * reads, kernels are not run, and every allocation, release and launch is
 * recorded.  Loaded before the library (RTLD_GLOBAL), it shows what a call
 * does on the host: the memory it takes and gives back, the grids it launches. */
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>

#include <stdint.h>
#include <stdio.h>
#include <string.h>

enum { MAX = 65536 };
static struct { uintptr_t p; size_t n; int live; } allocs[MAX];
static int n_allocs;
static struct { const void *f; const char *name; } kernels[MAX];
static int n_kernels;
static struct { const char *name; dim3 grid, block; size_t lds; } launches[MAX];
static int n_launches;
static uintptr_t next = (uintptr_t)1 << 40;
static dim3 cfg_grid, cfg_block;
static size_t cfg_lds;
static hipStream_t cfg_stream;

/* what the tests set: refuse memory; the call's stream is being captured;
 * another stream is, in global mode, which a call that takes, gives back or
 * waits for something in that mode breaks */
int fake_refuse_malloc, fake_capturing, fake_other_capture;
int fake_broken_captures;
static hipStreamCaptureMode mode = hipStreamCaptureModeGlobal;
static int unsafe(void) {
    if (!fake_other_capture || mode == hipStreamCaptureModeRelaxed) return 0;
    return ++fake_broken_captures;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *m) {
    hipStreamCaptureMode was = mode;
    return mode = *m, *m = was, hipSuccess;
}

int fake_allocs(void) { return n_allocs; }
int fake_live(int i) { return allocs[i].live; }
size_t fake_alloc_bytes(int i) { return allocs[i].n; }
int fake_launches(void) { return n_launches; }
const char *fake_launch(int i, unsigned v[6]) {
    v[0] = launches[i].grid.x, v[1] = launches[i].grid.y, v[2] = launches[i].grid.z;
    v[3] = launches[i].block.x, v[4] = launches[i].block.y, v[5] = launches[i].block.z;
    return launches[i].name;
}

hipError_t hipMalloc(void **p, size_t n) {
    if (unsafe()) return hipErrorStreamCaptureUnsupported;
    if (fake_refuse_malloc || n_allocs == MAX) return hipErrorOutOfMemory;
    allocs[n_allocs].p = next, allocs[n_allocs].n = n, allocs[n_allocs].live = 1;
    ++n_allocs;
    *p = (void *)next;
    next += (n + 4095) & ~(size_t)4095;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    if (unsafe()) return hipErrorStreamCaptureUnsupported;
    for (int i = 0; i < n_allocs; ++i)
        if (allocs[i].p == (uintptr_t)p && allocs[i].live) {
            allocs[i].live = 0;
            return hipSuccess;
        }
    return p ? hipErrorInvalidValue : hipSuccess;
}
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int d) {
    return *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 0, hipSuccess;
}
#undef hipGetDeviceProperties
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int d) {
    memset(p, 0, sizeof *p);
    strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
    return unsafe() ? hipErrorStreamCaptureUnsupported : hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *c) {
    return *c = fake_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone,
           hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t e) { return "fake HIP error"; }
hipError_t hipGetSymbolAddress(void **p, const void *s) { return hipMalloc(p, 64 << 20); }
hipError_t hipFuncSetAttribute(const void *f, hipFuncAttribute a, int v) { return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) { return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t t) {
    return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h,
                            hipMemcpyKind k, hipStream_t t) {
    return hipSuccess;
}
hipError_t hipMemset(void *p, int v, size_t n) {
    return unsafe() ? hipErrorStreamCaptureUnsupported : hipSuccess;
}
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t s) { return hipSuccess; }

/* the compiler's registration and launch entries */
static void *module;
void **__hipRegisterFatBinary(const void *d) { return &module; }
void __hipUnregisterFatBinary(void **m) {}
void __hipRegisterFunction(void **m, const void *host, char *dev, const char *name, unsigned tl,
                           void *tid, void *bid, dim3 *bd, dim3 *gd, int *ws) {
    if (n_kernels < MAX) kernels[n_kernels].f = host, kernels[n_kernels++].name = name;
}
void __hipRegisterVar(void **m, void *v, char *h, char *d, int e, size_t n, int c, int g) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
    return cfg_grid = g, cfg_block = b, cfg_lds = lds, cfg_stream = s, hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s) {
    return *g = cfg_grid, *b = cfg_block, *lds = cfg_lds, *s = cfg_stream, hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t lds,
                           hipStream_t s) {
    const char *name = "?";
    for (int i = 0; i < n_kernels; ++i)
        if (kernels[i].f == f) name = kernels[i].name;
    if (n_launches < MAX) {
        launches[n_launches].name = name, launches[n_launches].grid = g;
        launches[n_launches].block = b, launches[n_launches].lds = lds;
        ++n_launches;
    }
    return hipSuccess;
}
