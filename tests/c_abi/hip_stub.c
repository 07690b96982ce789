/*
 * A HIP runtime for tests of host code without a GPU, preloaded over the real one: one gfx950
 * device whose memory is the host's, copies done at once, kernels that do nothing (what they
 * would have read back is zero). A launch of a kernel whose name holds the text in
 * PX_STUB_FAIL_LAUNCH fails with hipErrorLaunchFailure; launches of kernels whose name holds the
 * text in PX_STUB_COUNT_LAUNCH are counted in px_stub_launches, waits for a stream in
 * px_stub_waits.
 */
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>

#include <stdlib.h>
#include <string.h>

static struct { const void* host; const char* name; } kernels[4096];
static int kernel_count;
static hipError_t last;
long px_stub_launches, px_stub_waits;

hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int d) { return d ? hipErrorInvalidDevice : hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int d) {
    (void)d;
    memset(p, 0, sizeof *p);
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* left, size_t* total) { *left = *total = (size_t)1 << 36; return hipSuccess; }
/* device memory: its size before it, the bytes held in px_stub_live */
#define HEAD 64
size_t px_stub_live;
hipError_t hipMalloc(void** p, size_t n) {
    char* m = calloc(1, n + HEAD);
    *p = m ? m + HEAD : 0;
    if (!m) return last = hipErrorOutOfMemory;
    *(size_t*)m = n;
    px_stub_live += n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    if (!p) return hipSuccess;
    px_stub_live -= *(size_t*)((char*)p - HEAD);
    free((char*)p - HEAD);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned flags) {
    (void)flags;
    *p = calloc(1, n ? n : 1);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned flags) { (void)flags; *d = h; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned flags) { (void)flags; *s = malloc(1); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { (void)s; ++px_stub_waits; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { free(s); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t st) {
    (void)k, (void)st;
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipGetLastError(void) { const hipError_t e = last; last = hipSuccess; return e; }

hipError_t hipFuncSetAttribute(const void* f, hipFuncAttribute a, int v) {
    (void)f, (void)a, (void)v;
    return hipSuccess;
}

void** __hipRegisterFatBinary(const void* data) { (void)data; static void* h; return &h; }
void __hipUnregisterFatBinary(void** h) { (void)h; }
void __hipRegisterFunction(void** h, const void* host, char* dev, const char* name, unsigned t,
                           void* a, void* b, void* c, void* d, int* e) {
    (void)h, (void)dev, (void)t, (void)a, (void)b, (void)c, (void)d, (void)e;
    if (kernel_count < 4096) {
        kernels[kernel_count].host = host;
        kernels[kernel_count++].name = name;
    }
}
void __hipRegisterVar(void** h, void* v, char* hv, char* dv, int e, size_t n, int c, int g) {
    (void)h, (void)v, (void)hv, (void)dv, (void)e, (void)n, (void)c, (void)g;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, hipStream_t s) {
    (void)g, (void)b, (void)m, (void)s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, hipStream_t* s) {
    (void)g, (void)b;
    *m = 0;
    *s = 0;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void** args, size_t m, hipStream_t s) {
    (void)g, (void)b, (void)args, (void)m, (void)s;
    const char* fail = getenv("PX_STUB_FAIL_LAUNCH");
    const char* count = getenv("PX_STUB_COUNT_LAUNCH");
    for (int i = 0; i < kernel_count; ++i) {
        if (kernels[i].host != f) continue;
        if (count && *count && strstr(kernels[i].name, count)) ++px_stub_launches;
        if (fail && *fail && strstr(kernels[i].name, fail)) return last = hipErrorLaunchFailure;
    }
    return hipSuccess;
}
