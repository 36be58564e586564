/* The HIP runtime's host entry points that libqcdhip.so calls, in host memory:
 * allocations come from calloc, copies and clears happen at once, kernels are
 * not run.  Every call is noted, and allocations can be made to fail, so that
 * the library's host side (error paths, order of work on streams) is tested
 * without a GPU.  Loaded with RTLD_GLOBAL before libqcdhip.so. */
#include <pthread.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

typedef int hipError_t;
typedef struct {
    uint32_t x, y, z;
} dim3;
enum { hipSuccess = 0, hipErrorOutOfMemory = 2 };

static pthread_mutex_t lock = PTHREAD_MUTEX_INITIALIZER;
static char* text;
static size_t used, room;
static size_t malloc_most = SIZE_MAX, host_most = SIZE_MAX;
static __thread hipError_t last;

static hipError_t note(hipError_t e, const char* fmt, uint64_t a, uint64_t b, uint64_t c)
{
    pthread_mutex_lock(&lock);
    if (used + 160 > room) {
        room = 2 * room + (1 << 16);
        text = realloc(text, room);
    }
    used += (size_t)snprintf(text + used, 120, fmt, (unsigned long long)a, (unsigned long long)b, (unsigned long long)c);
    used += (size_t)snprintf(text + used, 16, e ? " failed\n" : "\n");
    pthread_mutex_unlock(&lock);
    if (e) last = e;
    return e;
}

/* for the tests */
const char* fake_log(void) { return text ? text : ""; }
void fake_clear(void)
{
    used = 0;
    if (text) text[0] = 0;
}
void fake_limits(size_t device_bytes, size_t host_bytes)
{
    malloc_most = device_bytes;
    host_most = host_bytes;
}

static void* grab(size_t n)
{
    void* p = NULL;
    if (posix_memalign(&p, 4096, n ? n : 1)) return NULL;
    memset(p, 0, n);
    return p;
}
hipError_t hipMalloc(void** p, size_t n)
{
    *p = n <= malloc_most ? grab(n) : NULL;
    return note(*p ? hipSuccess : hipErrorOutOfMemory, "malloc %llu", n, 0, 0);
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned flags)
{
    *p = n <= host_most ? grab(n) : NULL;
    return note(*p ? hipSuccess : hipErrorOutOfMemory, "hostmalloc %llu flags %llu", n, flags, 0);
}
hipError_t hipFree(void* p)
{
    free(p);
    return hipSuccess;
}
hipError_t hipHostFree(void* p)
{
    free(p);
    return note(hipSuccess, "hostfree", 0, 0, 0);
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, int kind)
{
    memcpy(d, s, n);
    return note(hipSuccess, "copy kind %llu bytes %llu", (uint64_t)kind, n, 0);
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void* st)
{
    memcpy(d, s, n);
    return note(hipSuccess, "copy kind %llu bytes %llu on %llx", (uint64_t)kind, n, (uint64_t)(uintptr_t)st);
}
hipError_t hipMemset(void* d, int v, size_t n)
{
    memset(d, v, n);
    return note(hipSuccess, "clear bytes %llu", n, 0, 0);
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, void* st)
{
    memset(d, v, n);
    return note(hipSuccess, "clear bytes %llu on %llx", n, (uint64_t)(uintptr_t)st, 0);
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void** args, size_t lds, void* st)
{
    (void)f, (void)b, (void)args, (void)lds;
    return note(hipSuccess, "launch %llu on %llx", g.x, (uint64_t)(uintptr_t)st, 0);
}
hipError_t hipExtLaunchKernel(const void* f, dim3 g, dim3 b, void** args, size_t lds, void* st, void* e0, void* e1, int flags)
{
    (void)e0, (void)e1, (void)flags;
    return hipLaunchKernel(f, g, b, args, lds, st);
}
hipError_t hipStreamSynchronize(void* st) { return note(hipSuccess, "wait on %llx", (uint64_t)(uintptr_t)st, 0, 0); }
hipError_t hipDeviceSynchronize(void) { return note(hipSuccess, "wait", 0, 0, 0); }

static hipError_t handle(void** h)
{
    *h = grab(16);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(void** s, unsigned f) { return (void)f, handle(s); }
hipError_t hipStreamDestroy(void* s) { return hipFree(s); }
hipError_t hipStreamWaitEvent(void* s, void* e, unsigned f) { return (void)s, (void)e, (void)f, hipSuccess; }
hipError_t hipStreamIsCapturing(void* s, int* status) { return (void)s, *status = 0, hipSuccess; }
hipError_t hipStreamBeginCapture(void* s, int mode) { return (void)mode, note(hipSuccess, "record on %llx", (uint64_t)(uintptr_t)s, 0, 0); }
hipError_t hipStreamEndCapture(void* s, void** g) { return (void)s, handle(g); }
hipError_t hipThreadExchangeStreamCaptureMode(int* mode) { return (void)mode, hipSuccess; }
hipError_t hipGraphInstantiate(void** x, void* g, void** n, char* l, size_t z) { return (void)g, (void)n, (void)l, (void)z, handle(x); }
hipError_t hipGraphLaunch(void* x, void* s) { return (void)x, (void)s, hipSuccess; }
hipError_t hipGraphDestroy(void* g) { return hipFree(g); }
hipError_t hipGraphExecDestroy(void* x) { return hipFree(x); }
hipError_t hipEventCreate(void** e) { return handle(e); }
hipError_t hipEventCreateWithFlags(void** e, unsigned f) { return (void)f, handle(e); }
hipError_t hipEventDestroy(void* e) { return hipFree(e); }
hipError_t hipEventRecord(void* e, void* s) { return (void)e, (void)s, hipSuccess; }
hipError_t hipEventSynchronize(void* e) { return (void)e, hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, void* a, void* b) { return (void)a, (void)b, *ms = 1.0f, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int d) { return (void)d, hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void* sym)
{
    static char page[4096];
    (void)sym;
    *p = page;
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t e) { return e ? "fake error" : "no error"; }
hipError_t hipGetLastError(void)
{
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}

static __thread struct {
    dim3 g, b;
    size_t lds;
    void* st;
} call;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, void* st)
{
    call.g = g;
    call.b = b;
    call.lds = lds;
    call.st = st;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, void** st)
{
    *g = call.g;
    *b = call.b;
    *lds = call.lds;
    *st = call.st;
    return hipSuccess;
}
void** __hipRegisterFatBinary(const void* data)
{
    static void* h;
    (void)data;
    return &h;
}
void __hipUnregisterFatBinary(void** h) { (void)h; }
void __hipRegisterFunction(void** m, const void* f, char* d, const char* n, unsigned t, void* a, void* b, void* c, void* e, int* w)
{
    (void)m, (void)f, (void)d, (void)n, (void)t, (void)a, (void)b, (void)c, (void)e, (void)w;
}
void __hipRegisterVar(void** m, void* v, char* h, char* d, int e, size_t z, int c, int g)
{
    (void)m, (void)v, (void)h, (void)d, (void)e, (void)z, (void)c, (void)g;
}
