/* The part of the HIP host API that libdocc_rt_rocm.so calls, without a device: every call succeeds, and what matters to the tests (allocations,
 * events, waits, launches) is written down in order. Loaded with RTLD_GLOBAL before the library, it is found first. Device addresses are numbers. */
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

static char text[1 << 20];
static size_t used;
static void note(const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    if (used + 512 < sizeof(text)) used += (size_t) vsnprintf(text + used, sizeof(text) - used, fmt, ap);
    va_end(ap);
}

/* what the tests set: the stream another library is capturing, and the size from which on there is no memory */
static hipStream_t captured;
static size_t no_memory_from = (size_t) -1;
static int device_queries;
static hipError_t last;
void recorder_capture(void* stream) { captured = (hipStream_t) stream; }
void recorder_no_memory_from(size_t bytes) { no_memory_from = bytes; }
/* the copy from now on that fails, as a HIP call does whose arguments are not valid; -1: none */
static int failing_copy = -1;
void recorder_fail_copy(int nth) { failing_copy = nth; }
int recorder_device_queries(void) { int n = device_queries; device_queries = 0; return n; }
const char* recorder_take(void) {
    static char taken[1 << 20];
    memcpy(taken, text, used);
    taken[used] = 0;
    used = 0;
    return taken;
}

hipError_t hipGetDevice(int* d) { device_queries++; *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int d) { (void) d; return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int d) {
    (void) d;
    memset(p, 0, sizeof(*p));
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetLastError(void) { hipError_t e = last; last = hipSuccess; return e; }
hipError_t hipGetSymbolAddress(void** p, const void* s) { (void) s; *p = (void*) 0x1000; return hipSuccess; }
hipError_t hipModuleLoad(hipModule_t* m, const char* path) { (void) path; *m = (hipModule_t) 0x2000; return hipSuccess; }
hipError_t hipModuleUnload(hipModule_t m) { (void) m; return hipSuccess; }
hipError_t hipModuleGetFunction(hipFunction_t* f, hipModule_t m, const char* name) {
    (void) m;
    *f = (hipFunction_t) strdup(name);
    return hipSuccess;
}
hipError_t hipModuleLaunchKernel(hipFunction_t f, unsigned gx, unsigned gy, unsigned gz, unsigned bx, unsigned by, unsigned bz, unsigned lds, hipStream_t s,
                                 void** args, void** extra) {
    (void) by, (void) bz, (void) args, (void) extra;
    note("launch %s %u,%u,%u x %u lds %u on %p\n", (const char*) f, gx, gy, gz, bx, lds, (void*) s);
    return (unsigned long long) gx * bx >> 32 ? hipErrorInvalidConfiguration : hipSuccess;
}
hipError_t hipMalloc(void** p, size_t bytes) {
    static size_t next = 0x100000000;
    if (bytes >= no_memory_from) {
        note("malloc %zu refused\n", bytes);
        return last = hipErrorOutOfMemory;
    }
    *p = (void*) next;
    next += (bytes + 4095) / 4096 * 4096;
    note("malloc %zu\n", bytes);
    return hipSuccess;
}
hipError_t hipFree(void* p) { note("free %p\n", p); return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { note("device sync\n"); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned flags) {
    static size_t next = 0x10;
    (void) flags;
    *s = (hipStream_t) (next += 0x10);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { (void) s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { (void) s; return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* status) {
    *status = captured && s == captured ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned flags) {
    static size_t next;
    (void) flags;
    *e = (hipEvent_t) ++next;
    note("event %zu\n", next);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { (void) e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { note("record %zu on %p\n", (size_t) e, (void*) s); return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { note("host waits for %zu\n", (size_t) e); return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned flags) {
    (void) flags;
    note("%p waits for %zu\n", (void*) s, (size_t) e);
    return hipSuccess;
}
/* host memory is the process's own; a pointer nobody has pinned makes the query of its kind fail */
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned flags) {
    (void) flags;
    *p = malloc(bytes);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) { (void) a, (void) p; return last = hipErrorInvalidValue; }
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind kind, hipStream_t s) {
    (void) dst, (void) src;
    const int fails = failing_copy == 0;
    if (failing_copy >= 0) failing_copy--;
    note("copy %zu %s on %p%s\n", bytes, kind == hipMemcpyHostToDevice ? "up" : kind == hipMemcpyDeviceToHost ? "down" : "across", (void*) s, fails ? " failed" : "");
    return fails ? (last = hipErrorInvalidValue) : hipSuccess;
}
