/* A HIP runtime in host memory, for tests of the library's host side without a
 * device: preloaded, it takes the place of the runtime's functions that
 * libswmgpu.so calls.  Device memory is calloc'ed, copies and fills happen at
 * once, kernels do nothing, streams and events only count.  Two conditions can
 * be set from outside:
 *   host_hip_fail_event(n): the n-th hipEventSynchronize from now on fails
 *   host_hip_thread_delay_ms: threads made from now on begin that much later
 * and host_hip_copies_open() is the number of asynchronous copies enqueued
 * since their stream (there is one) was last waited for. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <pthread.h>
#include <stdlib.h>
#include <string.h>
#include <time.h>

typedef int err;
static int fail_at = 0, open_copies = 0;
int host_hip_thread_delay_ms = 0;
void host_hip_fail_event(int n) { fail_at = n; }
int host_hip_copies_open(void) { return open_copies; }

struct late {
    void* (*run)(void*);
    void* arg;
    int ms;
};
static void* late_start(void* p) {
    struct late l = *(struct late*)p;
    struct timespec t = {l.ms / 1000, (l.ms % 1000) * 1000000L};
    free(p);
    nanosleep(&t, NULL);
    return l.run(l.arg);
}
int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*run)(void*), void* arg) {
    static int (*real)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
    if (!real) *(void**)&real = dlsym(RTLD_NEXT, "pthread_create");
    if (!host_hip_thread_delay_ms) return real(t, a, run, arg);
    struct late* l = malloc(sizeof *l);
    l->run = run;
    l->arg = arg;
    l->ms = host_hip_thread_delay_ms;
    return real(t, a, late_start, l);
}

err hipGetDeviceCount(int* n) { *n = 1; return 0; }
err hipGetDevice(int* d) { *d = 0; return 0; }
err hipDeviceGetAttribute(int* v, int attr, int dev) { (void)attr; (void)dev; *v = 256; return 0; }
err hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void* f, int b, size_t s) {
    (void)f; (void)b; (void)s;
    *n = 4;
    return 0;
}
const char* hipGetErrorString(err e) { return e ? "injected" : "success"; }
err hipGetLastError(void) { return 0; }
err hipMalloc(void** p, size_t n) { *p = calloc(n ? n : 1, 1); return *p ? 0 : 2; }
err hipFree(void* p) { free(p); return 0; }
err hipHostMalloc(void** p, size_t n, unsigned f) { (void)f; return hipMalloc(p, n); }
err hipHostFree(void* p) { free(p); return 0; }
err hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void* stream) {
    (void)kind; (void)stream;
    memcpy(d, s, n);
    ++open_copies;
    return 0;
}
err hipMemsetAsync(void* d, int v, size_t n, void* stream) { (void)stream; memset(d, v, n); return 0; }
err hipStreamCreateWithFlags(void** s, unsigned f) { (void)f; *s = malloc(1); return 0; }
err hipStreamDestroy(void* s) { free(s); return 0; }
err hipStreamSynchronize(void* s) { (void)s; open_copies = 0; return 0; }
err hipEventCreate(void** e) { *e = malloc(1); return 0; }
err hipEventCreateWithFlags(void** e, unsigned f) { (void)f; return hipEventCreate(e); }
err hipEventDestroy(void* e) { free(e); return 0; }
err hipEventRecord(void* e, void* s) { (void)e; (void)s; return 0; }
err hipEventSynchronize(void* e) { (void)e; return fail_at && --fail_at == 0 ? 999 : 0; }
err hipEventElapsedTime(float* ms, void* a, void* b) { (void)a; (void)b; *ms = 1.0f; return 0; }
err hipLaunchKernel(const void* f, ...) { (void)f; return 0; }
err __hipPushCallConfiguration(void) { return 0; }
err __hipPopCallConfiguration(void) { return 0; }
