/* Stands between one copy of libeio_hip.so and the HIP runtime (tests/test_resident_fallback_gpu.py loads it
 * first, with RTLD_GLOBAL): a cooperative launch or an allocation is refused on the host, as a device that
 * another process holds or that is full would refuse it.  Nothing of a refused call reaches the device; every
 * other call passes through. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>

typedef struct { unsigned x, y, z; } dim3_t;

static int launch_code, launch_left, launch_after;   /* after `after` more launches, `left` of them return `code` */
static size_t malloc_limit = ~(size_t)0;             /* larger allocations: hipErrorOutOfMemory */
static size_t free_shown;                            /* free memory to report (0: the device's) */

void shim_launches(int code, int count, int after) {
    launch_code = code;
    launch_left = count;
    launch_after = after;
}
void shim_memory(size_t limit, size_t shown) {
    malloc_limit = limit;
    free_shown = shown;
}

int hipLaunchCooperativeKernel(const void* f, dim3_t g, dim3_t b, void** args, unsigned lds, void* stream) {
    static int (*real)(const void*, dim3_t, dim3_t, void**, unsigned, void*);
    if (!real) *(void**)&real = dlsym(RTLD_NEXT, "hipLaunchCooperativeKernel");
    if (launch_left > 0 && launch_after-- <= 0) {
        --launch_left;
        return launch_code;
    }
    return real(f, g, b, args, lds, stream);
}

int hipMalloc(void** p, size_t n) {
    static int (*real)(void**, size_t);
    if (!real) *(void**)&real = dlsym(RTLD_NEXT, "hipMalloc");
    return n > malloc_limit ? 2 : real(p, n);
}

int hipMemGetInfo(size_t* avail, size_t* total) {
    static int (*real)(size_t*, size_t*);
    if (!real) *(void**)&real = dlsym(RTLD_NEXT, "hipMemGetInfo");
    const int e = real(avail, total);
    if (!e && free_shown) *avail = free_shown;
    return e;
}
