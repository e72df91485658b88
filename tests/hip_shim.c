/* Stands between one copy of libeio_hip.so and the HIP runtime (tests/test_resident_fallback_gpu.py loads it
 * first, with RTLD_GLOBAL): a cooperative launch or an allocation is refused on the host, as a device that
 * another process holds or that is full would refuse it.  Nothing of a refused call reaches the device; every
 * other call passes through. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>

typedef struct { unsigned x, y, z; } dim3_t;

static int launch_code, launch_left, launch_after;   /* after `after` more launches, `left` of them return `code` */
static size_t capacity = ~(size_t)0, live;           /* the device's memory, and what is allocated of it here */

void shim_launches(int code, int count, int after) {
    launch_code = code;
    launch_left = count;
    launch_after = after;
}
void shim_capacity(size_t bytes) { capacity = bytes; }
size_t shim_live(void) { return live; }

int hipLaunchCooperativeKernel(const void* f, dim3_t g, dim3_t b, void** args, unsigned lds, void* stream) {
    static int (*real)(const void*, dim3_t, dim3_t, void**, unsigned, void*);
    if (!real) *(void**)&real = dlsym(RTLD_NEXT, "hipLaunchCooperativeKernel");
    if (launch_left > 0 && launch_after-- <= 0) {
        --launch_left;
        return launch_code;
    }
    return real(f, g, b, args, lds, stream);
}

static struct { void* p; size_t n; } table[4096];

int hipMalloc(void** p, size_t n) {
    static int (*real)(void**, size_t);
    if (!real) *(void**)&real = dlsym(RTLD_NEXT, "hipMalloc");
    if (n > capacity || live > capacity - n) return 2; /* hipErrorOutOfMemory */
    const int e = real(p, n);
    for (int i = 0; !e && i < 4096; ++i)
        if (!table[i].p) {
            table[i].p = *p;
            table[i].n = n;
            live += n;
            break;
        }
    return e;
}

int hipFree(void* p) {
    static int (*real)(void*);
    if (!real) *(void**)&real = dlsym(RTLD_NEXT, "hipFree");
    for (int i = 0; p && i < 4096; ++i)
        if (table[i].p == p) {
            live -= table[i].n;
            table[i].p = NULL;
            break;
        }
    return real(p);
}

int hipMemGetInfo(size_t* avail, size_t* total) {
    static int (*real)(size_t*, size_t*);
    if (!real) *(void**)&real = dlsym(RTLD_NEXT, "hipMemGetInfo");
    const int e = real(avail, total);
    const size_t left = capacity > live ? capacity - live : 0;
    if (!e && left < *avail) *avail = left;
    return e;
}
