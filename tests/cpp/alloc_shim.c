/* hipMalloc and hipFree in front of the HIP runtime's: counts the bytes that
 * are held and, once armed, lets the n-th allocation from there fail. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>

typedef int (*malloc_fn)(void**, size_t);
typedef int (*free_fn)(void*);

static struct {
    void* p;
    size_t n;
} held[4096];
static int countdown;

static void* real(const char* name) {
    static void* hip;
    if (!hip) hip = dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_LOCAL);
    return dlsym(hip, name);
}

void shim_fail(int nth) { countdown = nth; }

size_t shim_held(void) {
    size_t n = 0;
    for (int i = 0; i < 4096; ++i) n += held[i].n;
    return n;
}

int hipMalloc(void** p, size_t n) {
    if (countdown > 0 && --countdown == 0) return 2; /* hipErrorOutOfMemory */
    const int st = ((malloc_fn)real("hipMalloc"))(p, n);
    for (int i = 0; st == 0 && i < 4096; ++i)
        if (!held[i].p) {
            held[i].p = *p;
            held[i].n = n;
            break;
        }
    return st;
}

int hipFree(void* p) {
    for (int i = 0; p && i < 4096; ++i)
        if (held[i].p == p) {
            held[i].p = NULL;
            held[i].n = 0;
        }
    return ((free_fn)real("hipFree"))(p);
}
