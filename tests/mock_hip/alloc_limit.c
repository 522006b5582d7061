/* hipMalloc and hipFree that refuse what is asked for here, loaded (RTLD_GLOBAL) before the library under test:
 * an allocation beyond a number of bytes, or one of an exact size, fails as if the device were full. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <pthread.h>
#include <stddef.h>

enum { kOutOfMemory = 2, kMost = 4096 };
static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
static struct { void *p; size_t n; } held[kMost];
static int nheld, failures;
static size_t used, most = (size_t)-1, exact;

static void *real(const char *name) {
    void *lib = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
    return lib ? dlsym(lib, name) : NULL;
}

int hipMalloc(void **p, size_t n) {
    int (*f)(void **, size_t) = (int (*)(void **, size_t))real("hipMalloc");
    if (!f) return 1;
    pthread_mutex_lock(&mu);
    int rc = kOutOfMemory;
    if (used + n <= most && n != exact && nheld < kMost) {
        rc = f(p, n);
        if (rc == 0) {
            held[nheld].p = *p;
            held[nheld++].n = n;
            used += n;
        }
    } else {
        failures++;
    }
    pthread_mutex_unlock(&mu);
    return rc;
}

int hipFree(void *p) {
    int (*f)(void *) = (int (*)(void *))real("hipFree");
    if (!f) return 1;
    pthread_mutex_lock(&mu);
    for (int i = 0; i < nheld; i++)
        if (held[i].p == p) {
            used -= held[i].n;
            held[i] = held[--nheld];
            break;
        }
    pthread_mutex_unlock(&mu);
    return f(p);
}

/* room: bytes that may still be allocated; size: allocations of this size fail (0: none) */
void limit_room(size_t room) { most = room == (size_t)-1 ? room : used + room; }
void limit_size(size_t size) { exact = size; }
int limit_failures(void) { return failures; }
