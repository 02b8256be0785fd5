/* hipHostMalloc that has no memory for blocks of NO_PINNED_FROM (environment) bytes and more.
 * Loaded (RTLD_GLOBAL) before the library under test, whose calls then come here. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
#include <stdlib.h>

int no_pinned_refused;

int hipHostMalloc(void **p, size_t bytes, unsigned flags)
{
    static int (*real)(void **, size_t, unsigned);
    const char *from = getenv("NO_PINNED_FROM");
    if (from && bytes >= strtoull(from, NULL, 10)) {
        no_pinned_refused++;
        return 2; /* hipErrorOutOfMemory */
    }
    if (!real) {
        void *h = dlopen("libamdhip64.so", RTLD_LAZY | RTLD_NOLOAD);
        if (!h) h = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
        if (h) real = (int (*)(void **, size_t, unsigned))dlsym(h, "hipHostMalloc");
        if (!real) return 1; /* hipErrorInvalidValue */
    }
    return real(p, bytes, flags);
}
