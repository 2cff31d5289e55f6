/* hipHostMalloc as a system that has run out of pinned memory answers it:
 * blocks over 256 KB are refused, with the runtime's last error left set. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>

extern int hipSetDevice(int);

int hipHostMalloc(void **p, size_t bytes, unsigned flags) {
    static int (*real)(void **, size_t, unsigned);
    if (bytes > 262144) {
        *p = NULL;
        hipSetDevice(1 << 20); /* no such device: only the error stays */
        return 2;              /* hipErrorOutOfMemory */
    }
    if (!real) real = (int (*)(void **, size_t, unsigned))dlsym(RTLD_NEXT, "hipHostMalloc");
    return real(p, bytes, flags);
}
