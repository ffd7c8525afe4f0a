/* hipMalloc in front of the runtime's: keeps the sizes asked for and refuses
 * one size on request, as a card without that much memory left would. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>

long long shim_refuse = -1;      /* size to refuse */
long long shim_refused = 0;      /* how often it was */
long long shim_sizes[4096];
long long shim_count = 0;

int hipMalloc(void **ptr, size_t size) {
    static int (*next)(void **, size_t) = NULL;
    if (!next) {
        void *lib = dlopen("libamdhip64.so.7", RTLD_NOLOAD | RTLD_NOW);
        if (lib) next = (int (*)(void **, size_t))dlsym(lib, "hipMalloc");
        if (!next) return 3;     /* not initialised */
    }
    if (shim_count < 4096) shim_sizes[shim_count++] = (long long)size;
    if ((long long)size == shim_refuse) {
        ++shim_refused;
        *ptr = NULL;
        return 2;                /* out of memory */
    }
    return next(ptr, size);
}
