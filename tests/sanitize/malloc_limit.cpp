// hipMalloc that refuses allocations above limit_bytes, as a full GPU would:
// loaded (RTLD_GLOBAL) before the product library, whose calls then come here.
#include <dlfcn.h>

#include <cstddef>

extern "C" {
size_t limit_bytes = ~(size_t)0;
int refused = 0;

int hipMalloc(void **p, size_t bytes) {
    using Fn = int (*)(void **, size_t);
    static Fn real = (Fn)dlsym(dlopen("libamdhip64.so", RTLD_NOW | RTLD_NOLOAD), "hipMalloc");
    if (bytes > limit_bytes) {
        refused++;
        return 2;  // hipErrorOutOfMemory
    }
    return real(p, bytes);
}
}
