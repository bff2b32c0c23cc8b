// hipMemcpyAsync that counts the bytes of host-to-device copies: loaded
// (RTLD_GLOBAL) before the product library, whose calls then come here.
#include <dlfcn.h>

#include <cstddef>

extern "C" {
size_t uploaded = 0;

int hipMemcpyAsync(void *dst, const void *src, size_t bytes, int kind, void *stream) {
    using Fn = int (*)(void *, const void *, size_t, int, void *);
    static Fn real = (Fn)dlsym(dlopen("libamdhip64.so", RTLD_NOW | RTLD_NOLOAD), "hipMemcpyAsync");
    if (kind == 1) uploaded += bytes;  // hipMemcpyHostToDevice
    return real(dst, src, bytes, kind, stream);
}
}
