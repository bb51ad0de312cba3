// Refuses chosen device allocations, for tests of what counts do without them:
// loaded with RTLD_GLOBAL before libgat.so, its hipMalloc is the one that is
// called, and hands on what it does not refuse.
#include <hip/hip_runtime_api.h>

#include <dlfcn.h>

static size_t refuse_from[8], refuse_to[8];
static int ranges = 0, refused = 0;

extern "C" {
// Sizes in [from_bytes, to_bytes) are refused too.
void limit_refuse(size_t from_bytes, size_t to_bytes) {
    if (ranges == 8) return;
    refuse_from[ranges] = from_bytes;
    refuse_to[ranges++] = to_bytes;
}
int limit_refused() { return refused; }
hipError_t hipMalloc(void **p, size_t bytes) {
    using Fn = hipError_t (*)(void **, size_t);
    static const Fn real = [] {
        void *lib = dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_LOCAL);
        return lib ? reinterpret_cast<Fn>(dlsym(lib, "hipMalloc")) : nullptr;
    }();
    for (int i = 0; i < ranges; i++)
        if (bytes >= refuse_from[i] && bytes < refuse_to[i]) {
            refused++;
            *p = nullptr;
            return hipErrorOutOfMemory;
        }
    return real ? real(p, bytes) : hipErrorNotInitialized;
}
}
