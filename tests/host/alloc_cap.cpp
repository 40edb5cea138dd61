// A cap on single device allocations, for tests: loaded with RTLD_GLOBAL
// before the engine, its hipMalloc stands in front of the runtime's.  A
// request above the cap is passed on as one that no card can meet, so the
// caller sees the runtime's own failure, with the error state it leaves.
#include <dlfcn.h>
#include <stddef.h>

static size_t g_cap = ~size_t(0);

extern "C" void alloc_cap_set(size_t bytes) { g_cap = bytes; }

extern "C" int hipMalloc(void** p, size_t bytes) {
    using Fn = int (*)(void**, size_t);
    static const Fn real = [] {
        void* lib = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
        return lib ? reinterpret_cast<Fn>(dlsym(lib, "hipMalloc")) : nullptr;
    }();
    if (!real) return 2;   // hipErrorOutOfMemory
    return real(p, bytes > g_cap ? size_t(1) << 60 : bytes);
}
