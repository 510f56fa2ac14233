// Stands in front of hipHostMalloc and operator new in a test's process: refuses
// pinned memory, or host blocks from a size on, while the test asks for it.
#include <dlfcn.h>

#include <cstddef>
#include <cstdlib>
#include <new>

static bool refuse_pinned = false;
static size_t refuse_from = 0;

extern "C" {
void refuse_pinned_memory(int on) { refuse_pinned = on != 0; }
void refuse_host_blocks(size_t from) { refuse_from = from; }

int hipHostMalloc(void** p, size_t n, unsigned flags) {
    if (refuse_pinned) return 2;  // hipErrorOutOfMemory
    using Fn = int (*)(void**, size_t, unsigned);
    static Fn next = nullptr;
    if (!next) {
        void* hip = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
        if (hip) next = (Fn)dlsym(hip, "hipHostMalloc");
    }
    return next ? next(p, n, flags) : 2;
}
}

void* operator new(size_t n) {
    if (refuse_from && n >= refuse_from) throw std::bad_alloc();
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
