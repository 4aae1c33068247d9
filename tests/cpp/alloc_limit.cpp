// A limit on the device memory that the library holds, for tests: loaded
// before it with RTLD_GLOBAL, these two functions take the place of the
// runtime's for its stream-ordered allocations and frees.  No allocation
// that exceeds the limit reaches the runtime; it fails as one for which the
// device has no room.

#include <dlfcn.h>

#include <cstddef>
#include <map>
#include <mutex>

namespace {

std::mutex mu;
std::map<void*, size_t> held;
size_t total = 0, limit = ~size_t{0}, refused = 0;

template <typename F>
F real(const char* name) {
    void* lib = dlopen("libamdhip64.so.7", RTLD_NOW);
    return lib ? reinterpret_cast<F>(dlsym(lib, name)) : nullptr;
}

}  // namespace

extern "C" {

void alloc_limit(size_t bytes) { limit = bytes; }
size_t alloc_held() { return total; }
size_t alloc_refused() { return refused; }

int hipMallocFromPoolAsync(void** p, size_t bytes, void* pool, void* stream) {
    static const auto fn = real<int (*)(void**, size_t, void*, void*)>("hipMallocFromPoolAsync");
    {
        std::lock_guard<std::mutex> lock(mu);
        if (bytes > limit || total > limit - bytes) {
            ++refused;
            return 2;  // hipErrorOutOfMemory
        }
    }
    const int e = fn(p, bytes, pool, stream);
    std::lock_guard<std::mutex> lock(mu);
    if (e == 0) {
        held[*p] = bytes;
        total += bytes;
    }
    return e;
}

int hipFreeAsync(void* p, void* stream) {
    static const auto fn = real<int (*)(void*, void*)>("hipFreeAsync");
    {
        std::lock_guard<std::mutex> lock(mu);
        const auto it = held.find(p);
        if (it != held.end()) {
            total -= it->second;
            held.erase(it);
        }
    }
    return fn(p, stream);
}
}
