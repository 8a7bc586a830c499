// Device allocations above a limit fail as on a full device: loaded before the
// library, this definition of hipMalloc is the one its calls reach.
#include <cstddef>

extern "C" {
static int (*real)(void**, size_t);
static size_t most = ~(size_t)0;
static unsigned refused;

void malloc_limit(int (*hip_malloc)(void**, size_t), size_t bytes) {
    real = hip_malloc;
    most = bytes;
}
unsigned malloc_refused() { return refused; }

int hipMalloc(void** p, size_t bytes) {
    if (bytes <= most) return real(p, bytes);
    refused++;
    *p = nullptr;
    return 2;  // hipErrorOutOfMemory
}
}
