// Stands in front of a few HIP runtime calls so that a test can have one of
// them refused: loaded into the global scope before the library under test,
// which then binds to these.  Nothing reaches the GPU for a refused call.  Like
// the runtime's own refusals of memory, a refused allocation leaves its error to
// be read by hipGetLastError (the real call is made with a null pointer).
#include <dlfcn.h>
#include <stddef.h>

namespace {

struct Fault {
    size_t at_least = 0;  // bytes
    long skip = 0;        // calls let through first
    long times = 0;       // refusals left
    long calls = 0;       // calls of at least that size
};
Fault g_fault[3];  // hipHostMalloc, hipMallocAsync, hipEventRecord

void *real(const char *name) {
    void *h = dlopen("libamdhip64.so.7", RTLD_NOW);
    return h ? dlsym(h, name) : nullptr;
}

bool refused(int which, size_t bytes) {
    Fault &f = g_fault[which];
    if (bytes < f.at_least) return false;
    f.calls++;
    if (f.skip > 0) {
        f.skip--;
        return false;
    }
    if (f.times <= 0) return false;
    f.times--;
    return true;
}

constexpr int kOutOfMemory = 2, kInvalidHandle = 400;

}  // namespace

extern "C" {

void hip_fail_set(int which, size_t at_least, long skip, long times) {
    g_fault[which] = Fault{at_least, skip, times, 0};
}

long hip_fail_calls(int which) { return g_fault[which].calls; }

int hipHostMalloc(void **p, size_t bytes, unsigned flags) {
    static const auto f = (int (*)(void **, size_t, unsigned))real("hipHostMalloc");
    if (!refused(0, bytes)) return f(p, bytes, flags);
    (void)f(nullptr, bytes, flags);
    return kOutOfMemory;
}

int hipMallocAsync(void **p, size_t bytes, void *stream) {
    static const auto f = (int (*)(void **, size_t, void *))real("hipMallocAsync");
    if (!refused(1, bytes)) return f(p, bytes, stream);
    (void)f(nullptr, bytes, stream);
    return kOutOfMemory;
}

int hipEventRecord(void *event, void *stream) {
    static const auto f = (int (*)(void *, void *))real("hipEventRecord");
    return refused(2, 0) ? kInvalidHandle : f(event, stream);
}

}  // extern "C"
