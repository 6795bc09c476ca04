// The parts of the HIP runtime that the library's host code calls, on host memory, for tests
// of that code without a GPU: kernels do nothing, and the n-th allocation can be made to fail.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <set>

namespace {
std::set<void *> g_live;
long g_calls = 0, g_fail = 0;
double g_fill = 0.0;
int allocate(void **p, size_t n) {
    *p = nullptr;
    if (++g_calls == g_fail) return 2;  // hipErrorOutOfMemory
    *p = std::malloc(n ? n : 1);
    for (size_t i = 0; i + 8 <= n; i += 8) std::memcpy((char *)*p + i, &g_fill, 8);
    g_live.insert(*p);
    return 0;
}
int release(void *p) {
    if (p && g_live.erase(p) == 0) std::abort();  // not an allocation, or freed twice
    std::free(p);
    return 0;
}
}  // namespace

// the n-th allocation from now on fails (0: none)
void fail_allocation(long n) {
    g_calls = 0;
    g_fail = n;
}
// what new memory holds, as doubles: what is read back from kernels that did nothing
void fill_memory(double v) { g_fill = v; }
long allocations() { return g_calls; }
long live_allocations() { return (long)g_live.size(); }

extern "C" {
int hipMalloc(void **p, size_t n) { return allocate(p, n); }
int hipHostMalloc(void **p, size_t n, unsigned) { return allocate(p, n); }
int hipFree(void *p) { return release(p); }
int hipHostFree(void *p) { return release(p); }
int hipMemcpy(void *d, const void *s, size_t n, int) {
    std::memmove(d, s, n);
    return 0;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int, void *) {
    std::memmove(d, s, n);
    return 0;
}
int hipMemset(void *d, int v, size_t n) {
    std::memset(d, v, n);
    return 0;
}
int hipMemsetAsync(void *d, int v, size_t n, void *) {
    std::memset(d, v, n);
    return 0;
}
int hipGetDevice(int *d) { return *d = 0; }
int hipSetDevice(int) { return 0; }
int hipGetDeviceCount(int *n) {
    *n = 1;
    return 0;
}
int hipDeviceGetAttribute(int *v, int, int) {
    *v = 256;
    return 0;
}
int hipDeviceSynchronize() { return 0; }
int hipStreamSynchronize(void *) { return 0; }
int hipStreamCreateWithFlags(void **s, unsigned) {
    *s = nullptr;
    return 0;
}
int hipStreamDestroy(void *) { return 0; }
int hipEventCreate(void **e) {
    *e = nullptr;
    return 0;
}
int hipEventCreateWithFlags(void **e, unsigned) {
    *e = nullptr;
    return 0;
}
int hipEventDestroy(void *) { return 0; }
int hipGetLastError() { return 0; }
const char *hipGetErrorString(int) { return "error"; }
int hipLaunchKernel(const void *, ...) { return 0; }
int __hipPushCallConfiguration(...) { return 0; }
int __hipPopCallConfiguration(...) { return 0; }
void **__hipRegisterFatBinary(const void *) { return nullptr; }
void __hipRegisterFunction(...) {}
void __hipRegisterVar(...) {}
void __hipUnregisterFatBinary(void **) {}
}
