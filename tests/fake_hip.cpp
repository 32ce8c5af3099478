// A HIP runtime without a device, for tests of the library's host code: device
// memory is host memory, copies are copies, kernels do nothing.  Loaded with
// RTLD_GLOBAL before libnetflux.so, its functions are the ones that are called.
// fake_fail_above(n): device allocations of more than n bytes fail from now on;
// fake_capacity(n): those that would take the total above n bytes;
// fake_fail_host(1): pinned ones.
#include <atomic>
#include <cstddef>
#include <cstdlib>
#include <cstring>

typedef int err_t;
static constexpr err_t OOM = 2;
static constexpr size_t HEAD = 256;  // the size of an allocation, in front of it
static std::atomic<size_t> fail_above{~(size_t)0}, capacity{~(size_t)0}, allocated{0}, live{0};
static std::atomic<int> fail_host{0}, last{0}, allocations{0}, waits{0};

extern "C" {
void fake_fail_above(size_t n) { fail_above = n; }
void fake_capacity(size_t n) { capacity = n; }
void fake_fail_host(int on) { fail_host = on; }
size_t fake_allocated() { return allocated; }  // bytes of all successful device allocations so far
int fake_allocations() { return allocations; }
int fake_waits() { return waits; }             // blocking copies and waits for a stream
size_t fake_live() { return live; }            // bytes of those not freed

err_t hipGetDeviceCount(int *n) { return *n = 1, 0; }
err_t hipGetDevice(int *d) { return *d = 0, 0; }
err_t hipSetDevice(int) { return 0; }
const char *hipGetErrorString(err_t) { return "out of memory"; }
err_t hipGetLastError() { return last.exchange(0); }
err_t hipMalloc(void **p, size_t n) {
    if (n > fail_above || live + n > capacity) return last = OOM;
    char *q = static_cast<char *>(std::calloc(n + HEAD, 1));
    if (!q) return last = OOM;
    std::memcpy(q, &n, sizeof n);
    ++allocations;
    allocated += n;
    live += n;
    *p = q + HEAD;
    return 0;
}
err_t hipFree(void *p) {
    if (!p) return 0;
    char *q = static_cast<char *>(p) - HEAD;
    size_t n;
    std::memcpy(&n, q, sizeof n);
    live -= n;
    return std::free(q), 0;
}
err_t hipHostMalloc(void **p, size_t n, unsigned) {
    if (fail_host) return last = OOM;
    *p = std::calloc(n, 1);
    return *p ? 0 : OOM;
}
err_t hipHostFree(void *p) { return std::free(p), 0; }
err_t hipMemcpy(void *d, const void *s, size_t n, int) { return ++waits, std::memmove(d, s, n), 0; }
err_t hipMemcpyAsync(void *d, const void *s, size_t n, int, void *) { return std::memmove(d, s, n), 0; }
err_t hipMemcpy2DAsync(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, int, void *) {
    for (size_t q = 0; q < h; ++q) std::memmove((char *)d + q * dp, (const char *)s + q * sp, w);
    return 0;
}
err_t hipMemset(void *d, int v, size_t n) { return std::memset(d, v, n), 0; }
err_t hipMemsetAsync(void *d, int v, size_t n, void *) { return std::memset(d, v, n), 0; }
static char handle;
err_t hipStreamCreateWithFlags(void **s, unsigned) { return *s = &handle, 0; }
err_t hipStreamDestroy(void *) { return 0; }
err_t hipStreamSynchronize(void *) { return ++waits, 0; }
err_t hipEventCreate(void **e) { return *e = &handle, 0; }
err_t hipEventCreateWithFlags(void **e, unsigned) { return *e = &handle, 0; }
err_t hipEventDestroy(void *) { return 0; }
err_t hipEventRecord(void *, void *) { return 0; }
err_t hipEventSynchronize(void *) { return 0; }
err_t hipEventElapsedTime(float *ms, void *, void *) { return *ms = 1.0f, 0; }
err_t hipLaunchKernel(const void *, ...) { return 0; }
void **__hipRegisterFatBinary(const void *) {
    static void *h;
    return &h;
}
void __hipRegisterFunction(...) {}
void __hipUnregisterFatBinary(void **) {}
err_t __hipPushCallConfiguration(...) { return 0; }
err_t __hipPopCallConfiguration(...) { return 0; }
}
