// The copies between pageable memory and the device (transfer.hip) on a runtime of its own, whose copies happen at once, whose
// caller's stream stays busy until somebody waits for it on the host, and which may have no thread left to give.
#include <dlfcn.h>
#include <errno.h>
#include <pthread.h>

#include <cstdio>
#include <cstdlib>

#include "../../thundergbm_amd/csrc/transfer.hip"

namespace {
std::atomic<bool> busy{false};                // the caller's stream has a kernel to run
std::atomic<int> held_up{0}, too_early{0};    // waits for it on a shared stream, copies of its results that do not wait for it
std::atomic<int> caller_waits{0};             // of the caller's stream for a copy stream
std::atomic<bool> no_threads{false};
std::atomic<size_t> handles{0};
hipStream_t const kCaller = reinterpret_cast<hipStream_t>((size_t)1 << 40), kOther = reinterpret_cast<hipStream_t>((size_t)2 << 40);
std::atomic<bool> other_waits{false};  // the caller's second stream, for the first one
hipEvent_t of_caller;
void copy(void *dst, const void *src, size_t bytes) { std::memcpy(dst, src, bytes); }
}  // namespace

extern "C" {
int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *arg) {
    static auto real = reinterpret_cast<int (*)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *)>(dlsym(RTLD_NEXT, "pthread_create"));
    return no_threads ? EAGAIN : real(t, a, f, arg);
}
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return ""; }
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) { return *p = std::malloc(bytes), hipSuccess; }
hipError_t hipHostFree(void *p) { return std::free(p), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return *e = reinterpret_cast<hipEvent_t>(++handles), hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    if (s == kCaller) of_caller = e;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    if (e == of_caller) busy = false;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return *s = reinterpret_cast<hipStream_t>(++handles), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
    if (s == kCaller) busy = false;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    if (s == kCaller) ++caller_waits;
    if (s == kOther) other_waits = other_waits || e == of_caller;
    else if (s != kCaller && e == of_caller && busy) ++held_up;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes, hipMemcpyKind kind, hipStream_t s) {
    if (kind == hipMemcpyDeviceToHost && busy && s != kCaller && !(s == kOther && other_waits)) ++too_early;
    return copy(dst, src, bytes), hipSuccess;
}
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }
void **__hipRegisterFatBinary(const void *) { return nullptr; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *, int *) {}
}
namespace tgbm {
void fatal(const char *fmt, ...) { std::puts(fmt), std::_Exit(1); }
void *device_alloc(size_t bytes) { return std::malloc(bytes); }
void device_free(void *p) { std::free(p); }
}  // namespace tgbm

#define CHECK(c) \
    if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); return 1; }

int main(int argc, char **argv) {
    using namespace tgbm;
    no_threads = argc > 1;
    std::vector<char> from((size_t)40 << 20), to(from.size());
    for (size_t i = 0; i < from.size(); ++i) from[i] = (char)(i * 2654435761u >> 13);
    for (size_t bytes : {from.size(), from.size() - 77, ((size_t)1 << 20) + 1, (size_t)100}) {
        std::fill(to.begin(), to.end(), 0);
        busy = true;
        other_waits = false;
        download_large(kCaller, kOther, to.data(), from.data(), bytes);
        CHECK(std::memcmp(to.data(), from.data(), bytes) == 0 && (bytes == to.size() || to[bytes] == 0));
        CHECK(held_up == 0);
        CHECK(too_early == 0);
        busy = false;
        std::fill(to.begin(), to.end(), 0);
        upload_large(kCaller, to.data(), from.data(), bytes);
        CHECK(std::memcmp(to.data(), from.data(), bytes) == 0);
    }
    size_t arrived = 0;
    UploadSet set;
    for (size_t j = 0; j < 8; ++j) set.add(to.data() + j * ((size_t)5 << 20), from.data() + j * ((size_t)5 << 20), (size_t)5 << 20);
    set.send_in_order(kCaller, [&](size_t j) { arrived += j == arrived; });
    CHECK(arrived == 8 && to == from && caller_waits <= 2 * 8 + 2 * 3);  // (3: upload_large above, where it is staged)
    // a small array: the caller's stream waits for the two copy streams once, whoever else does
    const std::vector<double> x(1000, 0.5);
    std::vector<float> f(x.size());
    UploadSet one;
    one.add_doubles(f.data(), x.data(), x.size());
    caller_waits = 0;
    one.send_in_order(kCaller, [&](size_t) { arrived += caller_waits == 2; });
    CHECK(arrived == 9 && caller_waits == 2 && f.back() == 0.5f);
    // arrays that hipMemcpy takes as fast as the pieces do go without them
    UploadSet few;
    for (size_t j = 0; j < 2; ++j) few.add(to.data() + j * ((size_t)7 << 20), from.data(), (size_t)7 << 20);
    caller_waits = 0;
    few.send_in_order(kCaller, [&](size_t) { ++arrived; });
    CHECK(arrived == 11 && caller_waits == 0 && std::memcmp(to.data() + ((size_t)7 << 20), from.data(), (size_t)7 << 20) == 0);
    std::printf("ok\n");
    return 0;
}
