// The kept device blocks (device_memory.hip) on a driver of its own: 16 GB of memory that counts what is asked of it.
#include <cstdio>
#include <future>
#include <map>
#include <mutex>
#include <set>
#include <thread>

#include "../../thundergbm_amd/csrc/device_memory.hip"

namespace {
constexpr size_t kMB = (size_t)1 << 20, kTotal = (size_t)16 << 30;
std::mutex m;
std::map<char *, size_t> blocks;
size_t used = 0;
int mallocs = 0, frees = 0, streams = 0;
char *next_address = reinterpret_cast<char *>(1 << 20);
bool probe_lock = false, lock_held = false;

void probe() {  // can another thread use the pool while the driver works for this one?
    if (!probe_lock) return;
    probe_lock = false;
    auto other = std::async(std::launch::async, [] { tgbm::device_mem_info(new size_t, new size_t); });
    lock_held = other.wait_for(std::chrono::seconds(2)) != std::future_status::ready;
    if (lock_held) {
        std::printf("the driver is called under the lock\n");
        std::_Exit(1);
    }
}
}  // namespace

extern "C" {
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return ""; }
hipError_t hipMemGetInfo(size_t *f, size_t *t) {
    std::lock_guard<std::mutex> lock(m);
    return *f = kTotal - used, *t = kTotal, hipSuccess;
}
hipError_t hipFree(void *p) {
    probe();
    std::lock_guard<std::mutex> lock(m);
    used -= blocks.at(static_cast<char *>(p));
    blocks.erase(static_cast<char *>(p));
    ++frees;
    return hipSuccess;
}
hipError_t hipStreamCreate(hipStream_t *s) { return *s = reinterpret_cast<hipStream_t>((size_t)++streams), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
}
hipError_t hipMalloc(void **p, size_t bytes) {
    probe();
    std::lock_guard<std::mutex> lock(m);
    if (used + bytes > kTotal) return hipErrorOutOfMemory;
    used += bytes;
    blocks[next_address] = bytes;
    *p = next_address;
    next_address += bytes;
    ++mallocs;
    return hipSuccess;
}
namespace tgbm {
void fatal(const char *fmt, ...) { std::puts(fmt), std::_Exit(1); }
void release_transfer_memory() {}
}  // namespace tgbm

#define CHECK(c) \
    if (!(c)) { std::printf("line %d: %s (mallocs %d, frees %d, used %zu MB)\n", __LINE__, #c, mallocs, frees, used / kMB); return 1; }

int main() {
    using namespace tgbm;
    const size_t limit = kTotal / 32;  // (of 16 GB)
    // the second call of a size takes the first one's block
    void *a = device_alloc(10 * kMB);
    device_free(a);
    CHECK(device_alloc(10 * kMB - 5) == a && mallocs == 1);
    device_free(a);
    // a training call leaves its blocks; requests that come after it free none of them
    std::vector<void *> training;
    for (int i = 0; i < 8; ++i) training.push_back(device_alloc(limit / 16));
    for (void *p : training) device_free(p);
    frees = mallocs = 0;
    for (int i = 0; i < 1000; ++i) {
        hipStream_t s = stream_acquire();
        void *p = device_alloc(5000);
        device_free(p);
        stream_release(s);
    }
    CHECK(frees == 0 && mallocs == 1 && streams == 1);
    // ... and the next one of its size finds them
    for (void *&p : training) p = device_alloc(limit / 16);
    CHECK(mallocs == 1);
    for (void *p : training) device_free(p);
    // no more than the limit stays, the longest unused blocks go, a block beyond the limit is not kept
    size_t free_b = 0, total_b = 0;
    std::vector<void *> other;
    for (int i = 0; i < 12; ++i) other.push_back(device_alloc(limit / 8 + (size_t)i * limit / 512));
    for (void *p : other) device_free(p);
    CHECK(used <= limit);
    CHECK(blocks.count(static_cast<char *>(a)) == 0 && blocks.count(static_cast<char *>(other.back())) == 1);
    void *big = device_alloc(limit + kMB);
    frees = 0;
    device_free(big);
    CHECK(frees == 1 && used <= limit);
    device_mem_info(&free_b, &total_b);
    CHECK(free_b == kTotal);
    // what is kept makes room for an allocation that fails
    void *most = device_alloc(kTotal - 64 * kMB);
    CHECK(most != nullptr && used <= kTotal);
    device_free(most);
    // the driver works without the lock
    void *b = device_alloc(3 * kMB);
    device_free(b);
    probe_lock = true;
    void *c = device_alloc(300 * kMB);
    CHECK(!lock_held);
    device_free(c);
    probe_lock = true;
    release_device_memory();
    CHECK(!lock_held && used == 0 && blocks.empty());
    std::printf("ok\n");
    return 0;
}
