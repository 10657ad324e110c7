// Device blocks and streams that outlive one call. A training call needs about sixty buffers and a scoring call ten;
// the driver takes 5 to 500 us per block and as much to take it back (1 M x 100 k CSR rows: 17 of a call's 220 ms,
// 500 k rows x 8 classes: 4 of 31 ms, one scored row: a third of the call), a stream 60 to 200 us. Freed blocks are
// therefore kept, per device, for the next call of a similar size.
//
// What is kept is bounded: at most an eighth of the device's memory, no block longer than kKeepCalls calls without a
// use, four streams; everything goes back to the driver when an allocation fails or on tgbm_release_memory().
// Any thread may allocate and free; a block is only freed by its owner after the stream that used it was synchronised,
// so whichever stream the next owner works on finds it idle.
#include <list>
#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "../../include/thundergbm.h"
#include "device_api.h"

namespace tgbm {
namespace {

constexpr long kKeepCalls = 16;
constexpr size_t kKeepStreams = 4;

struct Kept {
    void *p;
    long call;  // DevicePool::calls when the block was given back
};

struct DevicePool {
    std::multimap<size_t, Kept> blocks;  // by size
    size_t kept_bytes = 0;
    size_t limit = 0;  // 0: not asked yet
    long calls = 0;
    std::vector<hipStream_t> streams;
};

struct Live {
    size_t bytes;
    int device;
};

struct Pools {
    std::mutex mutex;
    std::map<int, DevicePool> of_device;
    std::unordered_map<void *, Live> live;
    std::unordered_map<hipStream_t, int> stream_device;
};

// (never destroyed: sessions that the interpreter drops at its very end still give their blocks back)
Pools &pools() {
    static Pools *p = new Pools;
    return *p;
}

int current_device() {
    int dev = 0;
    HIP_CHECK(hipGetDevice(&dev));
    return dev;
}

// Sizes in steps of at most an eighth, so that calls on data of about the same size find each other's blocks.
size_t rounded(size_t bytes) {
    if (bytes <= 4096) return 4096;
    if (bytes >= (size_t)1 << 28) return (bytes + ((size_t)1 << 21) - 1) >> 21 << 21;
    size_t step = 512;
    while (step * 16 <= bytes) step *= 2;
    return (bytes + step - 1) / step * step;
}

void drop(DevicePool &pool, std::multimap<size_t, Kept>::iterator it) {
    pool.kept_bytes -= it->first;
    (void)hipFree(it->second.p);
    pool.blocks.erase(it);
}

void drop_all(DevicePool &pool) {
    while (!pool.blocks.empty()) drop(pool, pool.blocks.begin());
}

}  // namespace

void *device_alloc(size_t bytes) {
    const size_t want = rounded(bytes);
    const int dev = current_device();
    Pools &all = pools();
    std::lock_guard<std::mutex> lock(all.mutex);
    DevicePool &pool = all.of_device[dev];
    void *p = nullptr;
    size_t got = want;
    auto it = pool.blocks.lower_bound(want);
    if (it != pool.blocks.end() && it->first <= want + want / 4) {
        p = it->second.p;
        got = it->first;
        pool.kept_bytes -= got;
        pool.blocks.erase(it);
    } else if (hipMalloc(&p, want) != hipSuccess) {
        (void)hipGetLastError();
        drop_all(pool);
        HIP_CHECK(hipMalloc(&p, want));
    }
    if (pool.limit == 0) {
        size_t free_b = 0, total_b = 0;
        HIP_CHECK(hipMemGetInfo(&free_b, &total_b));
        pool.limit = total_b / 8;
    }
    all.live[p] = Live{got, dev};
    return p;
}

void device_free(void *p) {
    if (p == nullptr) return;
    Pools &all = pools();
    std::lock_guard<std::mutex> lock(all.mutex);
    auto live = all.live.find(p);
    TGBM_CHECK(live != all.live.end(), "device_free: not a block of device_alloc");
    const Live was = live->second;
    all.live.erase(live);
    DevicePool &pool = all.of_device[was.device];
    if (was.bytes > pool.limit) {
        (void)hipFree(p);
        return;
    }
    while (pool.kept_bytes + was.bytes > pool.limit) {  // the longest unused one goes
        auto oldest = pool.blocks.begin();
        for (auto it = pool.blocks.begin(); it != pool.blocks.end(); ++it)
            if (it->second.call < oldest->second.call) oldest = it;
        drop(pool, oldest);
    }
    pool.blocks.emplace(was.bytes, Kept{p, pool.calls});
    pool.kept_bytes += was.bytes;
}

void device_mem_info(size_t *free_b, size_t *total_b) {
    HIP_CHECK(hipMemGetInfo(free_b, total_b));
    const int dev = current_device();
    Pools &all = pools();
    std::lock_guard<std::mutex> lock(all.mutex);
    *free_b += all.of_device[dev].kept_bytes;
}

hipStream_t stream_acquire() {
    const int dev = current_device();
    Pools &all = pools();
    std::lock_guard<std::mutex> lock(all.mutex);
    DevicePool &pool = all.of_device[dev];
    hipStream_t s = nullptr;
    if (!pool.streams.empty()) {
        s = pool.streams.back();
        pool.streams.pop_back();
    } else {
        HIP_CHECK(hipStreamCreate(&s));
    }
    all.stream_device[s] = dev;
    return s;
}

void stream_release(hipStream_t s) {
    Pools &all = pools();
    std::lock_guard<std::mutex> lock(all.mutex);
    auto at = all.stream_device.find(s);
    TGBM_CHECK(at != all.stream_device.end(), "stream_release: not a stream of stream_acquire");
    DevicePool &pool = all.of_device[at->second];
    all.stream_device.erase(at);
    ++pool.calls;
    for (auto it = pool.blocks.begin(); it != pool.blocks.end();) {
        auto next = std::next(it);
        if (pool.calls - it->second.call > kKeepCalls) drop(pool, it);
        it = next;
    }
    if (pool.streams.size() < kKeepStreams)
        pool.streams.push_back(s);
    else
        (void)hipStreamDestroy(s);
}

void release_device_memory() {
    Pools &all = pools();
    std::lock_guard<std::mutex> lock(all.mutex);
    for (auto &entry : all.of_device) {
        drop_all(entry.second);
        for (hipStream_t s : entry.second.streams) (void)hipStreamDestroy(s);
        entry.second.streams.clear();
    }
}

}  // namespace tgbm

extern "C" void tgbm_release_memory(void) {
    tgbm::release_device_memory();
    tgbm::release_transfer_memory();
}
