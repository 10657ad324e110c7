// Device blocks and streams that outlive one call. A training call needs about sixty buffers and a scoring call ten;
// the driver takes 5 to 500 us per block and as much to take it back (1 M x 100 k CSR rows: 17 of a call's 220 ms,
// 500 k rows x 8 classes: 4 of 31 ms, one scored row: a third of the call), a stream 60 to 200 us. Freed blocks are
// therefore kept, per device, for the next call of a similar size.
//
// What is kept is bounded: a part of the device's memory (kKeepPart) and four streams. Beyond that the blocks that have
// lain there longest go back to the driver for those that a call gives: a call pays for its own bytes, never for what an
// earlier one has left (sixty blocks of a training call take the driver up to 13 ms: not in a request of 24 us that
// happens to come later). Everything goes back when an allocation fails or on tgbm_release_memory().
// Any thread may allocate and free, and the driver is called without the lock: a slow call of one thread holds up no
// other. A block is only freed by its owner after the stream that used it was synchronised, so whichever stream the
// next owner works on finds it idle.
#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "../../include/thundergbm.h"
#include "device_api.h"

namespace tgbm {
namespace {

// Part of the device's memory that an idle process may hold: 9 GB of 288. The calls of a 10 M x 28 training leave 6.2 GB, of
// 1 M x 100 k CSR rows 2.6 GB; with 4.5 GB the former take 179 instead of 159 ms, without any 184.
constexpr size_t kKeepPart = 32;
constexpr size_t kKeepStreams = 4;

struct Kept {
    void *p;
    long since;  // DevicePool::given when the block was given back
};

struct DevicePool {
    std::multimap<size_t, Kept> blocks;  // by size
    size_t kept_bytes = 0;
    size_t limit = 0;  // 0: not asked yet
    long given = 0;
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

// Takes a block out of the pool; the caller frees it once the lock is gone.
void *take(DevicePool &pool, std::multimap<size_t, Kept>::iterator it) {
    void *p = it->second.p;
    pool.kept_bytes -= it->first;
    pool.blocks.erase(it);
    return p;
}

std::vector<void *> take_all(DevicePool &pool) {
    std::vector<void *> out;
    while (!pool.blocks.empty()) out.push_back(take(pool, pool.blocks.begin()));
    return out;
}

void free_all(const std::vector<void *> &blocks) {
    for (void *p : blocks) (void)hipFree(p);
}

}  // namespace

void *device_alloc(size_t bytes) {
    const size_t want = rounded(bytes);
    const int dev = current_device();
    Pools &all = pools();
    bool first = false;
    {
        std::lock_guard<std::mutex> lock(all.mutex);
        DevicePool &pool = all.of_device[dev];
        first = pool.limit == 0;
        auto it = pool.blocks.lower_bound(want);
        if (it != pool.blocks.end() && it->first <= want + want / 4) {
            const size_t got = it->first;
            void *p = take(pool, it);
            all.live[p] = Live{got, dev};
            return p;
        }
    }
    void *p = nullptr;
    for (hipError_t e = hipMalloc(&p, want); e != hipSuccess; e = hipMalloc(&p, want)) {
        (void)hipGetLastError();
        std::vector<void *> kept;
        {
            std::lock_guard<std::mutex> lock(all.mutex);
            kept = take_all(all.of_device[dev]);
        }
        if (kept.empty()) HIP_CHECK(e);
        free_all(kept);
    }
    size_t free_b = 0, total_b = 0;
    if (first) HIP_CHECK(hipMemGetInfo(&free_b, &total_b));
    std::lock_guard<std::mutex> lock(all.mutex);
    if (first) all.of_device[dev].limit = total_b / kKeepPart;
    all.live[p] = Live{want, dev};
    return p;
}

void device_free(void *p) {
    if (p == nullptr) return;
    Pools &all = pools();
    std::vector<void *> out;
    {
        std::lock_guard<std::mutex> lock(all.mutex);
        auto live = all.live.find(p);
        TGBM_CHECK(live != all.live.end(), "device_free: not a block of device_alloc");
        const Live was = live->second;
        all.live.erase(live);
        DevicePool &pool = all.of_device[was.device];
        if (was.bytes > pool.limit) {
            out.push_back(p);
        } else {
            while (pool.kept_bytes + was.bytes > pool.limit) {  // the one that has lain there longest goes
                auto oldest = pool.blocks.begin();
                for (auto it = pool.blocks.begin(); it != pool.blocks.end(); ++it)
                    if (it->second.since < oldest->second.since) oldest = it;
                out.push_back(take(pool, oldest));
            }
            pool.blocks.emplace(was.bytes, Kept{p, pool.given++});
            pool.kept_bytes += was.bytes;
        }
    }
    free_all(out);
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
    hipStream_t s = nullptr;
    {
        std::lock_guard<std::mutex> lock(all.mutex);
        DevicePool &pool = all.of_device[dev];
        if (!pool.streams.empty()) {
            s = pool.streams.back();
            pool.streams.pop_back();
            all.stream_device[s] = dev;
            return s;
        }
    }
    HIP_CHECK(hipStreamCreate(&s));
    std::lock_guard<std::mutex> lock(all.mutex);
    all.stream_device[s] = dev;
    return s;
}

void stream_release(hipStream_t s) {
    Pools &all = pools();
    {
        std::lock_guard<std::mutex> lock(all.mutex);
        auto at = all.stream_device.find(s);
        TGBM_CHECK(at != all.stream_device.end(), "stream_release: not a stream of stream_acquire");
        DevicePool &pool = all.of_device[at->second];
        all.stream_device.erase(at);
        if (pool.streams.size() < kKeepStreams) {
            pool.streams.push_back(s);
            return;
        }
    }
    (void)hipStreamDestroy(s);
}

void release_device_memory() {
    Pools &all = pools();
    std::vector<void *> blocks;
    std::vector<hipStream_t> streams;
    {
        std::lock_guard<std::mutex> lock(all.mutex);
        for (auto &entry : all.of_device) {
            for (void *p : take_all(entry.second)) blocks.push_back(p);
            streams.insert(streams.end(), entry.second.streams.begin(), entry.second.streams.end());
            entry.second.streams.clear();
        }
    }
    free_all(blocks);
    for (hipStream_t s : streams) (void)hipStreamDestroy(s);
}

}  // namespace tgbm

extern "C" void tgbm_release_memory(void) {
    tgbm::release_device_memory();
    tgbm::release_transfer_memory();
}
