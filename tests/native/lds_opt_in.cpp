// LdsOptIn (device_api.h) on a runtime of its own: threads whose launches want different sizes, on two devices.
#include <atomic>
#include <cstdio>
#include <map>
#include <mutex>
#include <thread>

#include "../../thundergbm_amd/csrc/device_api.h"

namespace {
thread_local int device = 0;
std::mutex m;
std::map<std::pair<int, const void *>, int> limit, sets;
}  // namespace

extern "C" {
hipError_t hipGetDevice(int *d) { return *d = device, hipSuccess; }
hipError_t hipFuncGetAttributes(hipFuncAttributes *a, const void *k) {
    *a = hipFuncAttributes{};
    a->sharedSizeBytes = k == reinterpret_cast<const void *>(1) ? 4096 : 100;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *k, hipFuncAttribute, int bytes) {
    std::lock_guard<std::mutex> lock(m);
    limit[{device, k}] = bytes;
    ++sets[{device, k}];
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return ""; }
}
namespace tgbm {
void fatal(const char *fmt, ...) { std::puts(fmt), std::abort(); }
}  // namespace tgbm

int main() {
    static tgbm::LdsOptIn opt_in;
    const void *a = reinterpret_cast<const void *>(1), *b = reinterpret_cast<const void *>(2);
    std::atomic<int> refused{0};
    std::thread threads[8];
    for (int t = 0; t < 8; ++t)
        threads[t] = std::thread([&, t] {
            device = t & 1;
            for (int i = 0; i < 2000; ++i) {
                opt_in({a, b});
                std::lock_guard<std::mutex> lock(m);  // (the launch)
                if (limit[{device, a}] != 160 * 1024 - 4096 || limit[{device, b}] != 160 * 1024 - 100) ++refused;
            }
        });
    for (auto &t : threads) t.join();
    for (auto &s : sets)
        if (s.second != 1) ++refused;
    std::printf("%d launches refused, %zu limits set\n", refused.load(), sets.size());
    return refused == 0 && sets.size() == 4 ? 0 : 1;
}
