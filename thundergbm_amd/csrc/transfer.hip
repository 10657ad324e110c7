// Host -> device copies of the callers' pageable arrays.
//
// A hipMemcpy of pageable memory reaches 31 GB/s here, PCIe takes 57 GB/s. Arrays of kStagedBytes and more therefore go
// through pinned pieces that a few host threads fill side by side: every thread has two pieces of its own and sends one
// by DMA while it fills the other, so no thread waits for another. A DMA leaves a gap of about 16 us before the next
// one of its stream, so the pieces alternate between two streams. 1.12 GB: 35.9 ms as one hipMemcpy, 23.8 ms through
// 4 MB pieces on one stream, 19.9 ms (56.4 GB/s) on two (21.2 with two threads instead of four, the same with three
// streams or 8 MB pieces); 56 MB: 1.75 -> 1.15 ms; 12 MB: 0.34 -> 0.33 ms, which is where the line lies.
// The pinned pieces are kept for later calls, at most kKeepPieces.
#include <algorithm>
#include <array>
#include <atomic>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

#include "device_api.h"

namespace tgbm {
namespace {

constexpr size_t kPiece = kPinnedBytes;
constexpr size_t kStagedBytes = (size_t)12 << 20;
constexpr size_t kKeepPieces = 16;

struct Piece {
    char *host = nullptr;
    hipEvent_t sent = nullptr;  // the DMA that reads the piece
    bool in_flight = false;
};

struct PieceStore {
    std::mutex mutex;
    std::vector<Piece> pieces;
    std::map<int, std::array<hipStream_t, 2>> streams;  // per device
    std::map<char *, Piece> lent;                       // by pinned_acquire
};

PieceStore &piece_store() {
    static PieceStore *s = new PieceStore;  // (never destroyed, like the device pool)
    return *s;
}

Piece take_piece() {
    PieceStore &store = piece_store();
    {
        std::lock_guard<std::mutex> lock(store.mutex);
        if (!store.pieces.empty()) {
            Piece p = store.pieces.back();
            store.pieces.pop_back();
            return p;
        }
    }
    Piece p;
    HIP_CHECK(hipHostMalloc(reinterpret_cast<void **>(&p.host), kPiece, hipHostMallocPortable));
    HIP_CHECK(hipEventCreateWithFlags(&p.sent, hipEventDisableTiming));
    return p;
}

void destroy_piece(const Piece &p) {
    if (p.in_flight) (void)hipEventSynchronize(p.sent);
    (void)hipEventDestroy(p.sent);
    (void)hipHostFree(p.host);
}

void give_piece(const Piece &p) {  // (possibly still in flight: whoever fills it next waits for `sent`)
    PieceStore &store = piece_store();
    {
        std::lock_guard<std::mutex> lock(store.mutex);
        if (store.pieces.size() < kKeepPieces) {
            store.pieces.push_back(p);
            return;
        }
    }
    destroy_piece(p);
}

std::array<hipStream_t, 2> copy_streams(int dev) {
    PieceStore &store = piece_store();
    std::lock_guard<std::mutex> lock(store.mutex);
    auto it = store.streams.find(dev);
    if (it == store.streams.end()) {
        std::array<hipStream_t, 2> two;
        for (hipStream_t &c : two) HIP_CHECK(hipStreamCreateWithFlags(&c, hipStreamNonBlocking));
        it = store.streams.emplace(dev, two).first;
    }
    return it->second;
}

// Sends `bytes` of device data piece by piece; fill(to, offset, length) writes bytes [offset, offset + length) of it.
// The copies run after what is queued on s, and s waits for them.
template <typename Fill>
void send_staged(hipStream_t s, void *dst, size_t bytes, int threads, const Fill &fill) {
    const size_t n_pieces = (bytes + kPiece - 1) / kPiece;
    int dev = 0;
    HIP_CHECK(hipGetDevice(&dev));
    const int n_thr = (int)std::min<size_t>(n_pieces, (size_t)threads);
    const std::array<hipStream_t, 2> to = copy_streams(dev);
    hipEvent_t order[2];
    for (hipEvent_t &e : order) HIP_CHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    HIP_CHECK(hipEventRecord(order[0], s));
    for (hipStream_t c : to) HIP_CHECK(hipStreamWaitEvent(c, order[0], 0));
    auto work = [&](int t) {
        if (t > 0) HIP_CHECK(hipSetDevice(dev));
        Piece mine[2];
        int k = 0;
        for (size_t i = (size_t)t; i < n_pieces; i += (size_t)n_thr, k ^= 1) {
            if (mine[k].host == nullptr) mine[k] = take_piece();
            if (mine[k].in_flight) HIP_CHECK(hipEventSynchronize(mine[k].sent));
            const size_t off = i * kPiece, len = std::min(kPiece, bytes - off);
            fill(mine[k].host, off, len);
            HIP_CHECK(hipMemcpyAsync(static_cast<char *>(dst) + off, mine[k].host, len, hipMemcpyHostToDevice, to[i & 1]));
            HIP_CHECK(hipEventRecord(mine[k].sent, to[i & 1]));
            mine[k].in_flight = true;
        }
        for (Piece &p : mine)
            if (p.host != nullptr) give_piece(p);
    };
    std::vector<std::thread> pool;
    for (int t = 1; t < n_thr; ++t) pool.emplace_back(work, t);
    work(0);
    for (auto &th : pool) th.join();
    for (int b = 0; b < 2; ++b) {
        HIP_CHECK(hipEventRecord(order[b], to[b]));
        HIP_CHECK(hipStreamWaitEvent(s, order[b], 0));
        HIP_CHECK(hipEventDestroy(order[b]));
    }
}

}  // namespace

void upload_large(hipStream_t s, void *dst, const void *src, size_t bytes) {
    if (bytes < kStagedBytes) {
        if (bytes) HIP_CHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s));
        return;
    }
    send_staged(s, dst, bytes, 4,
                [&](char *to, size_t off, size_t len) { std::memcpy(to, static_cast<const char *>(src) + off, len); });
}

void doubles_to_floats(float *to, const double *from, size_t count) {
    unsigned *out = reinterpret_cast<unsigned *>(to);
    for (size_t i = 0; i < count; ++i) {
        const double d = from[i];
        const float f = (float)d;
        unsigned bits;
        std::memcpy(&bits, &f, 4);
        // zero: +0; a value that is only zero as a float: -0 (see dense_to_csr)
        out[i] = (bits & 0x7fffffffu) != 0 ? bits : (d == 0.0 ? 0u : 0x80000000u);
    }
}

// The conversion happens while the pieces are filled, so the doubles cross PCIe as floats.
void upload_doubles_as_floats(hipStream_t s, float *dst, const double *src, size_t count) {
    send_staged(s, dst, count * sizeof(float), 8, [&](char *to, size_t off, size_t len) {
        doubles_to_floats(reinterpret_cast<float *>(to), src + off / sizeof(float), len / sizeof(float));
    });
}

namespace {

template <typename Narrow>
__global__ __launch_bounds__(256) void k_widen(size_t n, const Narrow *__restrict__ in, int *__restrict__ out) {
    // four indices per thread: one 4- or 8-byte load, one 16-byte store
    struct alignas(4 * sizeof(Narrow)) In {
        Narrow v[4];
    };
    const size_t quads = n / 4;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < quads; i += (size_t)gridDim.x * 256) {
        const In q = reinterpret_cast<const In *>(in)[i];
        reinterpret_cast<int4 *>(out)[i] = make_int4(q.v[0], q.v[1], q.v[2], q.v[3]);
    }
    if (blockIdx.x == 0 && threadIdx.x < (unsigned)(n & 3)) out[quads * 4 + threadIdx.x] = in[quads * 4 + threadIdx.x];
}

// Sends the indices as `Narrow` words; false (and nothing usable on the device) if one does not fit.
template <typename Narrow>
bool send_narrow(hipStream_t s, int *dst, const int *src, size_t count) {
    constexpr unsigned kMost = (1u << (8 * sizeof(Narrow))) - 1u;
    // (the first and last few thousand tell most arrays that do not fit)
    unsigned seen = 0;
    for (size_t i = 0; i < std::min<size_t>(count, 4096); ++i) seen |= (unsigned)src[i] | (unsigned)src[count - 1 - i];
    if (seen > kMost) return false;
    Narrow *narrow = nullptr;
    device_alloc_to(narrow, count * sizeof(Narrow));
    std::atomic<bool> fits{true};
    send_staged(s, narrow, count * sizeof(Narrow), 8, [&](char *to, size_t off, size_t len) {
        const int *from = src + off / sizeof(Narrow);
        Narrow *out = reinterpret_cast<Narrow *>(to);
        const size_t m = len / sizeof(Narrow);
        unsigned any = 0;
        for (size_t i = 0; i < m; ++i) {
            any |= (unsigned)from[i];
            out[i] = (Narrow)from[i];
        }
        if (any > kMost) fits = false;
    });
    if (fits) k_widen<Narrow><<<(unsigned)std::min<size_t>(4096, count / 1024 + 1), 256, 0, s>>>(count, narrow, dst);
    HIP_CHECK(hipStreamSynchronize(s));
    device_free(narrow);
    return fits;
}

}  // namespace

// 280 M indices below 256: 20 -> 6 ms (the threads' conversion bounds it).
void upload_columns(hipStream_t s, int *dst, const int *src, size_t count) {
    if (count * sizeof(int) >= 4 * kStagedBytes &&
        (send_narrow<uint8_t>(s, dst, src, count) || send_narrow<uint16_t>(s, dst, src, count)))
        return;
    upload_large(s, dst, src, count * sizeof(int));
}

void *pinned_acquire() {
    const Piece p = take_piece();
    if (p.in_flight) HIP_CHECK(hipEventSynchronize(p.sent));
    PieceStore &store = piece_store();
    std::lock_guard<std::mutex> lock(store.mutex);
    store.lent[p.host] = p;
    return p.host;
}

void pinned_release(void *host) {
    PieceStore &store = piece_store();
    Piece p;
    {
        std::lock_guard<std::mutex> lock(store.mutex);
        auto it = store.lent.find(static_cast<char *>(host));
        TGBM_CHECK(it != store.lent.end(), "pinned_release: not a block of pinned_acquire");
        p = it->second;
        store.lent.erase(it);
    }
    p.in_flight = false;
    give_piece(p);
}

void release_transfer_memory() {
    PieceStore &store = piece_store();
    std::lock_guard<std::mutex> lock(store.mutex);
    for (const Piece &p : store.pieces) destroy_piece(p);
    store.pieces.clear();
}

}  // namespace tgbm
