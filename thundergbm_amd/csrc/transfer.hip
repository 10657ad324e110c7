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
#include <exception>
#include <map>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#include "device_api.h"

namespace tgbm {
namespace {

constexpr size_t kPiece = kPinnedBytes;
constexpr size_t kStagedBytes = (size_t)12 << 20;
// Several smaller arrays one after the other: 60 k rows of 30 values (14 MB with their columns) scored in 578 us by hipMemcpy, in
// 575 to 620 through the pieces; 80 k rows (19 MB) 709 and 690; 110 k rows 1080 and 690.
constexpr size_t kStagedTogether = (size_t)16 << 20;
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

struct TwoPieces {  // of a thread, given back however it ends
    Piece p[2];
    Piece &operator[](int k) { return p[k]; }
    ~TwoPieces() {
        for (const Piece &q : p)
            if (q.host != nullptr) give_piece(q);
    }
};

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

// work(0) .. work(n - 1) side by side; an exception of one of them comes out of the call.
template <typename Work>
void on_threads(int n, const Work &work) {
    std::exception_ptr failed;
    std::mutex mutex;
    auto guarded = [&](int t) {
        try {
            work(t);
        } catch (...) {
            std::lock_guard<std::mutex> lock(mutex);
            if (!failed) failed = std::current_exception();
        }
    };
    std::vector<std::thread> pool;
    pool.reserve((size_t)n);
    int on = 1;
    try {
        for (; on < n; ++on) pool.emplace_back(guarded, on);
    } catch (const std::system_error &) {  // (no thread is left: the caller does their work as well)
    }
    guarded(0);
    for (int t = on; t < n; ++t) guarded(t);
    for (auto &th : pool) th.join();
    if (failed) std::rethrow_exception(failed);
}

}  // namespace

// Sends the jobs' arrays piece by piece. The copies run after what is queued on s, and s waits for them. The pieces of the
// arrays take turns in proportion to their number, so that an array whose conversion is bound by the threads and one
// whose copy is bound by PCIe share the time. With the labels behind them, a session of 1.12 GB of floats, 280 M indices
// narrowed to bytes and 10 M labels: 54 -> 39 ms.
// arrived: UploadSet::send_in_order.
void send_jobs(hipStream_t s, const std::vector<UploadSet::Job> &jobs, int threads, const std::function<void(size_t)> *arrived) {
    struct Turn {
        double at;
        size_t job, offset;
    };
    std::vector<Turn> turns;
    std::vector<std::atomic<int>> unsent(jobs.size());  // pieces
    for (size_t j = 0; j < jobs.size(); ++j) {
        const size_t m = (jobs[j].bytes + kPiece - 1) / kPiece;
        const double from = arrived != nullptr ? (double)j : jobs[j].late ? 1.0 : 0.0;
        for (size_t i = 0; i < m; ++i) turns.push_back({((double)i + 0.5) / (double)m + from, j, i * kPiece});
        unsent[j] = (int)m;
    }
    if (turns.empty()) return;
    std::stable_sort(turns.begin(), turns.end(), [](const Turn &a, const Turn &b) { return a.at < b.at; });
    int dev = 0;
    HIP_CHECK(hipGetDevice(&dev));
    const int n_thr = (int)std::min<size_t>(turns.size(), (size_t)threads);
    const std::array<hipStream_t, 2> to = copy_streams(dev);
    hipEvent_t order[2];
    for (hipEvent_t &e : order) HIP_CHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    HIP_CHECK(hipEventRecord(order[0], s));
    for (hipStream_t c : to) HIP_CHECK(hipStreamWaitEvent(c, order[0], 0));
    std::atomic<size_t> next{0};
    std::mutex arrival;
    auto let_wait = [&] {
        for (int b = 0; b < 2; ++b) {
            HIP_CHECK(hipEventRecord(order[b], to[b]));
            HIP_CHECK(hipStreamWaitEvent(s, order[b], 0));
        }
    };
    size_t told = 0;  // jobs that `arrived` has been called for
    auto tell = [&] {
        std::lock_guard<std::mutex> lock(arrival);
        for (;;) {  // (while the calls below run, other threads may have queued the last copies of the next ones)
            size_t upto = told;
            while (upto < jobs.size() && unsent[upto] == 0) ++upto;
            if (upto == told) return;
            let_wait();  // (all copies of these jobs are queued - those of the next one may not have been when the last wait was)
            for (; told < upto; ++told) (*arrived)(told);
        }
    };
    if (arrived != nullptr) tell();  // (jobs without a byte)
    auto work = [&](int t) {
        if (t > 0) HIP_CHECK(hipSetDevice(dev));
        TwoPieces mine;
        int k = 0;
        for (size_t i = next++; i < turns.size(); i = next++, k ^= 1) {
            if (mine[k].host == nullptr) mine[k] = take_piece();
            if (mine[k].in_flight) HIP_CHECK(hipEventSynchronize(mine[k].sent));
            const UploadSet::Job &job = jobs[turns[i].job];
            const size_t off = turns[i].offset, len = std::min(kPiece, job.bytes - off);
            if (job.source) std::memcpy(mine[k].host, static_cast<const char *>(job.source()) + off, len);
            else job.fill(mine[k].host, off, len);
            HIP_CHECK(hipMemcpyAsync(static_cast<char *>(job.dst) + off, mine[k].host, len, hipMemcpyHostToDevice, to[i & 1]));
            HIP_CHECK(hipEventRecord(mine[k].sent, to[i & 1]));
            mine[k].in_flight = true;
            if (--unsent[turns[i].job] == 0 && arrived != nullptr) tell();
        }
    };
    on_threads(n_thr, work);
    if (arrived == nullptr) let_wait();  // (else it has happened after the last copy)
    for (hipEvent_t e : order) HIP_CHECK(hipEventDestroy(e));
}

void upload_large(hipStream_t s, void *dst, const void *src, size_t bytes) {
    if (bytes < kStagedBytes) {
        if (bytes) HIP_CHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s));
        return;
    }
    UploadSet set;
    set.add(dst, src, bytes);
    set.send(s);
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
    UploadSet set;
    set.add_doubles(dst, src, count);
    set.send(s);
}

void UploadSet::add(void *dst, const void *src, size_t bytes) { jobs_.push_back({dst, bytes, [src] { return src; }, nullptr, false}); }

void UploadSet::add_doubles(float *dst, const double *src, size_t count) {
    jobs_.push_back({dst, count * sizeof(float), nullptr, [src](char *to, size_t off, size_t len) {
        doubles_to_floats(reinterpret_cast<float *>(to), src + off / sizeof(float), len / sizeof(float));
    }, false});
}

void UploadSet::add_late(void *dst, size_t bytes, std::function<const void *()> source) {
    jobs_.push_back({dst, bytes, std::move(source), nullptr, true});
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

}  // namespace

template <typename Narrow>
bool UploadSet::add_narrow(int *dst, const int *src, size_t count) {
    constexpr unsigned kMost = (1u << (8 * sizeof(Narrow))) - 1u;
    // (the first and last few thousand tell most arrays that do not fit)
    unsigned seen = 0;
    for (size_t i = 0; i < std::min<size_t>(count, 4096); ++i) seen |= (unsigned)src[i] | (unsigned)src[count - 1 - i];
    if (seen > kMost) return false;
    Narrow *narrow = nullptr;
    device_alloc_to(narrow, count * sizeof(Narrow));
    auto fits = std::make_shared<std::atomic<bool>>(true);
    jobs_.push_back({narrow, count * sizeof(Narrow), nullptr, [src, fits](char *to, size_t off, size_t len) {
        const int *from = src + off / sizeof(Narrow);
        Narrow *out = reinterpret_cast<Narrow *>(to);
        const size_t m = len / sizeof(Narrow);
        unsigned any = 0;
        for (size_t i = 0; i < m; ++i) {
            any |= (unsigned)from[i];
            out[i] = (Narrow)from[i];
        }
        if (any > kMost) *fits = false;
    }, false});
    columns_.push_back({dst, src, count, (int)sizeof(Narrow), narrow, fits, jobs_.size() - 1});
    return true;
}

void UploadSet::add_columns(int *dst, const int *src, size_t count) {
    if (count * sizeof(int) >= kStagedBytes && (add_narrow<uint8_t>(dst, src, count) || add_narrow<uint16_t>(dst, src, count))) return;
    add(dst, src, count * sizeof(int));
}

void UploadSet::send(hipStream_t s) {
    size_t total = 0;
    bool plain = true;
    for (const Job &j : jobs_) {
        total += j.bytes;
        plain = plain && j.source;
    }
    if (plain && total < kStagedBytes) {
        for (const Job &j : jobs_)
            if (j.bytes) HIP_CHECK(hipMemcpyAsync(j.dst, j.source(), j.bytes, hipMemcpyHostToDevice, s));
        return;
    }
    send_jobs(s, jobs_, plain ? 4 : 8, nullptr);
    for (const Columns &c : columns_) widen(s, c);
    release_narrow(s);
}

// (a column index in the middle that did not fit: the array goes up once more)
void UploadSet::widen(hipStream_t s, const Columns &c) {
    const unsigned grid = (unsigned)std::min<size_t>(4096, c.count / 1024 + 1);
    if (*c.fits) {
        if (c.width == 1) k_widen<uint8_t><<<grid, 256, 0, s>>>(c.count, static_cast<const uint8_t *>(c.narrow), c.dst);
        else k_widen<uint16_t><<<grid, 256, 0, s>>>(c.count, static_cast<const uint16_t *>(c.narrow), c.dst);
        return;
    }
    UploadSet again;
    if (c.width == 2 || !again.add_narrow<uint16_t>(c.dst, c.src, c.count)) again.add(c.dst, c.src, c.count * sizeof(int));
    again.send(s);
}

void UploadSet::release_narrow(hipStream_t s) {
    if (columns_.empty()) return;
    HIP_CHECK(hipStreamSynchronize(s));
    for (const Columns &c : columns_) device_free(c.narrow);
    columns_.clear();
}

void UploadSet::send_in_order(hipStream_t s, const std::function<void(size_t)> &arrived) {
    size_t total = 0, largest = 0;
    bool plain = true;
    for (const Job &j : jobs_) {
        total += j.bytes;
        largest = std::max(largest, j.bytes);
        plain = plain && j.source;
    }
    if (!plain || largest >= kStagedBytes || total >= kStagedTogether) {
        const std::function<void(size_t)> widened = [&](size_t j) {
            for (const Columns &c : columns_)
                if (c.job == j) widen(s, c);
            arrived(j);
        };
        send_jobs(s, jobs_, plain ? 4 : 8, &widened);
        release_narrow(s);
        return;
    }
    for (size_t j = 0; j < jobs_.size(); ++j) {
        if (jobs_[j].bytes) HIP_CHECK(hipMemcpyAsync(jobs_[j].dst, jobs_[j].source(), jobs_[j].bytes, hipMemcpyHostToDevice, s));
        arrived(j);
    }
}

// Threads take turns at kDownChunk bytes: each has its next chunk copied to one half of a pinned piece while it empties the
// other. A hipMemcpy to pageable memory copies a megabyte to a buffer of its own, then empties that, then goes on:
// 4 MB in 320 us, here 220.
constexpr size_t kDownChunk = (size_t)512 << 10;
constexpr size_t kDownStaged = (size_t)1 << 20;

void download_large(hipStream_t s, hipStream_t other, void *dst, const void *src, size_t bytes) {
    if (bytes < kDownStaged) {
        if (bytes) HIP_CHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s));
        HIP_CHECK(hipStreamSynchronize(s));
        return;
    }
    const size_t chunks = (bytes + kDownChunk - 1) / kDownChunk;
    const int n_thr = (int)std::min<size_t>(4, (chunks + 1) / 2);
    int dev = 0;
    HIP_CHECK(hipGetDevice(&dev));
    // (the call's own streams: on the copy streams, which are the whole process's, other calls' copies would wait for its kernels)
    const std::array<hipStream_t, 2> from{s, other};
    hipEvent_t ready;
    HIP_CHECK(hipEventCreateWithFlags(&ready, hipEventDisableTiming));
    HIP_CHECK(hipEventRecord(ready, s));
    HIP_CHECK(hipStreamWaitEvent(other, ready, 0));
    auto work = [&](int t) {
        if (t > 0) HIP_CHECK(hipSetDevice(dev));
        TwoPieces half;
        for (Piece &p : half.p) {
            p = take_piece();
            if (p.in_flight) HIP_CHECK(hipEventSynchronize(p.sent));
        }
        auto length = [&](size_t c) { return std::min(kDownChunk, bytes - c * kDownChunk); };
        auto request = [&](size_t c, Piece &p, hipStream_t on) {
            HIP_CHECK(hipMemcpyAsync(p.host, static_cast<const char *>(src) + c * kDownChunk, length(c), hipMemcpyDeviceToHost, on));
            HIP_CHECK(hipEventRecord(p.sent, on));
            p.in_flight = true;
        };
        int k = 0;
        if ((size_t)t < chunks) request((size_t)t, half[0], from[t & 1]);
        for (size_t c = (size_t)t; c < chunks; c += (size_t)n_thr, k ^= 1) {
            if (c + (size_t)n_thr < chunks) request(c + (size_t)n_thr, half[k ^ 1], from[t & 1]);
            HIP_CHECK(hipEventSynchronize(half[k].sent));
            half[k].in_flight = false;
            std::memcpy(static_cast<char *>(dst) + c * kDownChunk, half[k].host, length(c));
        }
    };
    on_threads(n_thr, work);
    HIP_CHECK(hipEventDestroy(ready));
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
