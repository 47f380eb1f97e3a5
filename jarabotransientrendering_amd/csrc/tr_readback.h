// Results on their way from the GPU to pageable host memory. Kernels write the result into pinned
// host memory over PCIe, chunk by chunk, and host threads copy finished chunks to the caller's
// array while later ones are written. The runtime's own copy into pageable memory does the same two
// steps in turn on one thread (20 us of PCIe and 65 us of memcpy per MiB: 12-17 GB/s).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>

namespace trb {

// Bytes of a launch: PCIe takes 21 us per MiB, and each launch with its event 9 us more (the event
// writes the caches back), so chunks of 1 MiB reach 31 GB/s and chunks of 2 MiB 38. (One launch whose
// blocks raise a flag per MiB was slower, 24 GB/s: a release to the host per block costs more.)
constexpr size_t kChunk = size_t(2) << 20;
constexpr size_t kPiece = size_t(512) << 10;  // bytes a thread copies at a time
constexpr uint32_t kSlots = 8;                // chunks in a large staging block
constexpr uint32_t kStreams = 4;              // streams of a staging block (hardware queues of a process)
constexpr int kHelpers = 3;                   // copying threads besides the caller's
constexpr size_t kPerThread = size_t(1) << 20;  // least bytes per copying thread (starting one takes ~20 us)

// A pinned block with an event per chunk slot, and streams that take the chunks in turn (one for one slot). Made for
// one device, used by one read at a time.
struct Staging {
    int device = 0;
    uint32_t slots = 0;
    char* host = nullptr;
    hipStream_t stream[kStreams] = {};
    hipEvent_t done[kSlots] = {};

    bool make(int dev, uint32_t n)
    {
        device = dev;
        slots = n;
        if (hipHostMalloc(reinterpret_cast<void**>(&host), n * kChunk, hipHostMallocDefault) != hipSuccess) {
            host = nullptr;
            return false;
        }
        for (uint32_t k = 0; k < std::min(n, kStreams); ++k)
            if (hipStreamCreateWithFlags(&stream[k], hipStreamNonBlocking) != hipSuccess) return stream[k] = nullptr, false;
        for (uint32_t k = 0; k < n; ++k)
            if (hipEventCreateWithFlags(&done[k], hipEventDisableTiming) != hipSuccess) return done[k] = nullptr, false;
        return true;
    }
    void wait()
    {
        for (hipStream_t q : stream)
            if (q) (void)hipStreamSynchronize(q);
    }
    ~Staging()
    {
        for (hipEvent_t e : done)
            if (e) (void)hipEventDestroy(e);
        for (hipStream_t q : stream)
            if (q) (void)hipStreamDestroy(q);
        if (host) (void)hipHostFree(host);
    }
};

// Blocks kept between calls, for any thread: at most 8 of one chunk (a render holds one too) and 2 large
// ones, 48 MiB in all. The pool
// lives until the process ends (its blocks are not freed after the runtime has shut down).
class Pool {
public:
    static Pool& get()
    {
        static Pool* p = new Pool;
        return *p;
    }
    Staging* take(int device, size_t bytes)
    {
        const uint32_t slots = bytes <= kChunk ? 1u : kSlots;
        {
            std::lock_guard<std::mutex> lock(mutex_);
            for (Staging*& f : free_)
                if (f && f->device == device && f->slots == slots) {
                    Staging* s = f;
                    f = nullptr;
                    return s;
                }
        }
        Staging* s = new (std::nothrow) Staging;
        if (s && !s->make(device, slots)) {
            delete s;
            s = nullptr;
        }
        return s;
    }
    void give(Staging* s)
    {
        {
            std::lock_guard<std::mutex> lock(mutex_);
            int same = 0;
            for (Staging* f : free_) same += f && f->slots == s->slots;
            if (same < (s->slots == 1 ? kKeptSmall : kKeptLarge))
                for (Staging*& f : free_)
                    if (!f) {
                        f = s;
                        return;
                    }
        }
        delete s;
    }

private:
    static constexpr int kKeptSmall = 8, kKeptLarge = 2;
    std::mutex mutex_;
    Staging* free_[kKeptSmall + kKeptLarge] = {};
};

// A small pinned block for as long as this object lives.
class Lease {
public:
    Lease() = default;
    Lease(const Lease&) = delete;
    Lease& operator=(const Lease&) = delete;
    ~Lease()
    {
        if (block_) Pool::get().give(block_);
    }
    bool take()
    {
        int device = 0;
        if (hipGetDevice(&device) != hipSuccess) return false;
        block_ = Pool::get().take(device, 1);
        return block_ != nullptr;
    }
    char* host() const { return block_->host; }

private:
    Staging* block_ = nullptr;
};

// Fills out[0, bytes) with what `launch(stream, dst, offset, size)` makes the GPU write to the pinned
// address dst for the byte range [offset, offset + size) of the result, on that stream (offsets are
// multiples of kChunk, sizes at most kChunk). What the launches read must be complete when this is
// called, or be written on `own`, which then takes all the launches. Returns when `out` is complete; on
// an error, when nothing more is in flight.
template <class Launch>
hipError_t read_back(void* out, size_t bytes, Launch launch, hipStream_t own = nullptr)
{
    if (bytes == 0) return hipSuccess;
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    Staging* st = Pool::get().take(device, bytes);
    if (!st) return hipErrorOutOfMemory;
    constexpr uint64_t kPieces = kChunk / kPiece;
    const uint64_t chunks = (bytes + kChunk - 1) / kChunk, pieces = (bytes + kPiece - 1) / kPiece;
    std::atomic<uint64_t> next{0}, submitted{0}, copied{0};  // pieces claimed / submitted / copied
    std::atomic<uint32_t> slot_copied[kSlots] = {};           // pieces copied of the chunk in each slot
    std::atomic<int> error{int(hipSuccess)};
    // copies one submitted piece that nobody has claimed; false if there is none now
    auto copy_one = [&]() {
        uint64_t k = next.load();
        do {
            if (k >= submitted.load()) return false;
        } while (!next.compare_exchange_weak(k, k + 1));
        const uint32_t slot = uint32_t((k / kPieces) % st->slots);
        const hipError_t w = hipEventSynchronize(st->done[slot]);
        if (w != hipSuccess) {
            error = int(w);
            return false;
        }
        const size_t at = size_t(k) * kPiece;
        std::memcpy(static_cast<char*>(out) + at, st->host + slot * kChunk + at % kChunk, std::min(kPiece, bytes - at));
        slot_copied[slot].fetch_add(1);
        copied.fetch_add(1);
        return true;
    };
    auto help = [&]() {
        while (next.load() < pieces && error.load() == int(hipSuccess))
            if (!copy_one()) std::this_thread::yield();
    };
    std::thread helpers[kHelpers];
    int n_helpers = 0;
    const int want = int(std::min<size_t>(kHelpers, bytes / kPerThread));
    // the caller's thread submits chunks while slots are free and copies otherwise
    for (uint64_t k = 0; copied.load() < pieces && error.load() == int(hipSuccess);) {
        const uint32_t slot = uint32_t(k % st->slots);
        if (k < chunks && (k < st->slots || slot_copied[slot].load() == kPieces)) {
            slot_copied[slot].store(0);
            const size_t at = size_t(k) * kChunk;
            const hipStream_t stream = own ? own : st->stream[k & 1];
            e = launch(stream, st->host + slot * kChunk, at, std::min(kChunk, bytes - at));
            if (e == hipSuccess) e = hipEventRecord(st->done[slot], stream);
            if (e != hipSuccess) {
                error = int(e);
                break;
            }
            ++k;
            submitted.store(std::min(pieces, k * kPieces));
            if (k == std::min<uint64_t>(chunks, 2)) {
                try {
                    while (n_helpers < want) helpers[n_helpers] = std::thread(help), ++n_helpers;
                } catch (...) {  // no more threads: those that started and this one copy
                }
            }
        } else if (!copy_one()) {
            std::this_thread::yield();
        }
    }
    for (int t = 0; t < n_helpers; ++t) helpers[t].join();
    if (error.load() != int(hipSuccess)) {  // nothing writes the block any more
        st->wait();
        if (own) (void)hipStreamSynchronize(own);
    }
    Pool::get().give(st);
    return hipError_t(error.load());
}

// Calls work(stream, event, pinned, first, count) for every range of at most `per` items of [0, n), by
// `threads` threads at once, each with a chunk of pinned memory, an event and (up to kStreams) a stream
// of its own. `work` returns with nothing of its own in flight, unless it fails. Returns when
// all ranges are done, or on an error, when nothing is in flight.
template <class Work>
hipError_t run_chunks(size_t n, size_t per, uint32_t threads, Work work)
{
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    threads = std::min(std::max(threads, 1u), kSlots);
    Staging* st = Pool::get().take(device, threads * kChunk);
    if (!st) return hipErrorOutOfMemory;
    std::atomic<size_t> next{0};
    std::atomic<int> error{int(hipSuccess)};
    auto run = [&](uint32_t t) {
        for (size_t first; error.load() == int(hipSuccess) && (first = next.fetch_add(per)) < n;) {
            const hipError_t w = work(st->stream[t % kStreams], st->done[t], st->host + t * kChunk, first, std::min(per, n - first));
            if (w != hipSuccess) error = int(w);
        }
    };
    std::thread helpers[kSlots];
    uint32_t started = 0;
    try {
        for (uint32_t t = 1; t < threads; ++t, ++started)
            helpers[started] = std::thread([&run, t, device] {
                (void)hipSetDevice(device);
                run(t);
            });
    } catch (...) {  // no more threads: those that started and this one do the work
    }
    run(0);
    for (uint32_t t = 0; t < started; ++t) helpers[t].join();
    if (error.load() != int(hipSuccess)) st->wait();  // nothing uses the block any more
    Pool::get().give(st);
    return hipError_t(error.load());
}

}  // namespace trb
