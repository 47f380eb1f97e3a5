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
constexpr uint32_t kSlots = 8;                // chunks that one call uses at most
constexpr int kHelpers = 3;                   // copying threads besides the caller's
constexpr size_t kPerThread = size_t(1) << 20;  // least bytes per copying thread (starting one takes ~20 us)

// A chunk of pinned memory with a stream and an event, made for one device and used by one call at a time.
struct Chunk {
    int device = 0;
    uint32_t place = 0;  // in the pool
    char* host = nullptr;
    hipStream_t stream = nullptr;
    hipEvent_t done = nullptr;

    // without its memory
    static Chunk* make(int dev, uint32_t place)
    {
        Chunk* c = new (std::nothrow) Chunk;
        if (!c) return nullptr;
        c->device = dev;
        c->place = place;
        if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) c->stream = nullptr;
        else if (hipEventCreateWithFlags(&c->done, hipEventDisableTiming) != hipSuccess) c->done = nullptr;
        if (c->done) return c;
        (void)hipGetLastError();  // (the next launch would report it)
        delete c;
        return nullptr;
    }
    bool fill()
    {
        if (host) return true;
        if (hipHostMalloc(reinterpret_cast<void**>(&host), kChunk, hipHostMallocDefault) == hipSuccess) return true;
        (void)hipGetLastError();
        host = nullptr;
        return false;
    }
    ~Chunk()
    {
        if (done) (void)hipEventDestroy(done);
        if (stream) (void)hipStreamDestroy(stream);
        if (host) (void)hipHostFree(host);
    }
};

// Chunks kept between calls, for any thread: kMost in all, 64 MiB. A call takes as many as it wants of those
// that are free, and at least one, which is freed again where none was; so threads that read at once share the
// chunks instead of making more. (With blocks of eight chunks, two of them kept, 4, 8 and 16 threads reading
// 6 MB each took 0.68, 2.1 and 5.0 ms; 0.50, 0.95 and 1.94 with this, the rate of the link.) The streams of
// eight chunks are made together and the first chunks are taken first, so that a call that is alone has its
// streams spread over the hardware queues whatever other streams the process has made between two calls. The
// pool lives until the process ends (its chunks are not freed after the runtime has shut down).
class Pool {
public:
    static Pool& get()
    {
        static Pool* p = new Pool;
        return *p;
    }
    // up to `want` chunks; how many (0: no memory for one)
    uint32_t take(int device, uint32_t want, Chunk** out)
    {
        uint32_t n = 0;
        {
            std::lock_guard<std::mutex> lock(mutex_);
            for (uint32_t k = 0; k < kMost && n < want; ++k) {
                if (!at_[k])
                    for (uint32_t j = k; j < k / kSlots * kSlots + kSlots; ++j)
                        if (!at_[j]) at_[j] = Chunk::make(device, j);
                if (!at_[k]) break;
                if (used_[k] || at_[k]->device != device) continue;
                used_[k] = true;
                out[n++] = at_[k];
            }
        }
        uint32_t filled = 0;
        while (filled < n && out[filled]->fill()) ++filled;
        give(out + filled, n - filled);
        if (n == 0 && (out[0] = Chunk::make(device, kMost))) {
            if (out[0]->fill()) return 1;
            delete out[0];
        }
        return filled;
    }
    void give(Chunk* const* chunks, uint32_t n)
    {
        for (uint32_t k = 0; k < n; ++k) {
            if (chunks[k]->place == kMost) {
                delete chunks[k];
                continue;
            }
            std::lock_guard<std::mutex> lock(mutex_);
            used_[chunks[k]->place] = false;
        }
    }

private:
    static constexpr uint32_t kMost = 32;
    std::mutex mutex_;
    Chunk* at_[kMost] = {};
    bool used_[kMost] = {};
};

// The chunks of one call.
class Chunks {
public:
    Chunks() = default;
    Chunks(const Chunks&) = delete;
    Chunks& operator=(const Chunks&) = delete;
    ~Chunks() { Pool::get().give(chunk_, n_); }
    hipError_t take(uint32_t want)
    {
        int device = 0;
        const hipError_t e = hipGetDevice(&device);
        if (e != hipSuccess) return e;
        n_ = Pool::get().take(device, std::min(want, kSlots), chunk_);
        return n_ ? hipSuccess : hipErrorOutOfMemory;
    }
    uint32_t size() const { return n_; }
    Chunk& operator[](uint32_t k) const { return *chunk_[k]; }
    void wait() const
    {
        for (uint32_t k = 0; k < n_; ++k) (void)hipStreamSynchronize(chunk_[k]->stream);
    }

private:
    Chunk* chunk_[kSlots] = {};
    uint32_t n_ = 0;
};

// Threads that calls have started besides their own, kMost in all calls: more only take turns on the
// processors (a GPU's share of its host's: 16) and on the link, which two reads fill.
class Helpers {
public:
    Helpers() = default;
    Helpers(const Helpers&) = delete;
    Helpers& operator=(const Helpers&) = delete;
    ~Helpers() { join(); }
    template <class F>
    void start(uint32_t n, F f)
    {
        for (n = std::min(n, kSlots); n_ < n;) {
            if (running().fetch_add(1) >= kMost) {
                running().fetch_sub(1);
                return;
            }
            try {
                thread_[n_] = std::thread(f, n_);
                ++n_;
            } catch (...) {  // no more threads: those that started and the caller's do the work
                running().fetch_sub(1);
                return;
            }
        }
    }
    void join()
    {
        for (; n_; --n_) {
            thread_[n_ - 1].join();
            running().fetch_sub(1);
        }
    }

private:
    static constexpr int kMost = 12;
    static std::atomic<int>& running()
    {
        static std::atomic<int> n{0};
        return n;
    }
    std::thread thread_[kSlots];
    uint32_t n_ = 0;
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
    constexpr uint64_t kPieces = kChunk / kPiece;
    const uint64_t chunks = (bytes + kChunk - 1) / kChunk, pieces = (bytes + kPiece - 1) / kPiece;
    Chunks st;
    hipError_t e = st.take(uint32_t(std::min<uint64_t>(chunks, kSlots)));
    if (e != hipSuccess) {
        if (own) (void)hipStreamSynchronize(own);
        return e;
    }
    std::atomic<uint64_t> next{0}, submitted{0}, copied{0};  // pieces claimed / submitted / copied
    std::atomic<uint32_t> slot_copied[kSlots] = {};           // pieces copied of the chunk in each slot
    std::atomic<int> error{int(hipSuccess)};
    // copies one submitted piece that nobody has claimed; false if there is none now
    auto copy_one = [&]() {
        uint64_t k = next.load();
        do {
            if (k >= submitted.load()) return false;
        } while (!next.compare_exchange_weak(k, k + 1));
        const uint32_t slot = uint32_t((k / kPieces) % st.size());
        const hipError_t w = hipEventSynchronize(st[slot].done);
        if (w != hipSuccess) {
            error = int(w);
            return false;
        }
        const size_t at = size_t(k) * kPiece;
        std::memcpy(static_cast<char*>(out) + at, st[slot].host + at % kChunk, std::min(kPiece, bytes - at));
        slot_copied[slot].fetch_add(1);
        copied.fetch_add(1);
        return true;
    };
    auto help = [&](uint32_t) {
        while (next.load() < pieces && error.load() == int(hipSuccess))
            if (!copy_one()) std::this_thread::yield();
    };
    Helpers helpers;
    const uint32_t want = uint32_t(std::min<size_t>(kHelpers, bytes / kPerThread));
    // the caller's thread submits chunks while slots are free and copies otherwise
    for (uint64_t k = 0; copied.load() < pieces && error.load() == int(hipSuccess);) {
        const uint32_t slot = uint32_t(k % st.size());
        if (k < chunks && (k < st.size() || slot_copied[slot].load() == kPieces)) {
            slot_copied[slot].store(0);
            const size_t at = size_t(k) * kChunk;
            const hipStream_t stream = own ? own : st[std::min(uint32_t(k & 1), st.size() - 1u)].stream;
            e = launch(stream, st[slot].host, at, std::min(kChunk, bytes - at));
            if (e == hipSuccess) e = hipEventRecord(st[slot].done, stream);
            if (e != hipSuccess) {
                error = int(e);
                break;
            }
            ++k;
            submitted.store(std::min(pieces, k * kPieces));
            if (k == std::min<uint64_t>(chunks, 2)) helpers.start(want, help);
        } else if (!copy_one()) {
            std::this_thread::yield();
        }
    }
    helpers.join();
    if (error.load() != int(hipSuccess)) {  // nothing writes the chunks any more
        st.wait();
        if (own) (void)hipStreamSynchronize(own);
    }
    return hipError_t(error.load());
}

// Calls work(chunk, first, count) for every range of at most `per` items of [0, n), by up to `threads` threads
// at once, each with a chunk of its own. `work` returns with nothing of its own in flight, unless it fails.
// Returns when all ranges are done, or on an error, when nothing is in flight.
template <class Work>
hipError_t run_chunks(size_t n, size_t per, uint32_t threads, Work work)
{
    Chunks st;
    const hipError_t e = st.take(threads);
    if (e != hipSuccess) return e;
    const int device = st[0].device;
    std::atomic<size_t> next{0};
    std::atomic<int> error{int(hipSuccess)};
    auto run = [&](uint32_t t) {
        for (size_t first; error.load() == int(hipSuccess) && (first = next.fetch_add(per)) < n;) {
            const hipError_t w = work(st[t], first, std::min(per, n - first));
            if (w != hipSuccess) error = int(w);
        }
    };
    Helpers helpers;
    helpers.start(st.size() - 1u, [&](uint32_t t) {
        (void)hipSetDevice(device);
        run(t + 1u);
    });
    run(0);
    helpers.join();
    if (error.load() != int(hipSuccess)) st.wait();  // nothing uses the chunks any more
    return hipError_t(error.load());
}

}  // namespace trb
