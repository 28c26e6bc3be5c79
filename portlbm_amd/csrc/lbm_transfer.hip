// The runtime copies to pageable memory through its own staging in one thread:
// 2.5 GB/s for arrays up to 1 MB, 19 GB/s above, and 4 GB/s whenever the
// destination's pages are new, as a caller's fresh result arrays are (the page
// faults; 64 MB: 17 ms).  Here the device writes a ring of pinned slots and,
// for large results, several threads copy from it, faults included (64 MB with
// 8 threads: 3.3 ms).
#include "lbm_transfer.hpp"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

namespace lbm_dev
{
namespace
{

constexpr size_t kSlotBytes = size_t(1) << 20;
constexpr size_t kSlots = 16;
constexpr size_t kBytesPerThread = size_t(3) << 20;  // a thread costs 16 us to start: about 0.1 ms of copying
constexpr size_t kMaxThreads = 8;

// One ring for the process, made by the first call that uses it and used by one
// at a time; a call that finds it taken copies through the runtime.  It stays: a
// program that creates, runs, reads and destroys one lattice after another took
// 250 us per 64 x 32 lattice and 5.1 ms per 2048 x 512 one with a ring given
// back with the last object, 205 us and 3.2 ms so.
struct Ring
{
    std::mutex use;
    int device = -1;  // whose events these are
    char *slots = nullptr;
    hipEvent_t ready[kSlots] = {};

    hipError_t create()
    {
        int dev = 0;
        if (hipError_t err = hipGetDevice(&dev))
            return err;
        if (slots)
            return dev == device ? hipSuccess : hipErrorInvalidDevice;
        device = dev;
        for (hipEvent_t &e : ready)
            if (hipError_t err = hipEventCreateWithFlags(&e, hipEventDisableTiming))
            {
                e = nullptr;
                drop_events();
                return err;
            }
        if (hipError_t err = hipHostMalloc(reinterpret_cast<void **>(&slots), kSlots * kSlotBytes,
                                           hipHostMallocPortable))
        {
            slots = nullptr;
            drop_events();
            return err;
        }
        return hipSuccess;
    }
    void drop_events()
    {
        for (hipEvent_t &e : ready)
        {
            if (e)
                (void)hipEventDestroy(e);
            e = nullptr;
        }
    }
};

Ring &ring()
{
    static Ring *r = new Ring;  // never destroyed: objects may outlive static destruction
    return *r;
}

struct Chunk
{
    const char *src;
    size_t bytes;
    size_t at;  // first byte in the pieces laid end to end
};

// `bytes` bytes at `from` to the pieces, from byte `at` of them on.
void scatter(const HostPiece *pieces, size_t count, size_t at, const char *from, size_t bytes)
{
    for (size_t p = 0; p < count && bytes; ++p)
    {
        if (at >= pieces[p].bytes)
        {
            at -= pieces[p].bytes;
            continue;
        }
        const size_t n = std::min(bytes, pieces[p].bytes - at);
        std::memcpy(static_cast<char *>(pieces[p].dst) + at, from, n);
        from += n;
        bytes -= n;
        at = 0;
    }
}

hipError_t through_runtime(const HostPiece *pieces, size_t count, hipStream_t stream)
{
    for (size_t p = 0; p < count; ++p)
        if (pieces[p].bytes)
            if (hipError_t e = hipMemcpyAsync(pieces[p].dst, pieces[p].src, pieces[p].bytes, hipMemcpyDeviceToHost,
                                              stream))
                return e;
    return hipStreamSynchronize(stream);
}

}  // namespace

hipError_t download(const HostPiece *pieces, size_t count, hipStream_t stream)
{
    Ring &r = ring();
    std::unique_lock<std::mutex> lock(r.use, std::try_to_lock);
    if (!lock.owns_lock())
        return through_runtime(pieces, count, stream);
    if (r.create() != hipSuccess)
    {
        (void)hipGetLastError();
        return through_runtime(pieces, count, stream);
    }
    // chunks of at most a slot, over pieces that adjoin on the device
    std::vector<Chunk> chunks;
    size_t total = 0;
    try
    {
        size_t bytes = 0;
        for (size_t p = 0; p < count; ++p)
            bytes += pieces[p].bytes;
        chunks.reserve(bytes / kSlotBytes + count + 1);
    }
    catch (const std::bad_alloc &)
    {
        return through_runtime(pieces, count, stream);
    }
    for (size_t p = 0; p < count; ++p)
    {
        const char *src = static_cast<const char *>(pieces[p].src);
        for (size_t done = 0; done < pieces[p].bytes;)
        {
            if (chunks.empty() || chunks.back().bytes == kSlotBytes || chunks.back().src + chunks.back().bytes != src + done)
                chunks.push_back(Chunk{src + done, 0, total});
            const size_t n = std::min(kSlotBytes - chunks.back().bytes, pieces[p].bytes - done);
            chunks.back().bytes += n;
            done += n;
            total += n;
        }
    }
    const size_t nc = chunks.size();
    std::atomic<size_t> issued{0}, next{0};
    std::atomic<int> error{hipSuccess};
    const std::unique_ptr<std::atomic<bool>[]> emptied(new (std::nothrow) std::atomic<bool>[nc]);
    if (!emptied)
        return through_runtime(pieces, count, stream);
    for (size_t i = 0; i < nc; ++i)
        emptied[i].store(false, std::memory_order_relaxed);
    // takes the next chunk below `limit`, if there is one: waits for it to
    // arrive, copies it, frees its slot
    auto drain_one = [&](size_t limit) -> bool {
        size_t i = next.load();
        do
        {
            if (i >= limit || error.load())
                return false;
        } while (!next.compare_exchange_weak(i, i + 1));
        while (issued.load(std::memory_order_acquire) <= i)
        {
            if (error.load())
                return false;
            std::this_thread::yield();
        }
        if (hipError_t e = hipEventSynchronize(r.ready[i % kSlots]))
        {
            error.store(e);
            return false;
        }
        scatter(pieces, count, chunks[i].at, r.slots + (i % kSlots) * kSlotBytes, chunks[i].bytes);
        emptied[i].store(true, std::memory_order_release);
        return true;
    };
    std::vector<std::thread> threads;
    const size_t want = std::min({kMaxThreads, total / kBytesPerThread, size_t(std::thread::hardware_concurrency())});
    try
    {
        for (size_t t = 1; t < want; ++t)
            threads.emplace_back([&] {
                while (drain_one(nc))
                {
                }
            });
    }
    catch (...)
    {
        // fewer threads than wanted
    }
    for (size_t i = 0; i < nc && !error.load(); ++i)
    {
        if (i >= kSlots)
        {
            // the chunk before it in its slot: this thread drains too (what has
            // been issued) while it waits
            while (!emptied[i - kSlots].load(std::memory_order_acquire) && !error.load())
                if (!drain_one(i))
                    std::this_thread::yield();
        }
        char *slot = r.slots + (i % kSlots) * kSlotBytes;
        hipError_t e = hipMemcpyAsync(slot, chunks[i].src, chunks[i].bytes, hipMemcpyDeviceToHost, stream);
        if (e == hipSuccess)
            e = hipEventRecord(r.ready[i % kSlots], stream);
        if (e != hipSuccess)
            error.store(e);
        else
            issued.store(i + 1, std::memory_order_release);
    }
    while (drain_one(nc))
    {
    }
    for (std::thread &t : threads)
        t.join();
    const hipError_t e = hipError_t(error.load());
    const hipError_t s = hipStreamSynchronize(stream);
    return e != hipSuccess ? e : s;
}

}  // namespace lbm_dev
