// Pinned-slot transfers between host arrays and the device (hostio.hpp).
#include "hostio.hpp"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

namespace dxg {

namespace {

// Pinned slots and an event for each.
struct SlotSet {
    char* p = nullptr;
    hipEvent_t done[kIoSlots] = {};
    int device = -1;   // of the events

    hipError_t prepare(int dev)
    {
        if (!p)
            if (const hipError_t e = hipHostMalloc(reinterpret_cast<void**>(&p), kIoSlots * kIoSlotBytes, hipHostMallocPortable); e != hipSuccess)
                return e;
        if (device != dev) {
            dropEvents();
            for (hipEvent_t& ev : done)
                if (const hipError_t e = hipEventCreateWithFlags(&ev, hipEventDisableTiming); e != hipSuccess)
                    return e;
            device = dev;
        }
        return hipSuccess;
    }
    void dropEvents()
    {
        for (hipEvent_t& ev : done) {
            if (ev)
                (void)hipEventDestroy(ev);
            ev = nullptr;
        }
        device = -1;
    }
    ~SlotSet()
    {
        dropEvents();
        if (p)
            (void)hipHostFree(p);
    }
    char* slot(size_t chunk) const { return p + (chunk % kIoSlots) * kIoSlotBytes; }
    hipEvent_t event(size_t chunk) const { return done[chunk % kIoSlots]; }
};

struct Pool {
    std::mutex mu;
    SlotSet* idle[kIoIdle] = {};
    int owners = 0;
};

// Never destroyed: worlds may outlive static objects at the process's end.
Pool& pool()
{
    static Pool* p = new Pool;
    return *p;
}

// Makes a stream's device the current one for the length of a transfer: the
// events recorded on the stream have to be of its device, whatever device the
// calling thread is on.
struct StreamDevice {
    int device = 0, before = -1;   // before: to go back to, if another
    hipError_t status;
    explicit StreamDevice(hipStream_t stream)
        : status(hipGetDevice(&device))
    {
        int own = device;
        if (status == hipSuccess && stream)
            status = hipStreamGetDevice(stream, &own);
        if (status == hipSuccess && own != device && (status = hipSetDevice(own)) == hipSuccess) {
            before = device;
            device = own;
        }
    }
    ~StreamDevice()
    {
        if (before >= 0)
            (void)hipSetDevice(before);
    }
};

// A set for one call, from the pool or new, put back or freed at its end.
struct Lease {
    SlotSet* set = nullptr;
    Lease()
    {
        std::lock_guard<std::mutex> lock(pool().mu);
        for (SlotSet*& s : pool().idle)
            if (s && !set)
                std::swap(set, s);
    }
    ~Lease()
    {
        {
            std::lock_guard<std::mutex> lock(pool().mu);
            for (SlotSet*& s : pool().idle)
                if (!s && pool().owners > 0)
                    std::swap(set, s);
        }
        delete set;
    }
    // The set, or null where the system has no more pinned memory to give (the
    // refusal is cleared, so that no later check takes it for its own error).
    const SlotSet* prepare(const StreamDevice& at)
    {
        if (!set)
            set = new (std::nothrow) SlotSet;
        if (set && set->prepare(at.device) == hipSuccess)
            return set;
        (void)hipGetLastError();
        delete set;
        return set = nullptr;
    }
};

// A transfer without pinned slots: chunk after chunk through one piece of device
// memory and one of pageable memory.
hipError_t runUnpinned(hipStream_t stream, size_t chunks, const IoHost& fill, const IoEnqueue& enqueue, const IoHost& drain)
{
    struct DeviceSlot {
        void* p = nullptr;
        ~DeviceSlot()
        {
            if (p)
                (void)hipFree(p);
        }
    } slot;
    const std::unique_ptr<char[]> host(new (std::nothrow) char[kIoSlotBytes]());
    if (!host)
        return hipErrorOutOfMemory;
    hipError_t e = hipMalloc(&slot.p, kIoSlotBytes);
    for (size_t c = 0; c < chunks && e == hipSuccess; ++c) {
        if (fill) {
            fill(c, host.get());
            e = hipMemcpyAsync(slot.p, host.get(), kIoSlotBytes, hipMemcpyHostToDevice, stream);
        }
        if (e == hipSuccess)
            e = enqueue(c, static_cast<char*>(slot.p));
        if (e == hipSuccess && drain)
            e = hipMemcpyAsync(host.get(), slot.p, kIoSlotBytes, hipMemcpyDeviceToHost, stream);
        if (const hipError_t done = hipStreamSynchronize(stream); e == hipSuccess)
            e = done;
        if (e == hipSuccess && drain)
            drain(c, host.get());
    }
    return e;
}

// The calling thread enqueues chunks as their slots are ready and polls the
// oldest one's event; worker threads fill and drain, or the calling thread where
// none can be started.  With the runtime's calls spread over the workers instead,
// 16 MB to the device took 1.3 ms (0.9 now).
hipError_t run(const SlotSet& set, hipStream_t stream, size_t chunks, const IoHost& fill, const IoEnqueue& enqueue, const IoHost& drain)
{
    if (chunks == 1) {   // no thread is worth starting
        if (fill)
            fill(0, set.p);
        hipError_t e = enqueue(0, set.p);
        if (const hipError_t done = hipStreamSynchronize(stream); e == hipSuccess)
            e = done;
        if (e == hipSuccess && drain)
            drain(0, set.p);
        return e;
    }
    std::atomic<size_t> next { 0 };        // next chunk for a worker
    std::atomic<size_t> finished { 0 };    // chunks whose device work is done (in order)
    std::atomic<bool> stop { false };
    // of slot s: c + 1 once chunk c is filled or drained
    std::atomic<size_t> filled[kIoSlots] = {}, drained[kIoSlots] = {};
    auto at = [](size_t c) { return c % kIoSlots; };
    // chunk c's device work is done
    auto arrived = [&](size_t c) { return finished.load(std::memory_order_acquire) > c; };
    // the slot of chunk c is free: its former chunk is through
    auto vacant = [&](size_t c) {
        return c < kIoSlots || (drain ? drained[at(c)].load(std::memory_order_acquire) == c - kIoSlots + 1 : arrived(c - kIoSlots));
    };
    // A wait between chunks is short (3 MB take 57 us of the link); one for work
    // enqueued before, many layers of a network, say, must not keep every worker's
    // CPU busy.
    auto wait = [&](auto ready) {
        using Clock = std::chrono::steady_clock;
        Clock::time_point start;
        for (size_t spin = 0; !ready(); ++spin) {
            if (stop.load(std::memory_order_relaxed))
                return false;
            if (spin <= 64)
                continue;
            if (spin == 65)
                start = Clock::now();
            const Clock::duration waited = Clock::now() - start;
            if (waited < std::chrono::milliseconds(1))
                std::this_thread::yield();
            else
                std::this_thread::sleep_for(waited / 64);   // at most 1.6 % late
        }
        return true;
    };
    auto work = [&]() {
        for (size_t c; (c = next.fetch_add(1)) < chunks;) {
            if (fill) {
                if (!wait([&] { return vacant(c); }))
                    return;
                fill(c, set.slot(c));
                filled[at(c)].store(c + 1, std::memory_order_release);
            }
            if (drain) {
                if (!wait([&] { return arrived(c); }))
                    return;
                drain(c, set.slot(c));
                drained[at(c)].store(c + 1, std::memory_order_release);
            }
        }
    };
    size_t enqueued = 0;
    hipError_t status = hipSuccess;
    // enqueues what is ready and notes what is done; false when nothing moved
    auto advance = [&]() {
        bool moved = false;
        while (enqueued < chunks && status == hipSuccess) {
            const size_t c = enqueued;
            if (fill ? filled[at(c)].load(std::memory_order_acquire) != c + 1 : !vacant(c))
                break;
            status = enqueue(c, set.slot(c));
            if (status == hipSuccess)
                status = hipEventRecord(set.event(c), stream);
            ++enqueued;
            moved = true;
        }
        const size_t f = finished.load(std::memory_order_relaxed);
        if (f < enqueued && status == hipSuccess) {
            const hipError_t e = hipEventQuery(set.event(f));
            if (e == hipSuccess) {
                finished.store(f + 1, std::memory_order_release);
                moved = true;
            } else if (e != hipErrorNotReady) {   // not ready is not recorded as the last error
                status = e;
            }
        }
        return moved;
    };
    if (!fill)
        (void)advance();   // the device starts while the threads do
    const size_t cpus = std::max(2u, std::thread::hardware_concurrency());
    const size_t threads = fill || drain ? std::min({ chunks, cpus - 1, static_cast<size_t>(kIoThreads) }) : 0;
    std::vector<std::thread> workers;
    try {
        workers.reserve(threads);
        for (size_t k = 0; k < threads; ++k)
            workers.emplace_back(work);
    } catch (const std::exception&) {
        // fewer threads, or none
    }
    for (size_t c = 0; workers.empty() && c < chunks && status == hipSuccess; ++c) {   // the caller's part and theirs in turn
        if (fill) {
            fill(c, set.slot(c));
            filled[at(c)].store(c + 1, std::memory_order_release);
        }
        while (status == hipSuccess && !arrived(c))
            if (!advance())
                std::this_thread::yield();
        if (status == hipSuccess && drain) {
            drain(c, set.slot(c));
            drained[at(c)].store(c + 1, std::memory_order_release);
        }
    }
    while (status == hipSuccess && finished.load(std::memory_order_relaxed) < chunks)
        if (!advance())
            std::this_thread::yield();
    if (status != hipSuccess)
        stop.store(true);
    for (std::thread& t : workers)
        t.join();
    if (status != hipSuccess)
        (void)hipStreamSynchronize(stream);   // nothing may still use the slots
    return status;
}

hipError_t copyPageable(hipStream_t stream, void* dst, const void* src, size_t bytes, hipMemcpyKind kind)
{
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, kind, stream);
    return e == hipSuccess ? hipStreamSynchronize(stream) : e;
}

}  // namespace

hipError_t ioRun(const IoHold&, hipStream_t stream, size_t chunks, const IoHost& fill, const IoEnqueue& enqueue, const IoHost& drain)
{
    if (chunks == 0)
        return hipSuccess;
    const StreamDevice at(stream);
    if (at.status != hipSuccess)
        return at.status;
    Lease lease;
    const SlotSet* set = lease.prepare(at);
    return set ? run(*set, stream, chunks, fill, enqueue, drain) : runUnpinned(stream, chunks, fill, enqueue, drain);
}

IoHold::IoHold()
{
    std::lock_guard<std::mutex> lock(pool().mu);
    ++pool().owners;
}

IoHold::~IoHold()
{
    SlotSet* drop[kIoIdle] = {};
    {
        std::lock_guard<std::mutex> lock(pool().mu);
        if (--pool().owners == 0)
            std::swap(drop, pool().idle);
    }
    for (SlotSet* s : drop)
        delete s;
}

hipError_t ioUpload(const IoHold&, hipStream_t stream, void* dst, const void* src, size_t bytes)
{
    if (bytes >= kIoUploadLeast) {
        const StreamDevice at(stream);
        Lease lease;
        const size_t per = ioChunk(bytes, 1, 4096);
        auto size = [&](size_t i) { return std::min(per, bytes - i * per); };
        if (const SlotSet* set = at.status == hipSuccess ? lease.prepare(at) : nullptr)
            return run(
                *set, stream, (bytes + per - 1) / per,
                [&](size_t i, char* slot) { std::memcpy(slot, static_cast<const char*>(src) + i * per, size(i)); },
                [&](size_t i, char* slot) { return hipMemcpyAsync(static_cast<char*>(dst) + i * per, slot, size(i), hipMemcpyHostToDevice, stream); },
                nullptr);
    }
    return copyPageable(stream, dst, src, bytes, hipMemcpyHostToDevice);
}

hipError_t ioDownload(const IoHold&, hipStream_t stream, void* dst, const void* src, size_t bytes)
{
    if (bytes >= kIoDownloadLeast) {
        const StreamDevice at(stream);
        Lease lease;
        const size_t per = ioChunk(bytes, 1, 4096);
        auto size = [&](size_t i) { return std::min(per, bytes - i * per); };
        if (const SlotSet* set = at.status == hipSuccess ? lease.prepare(at) : nullptr)
            return run(
                *set, stream, (bytes + per - 1) / per, nullptr,
                [&](size_t i, char* slot) { return hipMemcpyAsync(slot, static_cast<const char*>(src) + i * per, size(i), hipMemcpyDeviceToHost, stream); },
                [&](size_t i, char* slot) { std::memcpy(static_cast<char*>(dst) + i * per, slot, size(i)); });
    }
    return copyPageable(stream, dst, src, bytes, hipMemcpyDeviceToHost);
}

}  // namespace dxg
