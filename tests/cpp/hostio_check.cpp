// The pinned-slot transfers of opendxmc_amd/csrc/hostio.cpp on a small stand-in
// for the HIP runtime (below), which can refuse what a real one refuses only
// now and then.  Device work runs when it is enqueued; events are ready after a
// set time.
//
// usage: hostio_check <case>
#include "hostio.hpp"

#include <dlfcn.h>
#include <pthread.h>

#include <chrono>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <ctime>
#include <map>
#include <mutex>
#include <set>
#include <string>
#include <vector>

// ---------------------------------------------------------------- the runtime

struct ihipStream_t {
    int device;
};
struct ihipEvent_t {
    int device;
    std::chrono::steady_clock::time_point ready;
};

namespace {

using Clock = std::chrono::steady_clock;

bool g_refuse_pinned = false, g_refuse_threads = false;
int g_current_device = 0, g_pinned = 0;
hipError_t g_last_error = hipSuccess;
Clock::duration g_lag {};
std::map<const char*, std::size_t> g_device_memory;   // start, bytes

hipError_t failed(hipError_t e)
{
    g_last_error = e;
    return e;
}

bool onDevice(const void* p)
{
    const char* c = static_cast<const char*>(p);
    auto it = g_device_memory.upper_bound(c);
    return it != g_device_memory.begin() && c < std::prev(it)->first + std::prev(it)->second;
}

}  // namespace

extern "C" {

hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    if (g_refuse_pinned)
        return failed(hipErrorOutOfMemory);
    ++g_pinned;
    *p = std::malloc(n);
    return hipSuccess;
}
hipError_t hipHostFree(void* p)
{
    std::free(p);
    return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n)
{
    *p = std::malloc(n);
    g_device_memory[static_cast<const char*>(*p)] = n;
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    g_device_memory.erase(static_cast<const char*>(p));
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind kind, hipStream_t)
{
    const bool to = kind == hipMemcpyHostToDevice, from = kind == hipMemcpyDeviceToHost;
    if ((!to && !from) || onDevice(dst) != to || onDevice(src) != from)
        return failed(hipErrorInvalidMemcpyDirection);
    std::memcpy(dst, src, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t* d)
{
    *d = s->device;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d)
{
    *d = g_current_device;
    return hipSuccess;
}
hipError_t hipSetDevice(int d)
{
    g_current_device = d;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
    *e = new ihipEvent_t { g_current_device, {} };
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e)
{
    delete e;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    if (e->device != s->device)
        return failed(hipErrorInvalidHandle);
    e->ready = Clock::now() + g_lag;
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) { return Clock::now() >= e->ready ? hipSuccess : hipErrorNotReady; }
hipError_t hipGetLastError()
{
    const hipError_t e = g_last_error;
    g_last_error = hipSuccess;
    return e;
}
hipError_t hipPeekAtLastError() { return g_last_error; }

int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* x)
{
    static const auto real = reinterpret_cast<decltype(&pthread_create)>(dlsym(RTLD_NEXT, "pthread_create"));
    return g_refuse_threads ? EAGAIN : real(t, a, f, x);
}

}  // extern "C"

// ---------------------------------------------------------------- the checks

namespace {

#define CHECK(x)                                                             \
    do {                                                                     \
        if (!(x)) {                                                          \
            std::printf("line %d: %s\n", __LINE__, #x);                      \
            std::exit(1);                                                    \
        }                                                                    \
    } while (0)

ihipStream_t g_stream { 0 };

// A transfer of `chunks` chunks of `n` values, filled and / or drained, whose
// device work adds 1000 to each value.
void transfer(const dxg::IoHold& hold, std::size_t chunks, bool fill, bool drain)
{
    constexpr std::size_t n = 100;
    std::vector<std::uint32_t> on_device(chunks * n, 7), back(chunks * n, 0);
    std::vector<int> filled(chunks, 0), drained(chunks, 0);
    std::size_t next = 0;
    auto values = [](char* slot) { return reinterpret_cast<std::uint32_t*>(slot); };
    const dxg::IoHost filler = [&](std::size_t c, char* slot) {
        CHECK(!onDevice(slot));
        for (std::size_t i = 0; i < n; ++i)
            values(slot)[i] = static_cast<std::uint32_t>(c * n + i);
        ++filled[c];
    };
    const dxg::IoHost drainer = [&](std::size_t c, char* slot) {
        CHECK(!onDevice(slot));
        std::memcpy(&back[c * n], slot, n * sizeof(std::uint32_t));
        ++drained[c];
    };
    const hipError_t e = dxg::ioRun(
        hold, &g_stream, chunks, fill ? filler : dxg::IoHost(),
        [&](std::size_t c, char* slot) {
            CHECK(c == next++);
            for (std::size_t i = 0; i < n; ++i) {
                if (fill)
                    on_device[c * n + i] = values(slot)[i];
                values(slot)[i] = on_device[c * n + i] + 1000;
            }
            return hipSuccess;
        },
        drain ? drainer : dxg::IoHost());
    CHECK(e == hipSuccess);
    CHECK(next == chunks);
    for (std::size_t c = 0; c < chunks; ++c) {
        CHECK(filled[c] == (fill ? 1 : 0) && drained[c] == (drain ? 1 : 0));
        for (std::size_t i = c * n; i < (c + 1) * n; ++i) {
            CHECK(on_device[i] == (fill ? i : 7));
            CHECK(back[i] == (drain ? on_device[i] + 1000 : 0));
        }
    }
}

void copies(const dxg::IoHold& hold, std::size_t bytes)
{
    std::vector<unsigned char> from(bytes), to(bytes);
    for (std::size_t i = 0; i < bytes; ++i)
        from[i] = static_cast<unsigned char>(i % 251);
    void* d = nullptr;
    CHECK(hipMalloc(&d, bytes) == hipSuccess);
    CHECK(dxg::ioUpload(hold, &g_stream, d, from.data(), bytes) == hipSuccess);
    CHECK(dxg::ioDownload(hold, &g_stream, to.data(), d, bytes) == hipSuccess);
    CHECK(from == to);
    CHECK(hipFree(d) == hipSuccess);
}

// Every kind of transfer, around one chunk and around one round of the slots.
void everything()
{
    dxg::IoHold hold;
    for (std::size_t chunks : { 0, 1, 2, dxg::kIoSlots, dxg::kIoSlots + 1, 5 * dxg::kIoSlots + 3 })
        for (int k = 1; k < 4; ++k)
            transfer(hold, chunks, k & 1, k & 2);
    for (std::size_t bytes : { std::size_t(1), dxg::kIoDownloadLeast - 1, dxg::kIoDownloadLeast, dxg::kIoUploadLeast - 1,
                               dxg::kIoUploadLeast, dxg::kIoUploadLeast + 12345 })
        copies(hold, bytes);
}

}  // namespace

int main(int argc, char** argv)
{
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "plain") {
        everything();
        CHECK(g_pinned == 1);
    } else if (what == "pinned memory refused") {
        g_refuse_pinned = true;
        everything();
        CHECK(g_last_error == hipSuccess);   // the next launch check must not report it
        g_refuse_pinned = false;
        everything();
    } else if (what == "stream of another device") {
        everything();   // leaves a set with the events of device 0
        g_stream.device = 1;
        everything();
        CHECK(g_current_device == 0);
        g_current_device = 1;
        everything();
        CHECK(g_current_device == 1);
    } else if (what == "earlier error") {   // stays for the caller to find, as after the runtime's own calls
        g_last_error = hipErrorInvalidDevice;
        g_lag = std::chrono::milliseconds(1);
        dxg::IoHold hold;
        transfer(hold, 5, true, true);
        CHECK(g_last_error == hipErrorInvalidDevice);
    } else if (what == "waiting") {   // on device work of 0.4 s: at most the caller keeps a CPU busy
        g_lag = std::chrono::milliseconds(400);
        dxg::IoHold hold;
        const std::clock_t before = std::clock();   // CPU time of all threads
        transfer(hold, 2 * dxg::kIoThreads, false, true);
        const double busy = static_cast<double>(std::clock() - before) / CLOCKS_PER_SEC;
        std::printf("%.2f s of CPU time\n", busy);
        CHECK(busy < 1.2);   // two waits (16 slots): 0.8 s of the caller
    } else if (what == "threads refused") {
        g_refuse_threads = true;
        everything();
    } else {
        return 64;
    }
    CHECK(g_device_memory.empty());
    return 0;
}
