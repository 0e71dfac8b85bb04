// Bulk data between host arrays and the device through pinned slots.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <functional>

namespace dxg {

// Host threads and pinned slots of a transfer.  A host thread copies into fresh
// pages at 14 GB/s (2 MB pages; 4 GB/s with 4 KB pages); a kernel writes pinned
// memory at 54 GB/s and a copy engine moves pieces of 3 MB at 48 GB/s.  Reading
// the dose of 256x256x200 voxels (315 MB to the host): 13.5 ms with 5 threads,
// 10.0 with 8, 8.4 with 12, 7.9 with 16 (which would leave the caller's other
// threads no CPU of a 16-CPU job).
constexpr int kIoThreads = 12;
constexpr int kIoSlots = 16;
constexpr size_t kIoSlotBytes = size_t(3) << 20;

// The pinned slots come from at most kIoIdle idle sets kept for the next call
// (allocating and freeing one takes 0.4 ms); they are freed when the last one
// that holds them is gone: worlds, denoisers, and threads that called the
// segmentation or the dose table with host arrays.  Every transfer names the
// hold it runs under: without one, it would allocate and free a set.
constexpr int kIoIdle = 2;
struct IoHold {
    IoHold();
    ~IoHold();
    IoHold(const IoHold&) = delete;
    IoHold& operator=(const IoHold&) = delete;
};

// Runs a transfer in chunks: fill(i, slot) puts host data of chunk i into its
// slot, enqueue(i, slot) puts the device work on `stream` that uses the slot
// (slots are device-accessible), drain(i, slot) takes results into host arrays.
// Where pinned memory is refused the chunks pass one after another through 3 MB
// of device memory and of pageable memory instead.
// fill and drain run in several threads and may be empty; enqueue, like every
// call of the runtime, runs in the caller's thread, in order, with the stream's
// device as the current one.  Returns when every chunk is through; the first
// error ends it.
using IoEnqueue = std::function<hipError_t(size_t chunk, char* slot)>;
using IoHost = std::function<void(size_t chunk, char* slot)>;
hipError_t ioRun(const IoHold& hold, hipStream_t stream, size_t chunks, const IoHost& fill, const IoEnqueue& enqueue, const IoHost& drain);

// Copies `bytes` to or from device memory, complete on return.  Short ones, and
// any where pinned memory is refused, go straight to the runtime's own copy: starting the threads costs 0.2 ms.  Runtime
// / slots, us, medians of two processes: up 24 MB 685 / 1050, 32 MB 930-1060 /
// 1220-1310, 40 MB 1280-1580 / 1390-1510, 44 MB 1460-1780 / 1470-1730, 48 MB
// 1610-1970 / 1540-1690, 64 MB 2200-2540 / 1850-2040; down 1 MB into warm pages 67
// / 77 and fresh ones 240 / 170, 3 MB 205 / 217 and 745-820 / 360-425.
hipError_t ioUpload(const IoHold& hold, hipStream_t stream, void* dst, const void* src, size_t bytes);
hipError_t ioDownload(const IoHold& hold, hipStream_t stream, void* dst, const void* src, size_t bytes);
constexpr size_t kIoUploadLeast = size_t(44) << 20, kIoDownloadLeast = size_t(3) << 20;

// Items of a chunk: about two chunks a thread for a small transfer, at most what
// a slot holds; a multiple of `multiple`.
inline size_t ioChunk(size_t items, size_t item_bytes, size_t multiple)
{
    const size_t most = kIoSlotBytes / item_bytes / multiple * multiple;
    const size_t least = (kIoSlotBytes / 8) / item_bytes / multiple * multiple + multiple;
    const size_t share = (items + 2 * kIoThreads - 1) / (2 * kIoThreads);
    const size_t want = (share + multiple - 1) / multiple * multiple;
    return want < least ? least : (want > most ? most : want);
}

}  // namespace dxg
