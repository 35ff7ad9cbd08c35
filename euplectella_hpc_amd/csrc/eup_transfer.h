// Arrays between the device and the caller's (pageable) host memory.
//
// Kernels write (read) pinned pieces directly over the bus, in the caller's element order, and up to
// four host threads copy each piece to (from) its place.  What bounds it is the host's side: one core copies
// 27 GB/s into warm and 14 GB/s into newly mapped memory, four 45 and 26, against the bus's 55; eight
// threads were slower than four.  84 MB to newly mapped memory, measured: the runtime's copy of
// pageable memory 8.0 ms in one call and 8.3 plane by plane, pinned pieces of 1 MB with one
// thread 6.3, with four 3.3.  To the device the bus is the limit (kernels read host memory at 36 GB/s, as
// fast as the runtime's copy): fewer threads, which take less time to start, keep it busy up to 32 MB.  us
// of the runtime's copy and with one, two and four threads: 3.1 MB 122, 111, 127, 123; 8.4 MB 262, 280,
// 245, 265; 17 MB 485, 545, 460, 480; 84 MB (19 populations) 3700, 3400, 2050, 2000.
#pragma once

#include <string.h>

#include <atomic>
#include <thread>

#include "eup_internal.h"

namespace eup {

constexpr int kMoveThreads = 4;               // host threads of a long transfer, the caller's among them
constexpr int kMoveSlots = 2 * kMoveThreads;  // pinned pieces: one in flight and one being copied per thread
constexpr int64_t kMovePiece = int64_t(1) << 20;

// the handle's pinned pieces, at least `bytes` of them, and the events that say when one is free
int transfer_ready(Handle *h, int64_t bytes);

// `bytes` between host memory and the device in pieces of whole `unit`s.  launch(offset, length,
// pinned) enqueues on the handle's stream the kernel that writes (In: reads) one piece; it is called
// from several threads, for disjoint pieces in no fixed order.  Returns when all is moved.
template <bool In, typename F>
int transfer(Handle *h, char *host, int64_t bytes, int64_t unit, F &&launch)
{
    const int64_t piece = bytes <= kMovePiece ? bytes : kMovePiece / unit * unit;
    const int64_t pieces = (bytes + piece - 1) / piece;
    const int most = !In || pieces >= 32 ? kMoveThreads : (pieces > 4 ? 2 : 1);
    const int threads = (int)(pieces < most ? pieces : most);
    const int64_t slot = (piece + 4095) / 4096 * 4096;
    int rc = transfer_ready(h, slot * (pieces < kMoveSlots ? pieces : kMoveSlots));
    if (rc) return rc;
    std::atomic<int> error{(int)hipSuccess};
    // pieces w, w + workers, ...: the slots of worker w are w and w + workers
    auto work = [&](int w, int workers) {
        hipError_t e = hipSetDevice(h->cfg.device);
        auto at = [&](int64_t it) { return (w + it * workers) * piece; };
        auto len = [&](int64_t it) { return bytes - at(it) < piece ? bytes - at(it) : piece; };
        auto index = [&](int64_t it) { return w + (int)(it & 1) * workers; };
        auto pinned = [&](int64_t it) { return h->pinned + index(it) * slot; };
        auto enqueue = [&](int64_t it) {
            launch(at(it), len(it), pinned(it));
            e = hipGetLastError();
            if (e == hipSuccess) e = hipEventRecord(h->moved[index(it)], h->stream);
        };
        const int64_t mine = (pieces - w + workers - 1) / workers;
        for (int64_t it = 0; it < (In ? 0 : 2) && it < mine && e == hipSuccess; ++it) enqueue(it);
        for (int64_t it = 0; it < mine && e == hipSuccess; ++it) {
            if (!In || it >= 2) e = hipEventSynchronize(h->moved[index(it)]);
            if (e != hipSuccess) break;
            if (In) {
                memcpy(pinned(it), host + at(it), (size_t)len(it));
                enqueue(it);
            } else {
                memcpy(host + at(it), pinned(it), (size_t)len(it));
                if (it + 2 < mine) enqueue(it + 2);
            }
        }
        if (e != hipSuccess) error = (int)e;
    };
    std::thread helper[kMoveThreads];
    int started = 1;
    if (threads > 1) {
        // a helper waits until it is known how many there are
        std::atomic<int> workers{0};
        try {
            for (; started < threads; ++started)
                helper[started] = std::thread([&work, &workers, w = started] {
                    while (workers.load(std::memory_order_acquire) == 0) std::this_thread::yield();
                    work(w, workers.load(std::memory_order_acquire));
                });
        } catch (...) { // no more threads (or memory for one) to be had: those that run do the work
        }
        workers.store(started, std::memory_order_release);
        work(0, started);
        for (int w = 1; w < started; ++w) helper[w].join();
    } else {
        work(0, 1);
    }
    // also after an error: no kernel may use a piece once this returns
    const hipError_t done = hipStreamSynchronize(h->stream);
    const hipError_t first = (hipError_t)error.load();
    return hip_check(h, first != hipSuccess ? first : done, "transfer") ? EUP_EHIP : 0;
}

} // namespace eup
