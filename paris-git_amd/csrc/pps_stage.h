// pps_stage.h -- a caller's pageable arrays to the device and back.
//
// The runtime copies pageable memory in one thread (A of a 128^3 grid, 134 MB:
// 4400 us, of which a plain memcpy takes 4300; p back, 18 MB: 1130 us), while
// the link takes 2350 us from pinned memory.  Here up to four threads each move
// chunks between the arrays and two pinned pieces of their own, one being
// filled while the other is on the link: A up 2800 us, the host solve at 128^3
// 9000 -> 6770 us.
#pragma once

#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>

#include "pps_internal.h"

namespace pps {

constexpr int kStageWorkers = 4;               // 2: 3000 us for that A, 4: 2800, 8: 3300
constexpr size_t kStageChunk = 2u << 20;
// Less in all goes by the runtime's own copy: starting the threads takes some
// 100 us, as long as 4 MB do.
constexpr size_t kStageMin = 8u << 20;
static_assert(2 * kStageWorkers == sizeof(StageRing::ev) / sizeof(hipEvent_t), "two pieces a worker");

struct Span {
    char *dev, *host;
    size_t n;
};

// memory that the runtime does not know (it copies pinned, managed and device
// memory directly)
inline bool pageable(const void *p) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return a.type == hipMemoryTypeUnregistered;
}

inline bool stage_ready(StageRing &r) {
    if (r.mem) return true;
    for (auto &e : r.ev)
        if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
            e = nullptr;
            (void)hipGetLastError();
            return false;
        }
    if (hipHostMalloc((void **)&r.mem, 2 * kStageWorkers * kStageChunk, 0) != hipSuccess) {
        r.mem = nullptr;
        (void)hipGetLastError();
        return false;
    }
    return true;
}

// The spans to the device (up) or back, in stream order on s.  Up, the arrays
// have been read when it returns; back, they have been written.
inline int stage_copy(pps_handle *h, const Span *sp, int count, bool up, hipStream_t s) {
    size_t tot = 0, chunks = 0;
    bool staged = true;
    for (int q = 0; q < count; ++q) {
        tot += sp[q].n;
        chunks += (sp[q].n + kStageChunk - 1) / kStageChunk;
        staged = staged && pageable(sp[q].host);
    }
    if (tot < kStageMin || !staged || !stage_ready(h->stage)) {
        for (int q = 0; q < count; ++q) {
            if (up) PPS_HIP(hipMemcpyAsync(sp[q].dev, sp[q].host, sp[q].n, hipMemcpyHostToDevice, s));
            else PPS_HIP(hipMemcpyAsync(sp[q].host, sp[q].dev, sp[q].n, hipMemcpyDeviceToHost, s));
        }
        if (!up) PPS_HIP(hipStreamSynchronize(s));
        return PPS_OK;
    }
    std::atomic<size_t> next{0};
    std::atomic<int> err{(int)hipSuccess};
    auto work = [&](int w) {
        auto good = [&](hipError_t e) {
            if (e != hipSuccess) err = (int)e;
            return e == hipSuccess;
        };
        if (!good(hipSetDevice(h->device))) return;
        Span last{nullptr, nullptr, 0};   // back: the chunk on its way
        for (int k = 0;; ++k) {
            const size_t c0 = next++;
            const int slot = 2 * w + (k & 1);
            char *piece = h->stage.mem + slot * kStageChunk;
            Span ch{nullptr, nullptr, 0};
            if (c0 < chunks && err == (int)hipSuccess) {
                size_t c = c0;
                int q = 0;
                for (;; ++q) {
                    const size_t m = (sp[q].n + kStageChunk - 1) / kStageChunk;
                    if (c < m) break;
                    c -= m;
                }
                const size_t o = c * kStageChunk;
                ch = Span{sp[q].dev + o, sp[q].host + o, std::min(kStageChunk, sp[q].n - o)};
            }
            if (up) {
                if (!ch.n || !good(hipEventSynchronize(h->stage.ev[slot]))) return;   // the piece is free
                std::memcpy(piece, ch.host, ch.n);
                if (!good(hipMemcpyAsync(ch.dev, piece, ch.n, hipMemcpyHostToDevice, s)) ||
                    !good(hipEventRecord(h->stage.ev[slot], s)))
                    return;
            } else {
                // (the piece's earlier use is over: its chunk was waited for,
                // or went up earlier on this stream)
                if (ch.n && (!good(hipMemcpyAsync(piece, ch.dev, ch.n, hipMemcpyDeviceToHost, s)) ||
                             !good(hipEventRecord(h->stage.ev[slot], s))))
                    return;
                if (last.n) {
                    if (!good(hipEventSynchronize(h->stage.ev[slot ^ 1]))) return;
                    std::memcpy(last.host, h->stage.mem + (slot ^ 1) * kStageChunk, last.n);
                }
                if (!ch.n) return;
                last = ch;
            }
        }
    };
    std::thread th[kStageWorkers];
    const int workers = (int)std::min<size_t>(
        {(size_t)kStageWorkers, chunks, (size_t)std::max(1u, std::thread::hardware_concurrency())});
    for (int w = 1; w < workers; ++w) {
        try {
            th[w] = std::thread(work, w);
        } catch (...) {   // no more threads: those there are take all chunks
            break;
        }
    }
    work(0);
    for (auto &t : th)
        if (t.joinable()) t.join();
    PPS_HIP((hipError_t)err.load());
    return PPS_OK;
}

}  // namespace pps
