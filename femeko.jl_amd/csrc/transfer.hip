// Large results to the caller's memory.
//
// A copy to ordinary (pageable) memory is bound by the host: the runtime
// stages it with one thread, and that thread also takes the page faults of a
// result array the caller has just allocated. Here the transfer engine fills a
// ring of pinned chunks and several threads empty it, so that faults and copies
// overlap with one another and with the transfer.
#include <cstring>
#include <system_error>

#include "internal.h"

namespace fk {

// A chunk takes 20 to 40 us on the link (50 GB/s) against about 10 us for its
// event and wake-up; long copies take the larger ones. H of 1.5M elements
// (36 MB, a new array each time) 3.8 to 1.2 ms, |H| of 24.6M elements (197 MB)
// 19.6 to 6.0 ms; 4 threads 1.4 and 7.4 ms, 12 as 8; chunks of 256 KB 1.9 and
// 10.4 ms. Below kLinkMin the runtime's own staging is as fast or faster (74 KB
// 12 us against 20, 592 KB 57 us both ways); one thread does below kLinkMany.
constexpr int kThreads = 8, kSlots = 2 * kThreads;
constexpr size_t kChunk = 2 << 20, kPiece = 1 << 20, kLong = 16 << 20;
constexpr size_t kLinkMin = 512 << 10, kLinkMany = 2 << 20;

std::unique_ptr<HostLink> HostLink::make(int device) {
    try {
        std::unique_ptr<HostLink> l(new HostLink(device));
        l->ring.alloc(kSlots * kChunk);
        l->ev.reserve(kSlots);
        for (int i = 0; i < kSlots; ++i) {
            hipEvent_t e = nullptr;
            FK_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
            l->ev.push_back(e);
        }
        l->threads.reserve(kThreads);
        try {
            for (int t = 1; t < kThreads; ++t) l->threads.emplace_back([p = l.get(), t] { p->work(t); });
        } catch (const std::system_error &) {  // no more threads: those there are, the caller's at least
        }
        while (2 * l->most <= static_cast<int>(l->threads.size()) + 1) l->most *= 2;
        return l;
    } catch (...) {
        (void)hipGetLastError();
        return nullptr;
    }
}

HostLink::~HostLink() {
    {
        const std::lock_guard<std::mutex> l(mu);
        quit = true;
    }
    go.notify_all();
    for (std::thread &t : threads) t.join();
    for (hipEvent_t e : ev) (void)hipEventDestroy(e);
}

void HostLink::work(int t) {
    (void)hipSetDevice(device);
    uint64_t seen = 0;
    while (true) {
        {
            std::unique_lock<std::mutex> l(mu);
            go.wait(l, [&] { return quit || job != seen; });
            if (quit) return;
            seen = job;
        }
        if (t < takers) share(t);
        const std::lock_guard<std::mutex> l(mu);
        if (--left == 0) done.notify_one();
    }
}

hipError_t HostLink::issue(size_t c) {
    const size_t at = c * piece, len = std::min(piece, bytes - at);
    const int slot = static_cast<int>(c % kSlots);
    const hipError_t e = hipMemcpyAsync(ring.ptr + slot * kChunk, src + at, len, hipMemcpyDeviceToHost, stream);
    return e != hipSuccess ? e : hipEventRecord(ev[slot], stream);
}

// chunks t, t + takers, ...: each in the slot its index gives, which this
// thread alone empties and refills (takers divides kSlots)
void HostLink::share(int t) {
    for (size_t c = t; c * piece < bytes; c += takers) {
        const int slot = static_cast<int>(c % kSlots);
        hipError_t e = hipEventSynchronize(ev[slot]);
        if (e == hipSuccess) {
            std::memcpy(dst + c * piece, ring.ptr + slot * kChunk, std::min(piece, bytes - c * piece));
            if ((c + kSlots) * piece < bytes) e = issue(c + kSlots);
        }
        if (e != hipSuccess) {
            const std::lock_guard<std::mutex> l(mu);
            error = e;
            return;
        }
    }
}

void HostLink::copy(void *to, const void *from, size_t n, hipStream_t st) {
    const std::lock_guard<std::mutex> one(use);
    dst = static_cast<char *>(to);
    src = static_cast<const char *>(from);
    bytes = n;
    stream = st;
    error = hipSuccess;
    piece = n < kLong ? kPiece : kChunk;
    takers = n < kLinkMany ? 1 : most;
    for (int c = 0; c < kSlots && c * piece < n; ++c) FK_HIP(issue(c));
    if (takers > 1) {
        const std::lock_guard<std::mutex> l(mu);
        ++job;
        left = static_cast<int>(threads.size());
    }
    if (takers > 1) go.notify_all();
    share(0);
    std::unique_lock<std::mutex> l(mu);
    done.wait(l, [&] { return left == 0; });
    FK_HIP(error);
}

void copy_out(fk_context *ctx, void *to, const void *from, size_t bytes) {
    hipStream_t st = ctx->stream;
    if (bytes >= kLinkMin && !ctx->one_shot) {
        hipPointerAttribute_t a{};
        const hipError_t e = hipPointerGetAttributes(&a, to);
        if (e != hipSuccess) (void)hipGetLastError();
        if (e != hipSuccess || a.type == hipMemoryTypeUnregistered) {
            if (!ctx->link && !ctx->no_link) ctx->link = HostLink::make(ctx->device);
            ctx->no_link = !ctx->link;
            if (ctx->link) {
                ctx->link->copy(to, from, bytes, st);
                return;
            }
        }
    }
    FK_HIP(hipMemcpyAsync(to, from, bytes, hipMemcpyDeviceToHost, st));
    FK_HIP(hipStreamSynchronize(st));
}

}  // namespace fk
