// wr_transfer.h -- large host <-> device transfers through a small ring of
// pinned buffers, for downloads emptied by several host threads.
//
// A hipMemcpy of pageable memory is one host thread's work: 50 MB into a fresh
// array measured 11.3 ms (4.4 GB/s: the thread also takes the array's page
// faults), while the link moves 55 GB/s and eight threads touch and copy a fresh
// 50 MB in 2.3 ms.  So a transfer is cut into chunks of 1 MB; chunk c uses ring
// slot c mod kSlots and host thread c mod threads, and because kSlots is a
// multiple of the thread count a slot belongs to one thread, which alone waits
// for its event, copies, and issues the slot's next chunk.  Downloads below
// kThreadedBytes run on the calling thread (starting the others costs about
// 100 us), and so do all uploads: their sources are written already, and one
// thread's copies keep up with the link's (records of a gradient, 4 MB, 310 us
// with the call, 650 with eight threads; 13.6 MB 620 and 710; scene of 41 MB 4.05
// and 4.35 ms).
//
// The ring (16 MB) belongs to a device handle, is allocated on its first
// transfer and freed with the handle; a mutex lets one transfer use it at a
// time, from any thread and stream.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <initializer_list>
#include <mutex>
#include <thread>
#include <vector>

namespace wr {

struct TransferRing {
    static constexpr int kSlots = 16, kThreads = 8;
    static constexpr size_t kChunk = size_t(1) << 20, kThreadedBytes = size_t(3) << 20;
    static constexpr size_t kPlainAbove = size_t(16) << 10, kPlainBelow = 1200000;
    static_assert(kSlots % kThreads == 0, "a slot belongs to one thread");
    static int threads_for(size_t bytes) { return bytes < kThreadedBytes ? 1 : kThreads; }

    std::mutex busy;
    char *pinned = nullptr;
    hipEvent_t done[kSlots] = {};  // the slot's device work

    TransferRing() = default;
    TransferRing(const TransferRing &) = delete;
    TransferRing &operator=(const TransferRing &) = delete;
    ~TransferRing() {
        for (hipEvent_t e : done)
            if (e) (void)hipEventDestroy(e);
        if (pinned) (void)hipHostFree(pinned);
    }

    // Device to host: issue(offset, bytes, slot) enqueues on `stream` the work
    // that leaves bytes [offset, offset + bytes) of the result in pinned memory.
    // Returns when dst is complete.
    template <class Issue>
    hipError_t download(int ordinal, hipStream_t stream, void *dst, size_t bytes, Issue &&issue) {
        char *out = static_cast<char *>(dst);
        return run(ordinal, stream, bytes, threads_for(bytes), true, issue,
                   [out](size_t off, size_t n, char *slot) { std::memcpy(out + off, slot, n); });
    }
    // The same for arrays in device memory, each to its own place on the host, in
    // one transfer: the host copies one array while the device copies the next.
    // Arrays above 16 KB and below 1.2 MB go by the runtime's own copy, which pins
    // the caller's pages there and needs no second copy (film reads, two arrays, of
    // 28^2 / 64^2 / 200^2 pixels 20 / 28 / 113 us, through the ring 29 / 36 / 109;
    // 24^2 28 and 19, 256^2 215 and 184).
    struct Out { void *dst; const void *src; size_t bytes; };
    hipError_t download(int ordinal, hipStream_t stream, std::initializer_list<Out> parts) {
        size_t total = 0, most = 0;
        for (const Out &p : parts) {
            total += p.bytes;
            most = std::max(most, p.bytes);
        }
        if (most > kPlainAbove && most < kPlainBelow) return plain(stream, parts);
        return run(
            ordinal, stream, total, threads_for(most), true,
            [&parts, stream](size_t off, size_t n, char *slot) {
                hipError_t e = hipSuccess;
                pieces(parts, off, n, slot, [&](const Out &p, size_t at, char *piece, size_t m) {
                    if (e == hipSuccess)
                        e = hipMemcpyAsync(piece, static_cast<const char *>(p.src) + at, m, hipMemcpyDeviceToHost, stream);
                });
                return e;
            },
            [&parts](size_t off, size_t n, char *slot) {
                pieces(parts, off, n, slot, [](const Out &p, size_t at, char *piece, size_t m) {
                    std::memcpy(static_cast<char *>(p.dst) + at, piece, m);
                });
            });
    }
    // By the runtime's own copies, without the ring.
    static hipError_t plain(hipStream_t stream, std::initializer_list<Out> parts) {
        hipError_t e = hipSuccess;
        for (const Out &p : parts)
            if (e == hipSuccess && p.bytes) e = hipMemcpyAsync(p.dst, p.src, p.bytes, hipMemcpyDeviceToHost, stream);
        const hipError_t w = hipStreamSynchronize(stream);
        return e != hipSuccess ? e : w;
    }
    // Host to device on `stream`: the parts, one behind the other.  The sources
    // may be reused when it returns, and the copies are complete.
    struct Part { const void *src; size_t bytes; };
    hipError_t upload(int ordinal, hipStream_t stream, void *device, std::initializer_list<Part> parts) {
        char *out = static_cast<char *>(device);
        size_t total = 0;
        for (const Part &p : parts) total += p.bytes;
        return run(
            ordinal, stream, total, 1, false,
            [out, stream](size_t off, size_t n, char *slot) {
                return hipMemcpyAsync(out + off, slot, n, hipMemcpyHostToDevice, stream);
            },
            [&parts](size_t off, size_t n, char *slot) {
                pieces(parts, off, n, slot, [](const Part &p, size_t at, char *piece, size_t m) {
                    std::memcpy(piece, static_cast<const char *>(p.src) + at, m);
                });
            });
    }
    // The ring for one caller, whose device work reads and writes pinned memory
    // itself: a chunk `in` and kSlots - 1 chunks `out`, until the lease is given back
    // or dies.  The caller waits for that work before (stage() has its own wait).
    static constexpr size_t kLeaseIn = kChunk, kLeaseOut = (kSlots - 1) * kChunk;
    struct Lease {
        std::unique_lock<std::mutex> lock;
        char *in = nullptr, *out = nullptr;
        hipEvent_t used = nullptr;      // behind the copies of stage(), on `stream`
        hipStream_t stream = nullptr;
        Lease() = default;
        Lease(const Lease &) = delete;
        Lease &operator=(const Lease &) = delete;
        ~Lease() { give(); }
        void give() {
            if (used && hipEventSynchronize(used) != hipSuccess) (void)hipStreamSynchronize(stream);
            used = nullptr;
            if (lock.owns_lock()) lock.unlock();
        }
    };
    hipError_t lease(Lease *l) {
        l->lock = std::unique_lock<std::mutex>(busy);
        return leased(l);
    }
    // The same if no other transfer has the ring; `in` stays null where one has.
    hipError_t try_lease(Lease *l) {
        l->lock = std::unique_lock<std::mutex>(busy, std::try_to_lock);
        return l->lock.owns_lock() ? leased(l) : hipSuccess;
    }
    // Host to device through a lease of the whole ring, for parts of up to
    // kLeaseAll bytes: enqueued on `stream` when it returns, and the sources may be
    // reused.  Giving the lease back waits for the copies.
    static constexpr size_t kLeaseAll = kSlots * kChunk;
    hipError_t stage(Lease *l, hipStream_t stream, void *device, std::initializer_list<Part> parts) {
        hipError_t e = lease(l);
        size_t total = 0;
        for (const Part &p : parts) total += p.bytes;
        for (size_t off = 0; off < total && e == hipSuccess; off += kChunk) {
            const size_t n = std::min(kChunk, total - off);
            pieces(parts, off, n, pinned + off, [](const Part &p, size_t at, char *piece, size_t m) {
                std::memcpy(piece, static_cast<const char *>(p.src) + at, m);
            });
            e = hipMemcpyAsync(static_cast<char *>(device) + off, pinned + off, n, hipMemcpyHostToDevice, stream);
        }
        if (e == hipSuccess && !done[0]) {
            e = hipEventCreateWithFlags(&done[0], hipEventDisableTiming);
            if (e != hipSuccess) done[0] = nullptr;
        }
        if (e == hipSuccess) e = hipEventRecord(done[0], stream);
        l->stream = stream;
        if (e == hipSuccess) l->used = done[0];
        else (void)hipStreamSynchronize(stream);
        return e;
    }
    // Host copies of the parts, by several threads from kThreadedBytes on.
    static void copy(std::initializer_list<Out> parts) {
        constexpr size_t kPiece = kChunk / 4;
        size_t total = 0;
        for (const Out &p : parts) total += p.bytes;
        const int threads = threads_for(total);
        on_threads(threads, [&](int t) {
            for (size_t off = size_t(t) * kPiece; off < total; off += size_t(threads) * kPiece)
                pieces(parts, off, std::min(kPiece, total - off), nullptr, [](const Out &p, size_t at, char *, size_t m) {
                    std::memcpy(static_cast<char *>(p.dst) + at, static_cast<const char *>(p.src) + at, m);
                });
        });
    }

private:
    hipError_t leased(Lease *l) {
        const hipError_t e = allocate();
        if (e != hipSuccess) return e;
        l->in = pinned;
        l->out = pinned + kLeaseIn;
        return hipSuccess;
    }
    // The ring's memory, on first use; `busy` is held.
    hipError_t allocate() {
        if (pinned) return hipSuccess;
        const hipError_t e = hipHostMalloc(reinterpret_cast<void **>(&pinned), kSlots * kChunk, hipHostMallocDefault);
        if (e != hipSuccess) pinned = nullptr;
        return e;
    }
    // work(0) ... work(threads - 1), on the calling thread and as many others as can be had.
    template <class Work>
    static void on_threads(int threads, Work &&work) {
        std::vector<std::thread> pool;
        int started = 1;
        try {
            pool.reserve(size_t(threads));
            for (; started < threads; started++) pool.emplace_back([&work, started] { work(started); });
        } catch (const std::exception &) {  // no thread to be had: the calling one does the rest
        }
        work(0);
        for (int t = started; t < threads; t++) work(t);
        for (std::thread &t : pool) t.join();
    }
    // Calls f(part, offset in the part, slot address, bytes) for the piece of each
    // part that lies in bytes [off, off + n) of all parts laid end to end.
    template <class P, class F>
    static void pieces(std::initializer_list<P> parts, size_t off, size_t n, char *slot, F &&f) {
        for (const P &p : parts) {
            const size_t m = off < p.bytes ? std::min(n, p.bytes - off) : 0;
            if (m) f(p, off, slot, m);
            if (slot) slot += m;
            n -= m;
            off = off < p.bytes ? 0 : off - p.bytes;
        }
    }
    // Per chunk, device(offset, bytes, slot) enqueues its device work and
    // host(offset, bytes, slot) does its host copy; `down`: device first.
    template <class Device, class Host>
    hipError_t run(int ordinal, hipStream_t stream, size_t bytes, int threads, bool down, Device &&device, Host &&host) {
        if (bytes == 0) return hipSuccess;
        std::lock_guard<std::mutex> lock(busy);
        if (const hipError_t e = allocate(); e != hipSuccess) return e;
        const size_t chunks = (bytes + kChunk - 1) / kChunk;
        for (size_t k = 0; k < std::min<size_t>(chunks, kSlots); k++)
            if (!done[k]) {
                hipError_t e = hipEventCreateWithFlags(&done[k], hipEventDisableTiming);
                if (e != hipSuccess) { done[k] = nullptr; return e; }
            }
        std::atomic<int> first_error{hipSuccess};
        auto note = [&](hipError_t e) {
            int none = hipSuccess;
            if (e != hipSuccess) first_error.compare_exchange_strong(none, e);
            return e == hipSuccess;
        };
        auto slot_of = [&](size_t c) { return pinned + (c % kSlots) * kChunk; };
        auto size_of = [&](size_t c) { return std::min(kChunk, bytes - c * kChunk); };
        auto issue = [&](size_t c) {
            return note(device(c * kChunk, size_of(c), slot_of(c))) && note(hipEventRecord(done[c % kSlots], stream));
        };
        auto wait = [&](size_t c) { return note(hipEventSynchronize(done[c % kSlots])); };
        // chunks t, t + threads, ...; every event the thread recorded is waited for
        // before it returns
        auto work = [&](int t) {
            if (!note(hipSetDevice(ordinal))) return;
            size_t issued = size_t(t), next = size_t(t);
            if (down) {
                for (; issued < chunks && issued < size_t(kSlots); issued += threads)
                    if (!issue(issued)) break;
                for (; next < issued; next += threads) {
                    if (!wait(next)) continue;
                    host(next * kChunk, size_of(next), slot_of(next));
                    if (issued < chunks && first_error == hipSuccess && issue(issued)) issued += threads;
                }
            } else {
                for (; issued < chunks && first_error == hipSuccess; issued += threads) {
                    if (issued >= size_t(kSlots)) {
                        if (!wait(next)) break;  // the slot may still be read
                        next += threads;
                    }
                    host(issued * kChunk, size_of(issued), slot_of(issued));
                    if (!issue(issued)) break;
                }
                for (; next < issued; next += threads) (void)wait(next);
            }
        };
        on_threads(threads, work);
        // after a failure there may be device work that no event stands for: nothing
        // may use the slots or the caller's memory once this returns
        if (first_error != hipSuccess) (void)hipStreamSynchronize(stream);
        return hipError_t(first_error.load());
    }
};

}  // namespace wr
