// host_link.hpp -- large copies between ordinary host memory and the device,
// and device memory that is kept from one call to the next.
//
// The runtime copies pageable memory through its own pinned buffers with one
// host thread: 28 GB/s to the device and 17 GB/s back (10 into pages the
// process has not touched yet) on a link that carries 57.  Here a few threads
// share a copy, each moving chunks through its own pinned slot, so that one
// thread's memcpy (and its page faults) overlaps the others' transfers.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstring>
#include <stdexcept>
#include <string>
#include <thread>
#include <vector>

namespace lpa {

struct HostLinkError : std::runtime_error {
    using std::runtime_error::runtime_error;
};

// One per engine or model, used by one host thread at a time.  The slots (16
// MiB of pinned memory) cost about 2 ms to make, so the copies go to the
// runtime until WORTH bytes have been copied, and where the slots cannot be
// had; they are freed with the object.  The caller's side may be any memory that
// hipMemcpy takes: only ordinary pages go through the slots, since pinned
// memory is copied at the link's rate by the runtime and device memory is not
// a thread's to touch.
// 134 MB of labels to new host pages: 12.8 -> 3.6 ms; 33 MB of samples in and 13
// MB of results out: 2.3 -> 1.6 ms (from the second such call of a model on; the
// first takes 2.5 ms either way).
class HostLink {
  public:
    static constexpr size_t CHUNK = 2u << 20;
    static constexpr int SLOTS = 8;
    // below these the runtime's own copy is as fast (a thread takes 20 us to start)
    static constexpr size_t MIN_IN = 8u << 20, MIN_OUT = 4u << 20;
    static constexpr size_t WORTH = 64u << 20;

    HostLink() = default;
    HostLink(const HostLink &) = delete;
    HostLink &operator=(const HostLink &) = delete;
    ~HostLink() {
        for (hipEvent_t x : ev_)
            if (x) (void)hipEventDestroy(x);
        if (pinned_) (void)hipHostFree(pinned_);
    }

    // Queues the copy on stream s; src stays as it is until the stream has
    // been waited for.
    void in(void *dst, const void *src, size_t n, hipStream_t s) {
        if (n < MIN_IN || !ordinary(src) || !worth(n)) {
            if (n) check(hipMemcpyAsync(dst, src, n, hipMemcpyDefault, s));
            return;
        }
        run(n, [&](int slot, size_t at, size_t len) {
            // the slot's last transfer has read it
            hipError_t e = hipEventSynchronize(ev_[slot]);
            if (e != hipSuccess) return e;
            std::memcpy(pinned_ + slot * CHUNK, (const char *)src + at, len);
            e = hipMemcpyAsync((char *)dst + at, pinned_ + slot * CHUNK, len, hipMemcpyHostToDevice, s);
            return e == hipSuccess ? hipEventRecord(ev_[slot], s) : e;
        });
    }
    // Copies after the work queued on stream s; done on return.  Every piece
    // goes through put(dst, src, bytes) (a memcpy by default).
    template <class Put> void out(void *dst, const void *src, size_t n, hipStream_t s, Put &&put) {
        if (n < MIN_OUT || !ordinary(dst) || !worth(n)) {
            if (n) check(hipMemcpyAsync(dst, src, n, hipMemcpyDefault, s));
            check(hipStreamSynchronize(s));
            if (n) put(dst, dst, n);
            return;
        }
        run(n, [&](int slot, size_t at, size_t len) {
            char *p = pinned_ + slot * CHUNK;
            // a transfer to the device may still read the slot: same stream, so it is over first
            hipError_t e = hipMemcpyAsync(p, (const char *)src + at, len, hipMemcpyDeviceToHost, s);
            if (e == hipSuccess) e = hipEventRecord(ev_[slot], s);
            if (e == hipSuccess) e = hipEventSynchronize(ev_[slot]);
            if (e == hipSuccess) put((char *)dst + at, p, len);
            return e;
        });
    }
    void out(void *dst, const void *src, size_t n, hipStream_t s) {
        out(dst, src, n, s, [](void *d, const void *p, size_t len) {
            if (d != p) std::memcpy(d, p, len);
        });
    }

  private:
    char *pinned_ = nullptr;
    hipEvent_t ev_[SLOTS] = {};
    size_t copied_ = 0;

    // pages that the runtime knows nothing of
    static bool ordinary(const void *p) {
        hipPointerAttribute_t a{};
        if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
        (void)hipGetLastError();
        return true;
    }
    bool worth(size_t n) {
        copied_ = copied_ + n < copied_ ? copied_ : copied_ + n;
        return copied_ >= WORTH && prepare();
    }

    static void check(hipError_t e) {
        if (e != hipSuccess) throw HostLinkError(std::string("host copy: ") + hipGetErrorString(e));
    }
    bool prepare() {
        if (!pinned_ && hipHostMalloc((void **)&pinned_, SLOTS * CHUNK, hipHostMallocDefault) != hipSuccess) {
            pinned_ = nullptr;
            (void)hipGetLastError();
            return false;
        }
        for (hipEvent_t &x : ev_)
            if (!x && hipEventCreateWithFlags(&x, hipEventDisableTiming) != hipSuccess) {
                x = nullptr;
                (void)hipGetLastError();
                return false;
            }
        return true;
    }
    // piece(slot, at, len) for every chunk, slot w's chunks in order by thread
    // w (this one is thread 0).
    template <class Piece> void run(size_t n, Piece &&piece) {
        int device = 0;
        check(hipGetDevice(&device));
        const size_t chunks = (n + CHUNK - 1) / CHUNK;
        const int T = (int)(chunks / 2 < (size_t)SLOTS ? (chunks / 2 > 1 ? chunks / 2 : 1) : SLOTS);
        std::atomic<int> err{(int)hipSuccess};
        std::atomic<size_t> next{0};
        auto work = [&](int w) {
            hipError_t e = w ? hipSetDevice(device) : hipSuccess;
            while (e == hipSuccess && err.load(std::memory_order_relaxed) == (int)hipSuccess) {
                const size_t c = next.fetch_add(1);
                if (c >= chunks) return;
                e = piece(w, c * CHUNK, c + 1 < chunks ? CHUNK : n - c * CHUNK);
            }
            if (e != hipSuccess) err.store((int)e);
        };
        std::vector<std::thread> th;
        th.reserve(T);
        try {
            for (int w = 1; w < T; w++) th.emplace_back(work, w);
        } catch (...) {   // fewer threads will do
        }
        work(0);
        for (auto &x : th) x.join();
        check((hipError_t)err.load());
    }
};

}  // namespace lpa
