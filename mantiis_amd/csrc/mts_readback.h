// Field readback: device arrays to the caller's (pageable) arrays.
//
// A plain copy to pageable memory is staged by the runtime on one thread,
// copy and page faults one after the other: 10.6 GB/s measured for the three
// fields of a 3000 x 2600 lattice (187 MB, 17.7 ms of a 112 ms call).  Here a
// few host threads each own one pinned slot, take the next chunk, bring it
// over on the handle's stream and move it to its destination while the other
// threads' chunks cross the bus.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>

#include "mts_threads.h"

namespace mts {

class Readback {
  public:
    struct Piece {
        void* dst;
        const void* src;
        size_t bytes;
    };
    static constexpr int MAX_PIECES = 3;
    static constexpr size_t SLOT = (size_t)1 << 20;  // bytes per thread: 8 MB pinned per handle (256 KB slots read at half the rate)
    // Bytes of a lattice's three fields from which they are read through slots:
    // a handle's 8 MB of pinned memory stay below a third of what it reads with
    // them.  It is not where the slots begin to pay once they are pinned, which
    // is at 4 MB (microseconds, plain / slots: 1.6 MB 115 / 140, 3.8 MB 282 / 271,
    // 6.3 MB 453 / 351, 12 MB 809 / 638, 24.0 MB 1709 / 1196, 25.2 MB 1766 / 1217,
    // 100 MB 9520 / 3778).
    static constexpr size_t MIN_BYTES = (size_t)24 << 20;

    // Pins the slots (a handle whose fields are large does so when it is made).
    bool ready() {
        if (pin_) return true;
        if (failed_) return false;
        slots_ = host_threads();
        if (hipHostMalloc((void**)&pin_, slots_ * SLOT, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            pin_ = nullptr;
            failed_ = true;
            return false;
        }
        for (int t = 0; t < slots_; t++)
            if (hipEventCreateWithFlags(&ev_[t], hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                ev_[t] = nullptr;
                release();
                failed_ = true;
                return false;
            }
        return true;
    }
    // Copies n pieces (device to host, at most MAX_PIECES) behind the work of
    // `stream` and returns when they are there.
    hipError_t run(int device, hipStream_t stream, const Piece* pieces, int n) noexcept {
        if (n > MAX_PIECES) return hipErrorInvalidValue;
        size_t total = 0, first[MAX_PIECES + 1] = {};  // chunks before piece i
        for (int i = 0; i < n; i++) {
            total += pieces[i].bytes;
            first[i + 1] = first[i] + (pieces[i].bytes + SLOT - 1) / SLOT;
        }
        if (total < MIN_BYTES || !ready()) {
            for (int i = 0; i < n; i++) {
                const hipError_t e = hipMemcpyAsync(pieces[i].dst, pieces[i].src, pieces[i].bytes, hipMemcpyDeviceToHost, stream);
                if (e != hipSuccess) return e;
            }
            return hipStreamSynchronize(stream);
        }
        auto at = [&](size_t c, size_t& i, size_t& off) -> size_t {
            i = std::upper_bound(first, first + n + 1, c) - first - 1;
            off = (c - first[i]) * SLOT;
            return std::min(SLOT, pieces[i].bytes - off);
        };
        return each(
            device, stream, first[n],
            [&](size_t c, char* slot) {
                size_t i, off;
                const size_t len = at(c, i, off);
                return hipMemcpyAsync(slot, (const char*)pieces[i].src + off, len, hipMemcpyDeviceToHost, stream);
            },
            [&](size_t c, const char* slot) {
                size_t i, off;
                const size_t len = at(c, i, off);
                std::memcpy((char*)pieces[i].dst + off, slot, len);
            });
    }
    // n chunks on the slots' threads (ready() must hold): fetch(i, slot) queues
    // the copies of chunk i into the slot on `stream`, take(i, slot) uses it
    // when they are done.
    template <class Fetch, class Take>
    hipError_t each(int device, hipStream_t stream, size_t n, Fetch fetch, Take take) {
        std::atomic<size_t> next{0};
        std::atomic<int> err{(int)hipSuccess};
        on_threads((int)std::min<size_t>(slots_, n), [&](int t) {
            hipError_t e = t ? hipSetDevice(device) : hipSuccess;  // the caller's thread keeps its current device
            char* slot = pin_ + (size_t)t * SLOT;
            for (size_t c; e == hipSuccess && (c = next.fetch_add(1)) < n;) {
                e = fetch(c, slot);
                if (e == hipSuccess) e = hipEventRecord(ev_[t], stream);
                if (e == hipSuccess) e = hipEventSynchronize(ev_[t]);
                if (e == hipSuccess) take(c, slot);
            }
            if (e != hipSuccess) err = (int)e;
        });
        if (err.load() != (int)hipSuccess) (void)hipStreamSynchronize(stream);  // no copy into a slot is left behind
        return (hipError_t)err.load();
    }
    void release() {
        for (hipEvent_t& e : ev_) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
        if (pin_) (void)hipHostFree(pin_);
        pin_ = nullptr;
    }
    ~Readback() { release(); }

  private:
    char* pin_ = nullptr;
    hipEvent_t ev_[MAX_HOST_THREADS] = {};
    int slots_ = 0;
    bool failed_ = false;
};

}  // namespace mts
