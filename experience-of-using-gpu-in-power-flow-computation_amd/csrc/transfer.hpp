// Copies between a caller's ordinary memory and the GPU through pinned slots.
//
// hipMemcpy on pageable memory moves some 18 GB/s (15 MB of results, touched
// pages: 850 us) and costs 15 us however little it moves.  Here the GPU's
// copies run ahead, a slot each, while the host empties or fills the others:
// the same results take 350 us, and pieces that fit a slot share one wait.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <mutex>
#include <vector>

namespace pf {

struct CopyPiece {
    void *host;
    void *dev;
    size_t bytes;
};

// A plan's small arrays, packed on the host and copied at once, after which
// their pointers are set: an allocation and a copy each took some 15 us, 70 of
// them half the 2.3 ms of a 118-bus case from file to report.  From 64 KB on
// the packing costs as much.
class PackedUploads {
public:
    template <typename T>
    static bool small(const std::vector<T> &v) {
        return sizeof(T) * v.size() < 65536;
    }
    template <typename T>
    void add(T **p, const std::vector<T> &v) {
        at_.push_back({(void **)p, bytes_.size()});
        const char *b = (const char *)v.data();
        bytes_.insert(bytes_.end(), b, b + sizeof(T) * v.size());
        bytes_.resize((bytes_.size() + 255) / 256 * 256);
    }
    size_t bytes() const { return bytes_.size(); }
    // d: bytes() of device memory
    hipError_t copy_to(char *d) {
        const hipError_t e = bytes_.empty() ? hipSuccess
                                            : hipMemcpy(d, bytes_.data(), bytes_.size(), hipMemcpyHostToDevice);
        for (const At &a : at_) *a.p = d + a.off;
        at_.clear();
        std::vector<char>().swap(bytes_);
        return e;
    }

private:
    struct At {
        void **p;
        size_t off;
    };
    std::vector<At> at_;
    std::vector<char> bytes_;
};

// One object's slots, allocated by reserve or the first copy.  Calls take
// turns; each returns when the caller's memory is read (send) or written (fetch).
class PinnedSlots {
public:
    PinnedSlots() = default;
    PinnedSlots(const PinnedSlots &) = delete;
    PinnedSlots &operator=(const PinnedSlots &) = delete;
    ~PinnedSlots() {   // a failed copy may have left some under way
        for (int i = 0; i < kSlots; i++)
            if (ev_[i]) {
                (void)hipEventSynchronize(ev_[i]);
                (void)hipEventDestroy(ev_[i]);
            }
        if (mem_) (void)hipHostFree(mem_);
    }

    hipError_t reserve() {
        std::lock_guard<std::mutex> lk(mu_);
        return ready();
    }
    // device to host, after the stream's earlier work
    hipError_t fetch(const CopyPiece *pieces, int n, hipStream_t st) noexcept { return caught(pieces, n, st, false); }
    // host to device, before the stream's later work
    hipError_t send(const CopyPiece *pieces, int n, hipStream_t st) noexcept { return caught(pieces, n, st, true); }

private:
    static constexpr int kSlots = 4;
    static constexpr size_t kBytes = 1u << 20;
    char *mem_ = nullptr;
    hipEvent_t ev_[kSlots] = {};
    std::mutex mu_;

    struct Part {
        char *host;
        size_t off, bytes;
    };

    hipError_t ready() {
        hipError_t e = hipSuccess;
        if (!mem_) e = hipHostMalloc((void **)&mem_, kSlots * kBytes, hipHostMallocDefault);
        for (int i = 0; i < kSlots && e == hipSuccess; i++)
            if (!ev_[i]) e = hipEventCreateWithFlags(&ev_[i], hipEventDisableTiming);
        return e;
    }

    hipError_t caught(const CopyPiece *pieces, int n, hipStream_t st, bool send) noexcept {
        try {
            return run(pieces, n, st, send);
        } catch (...) {   // no memory for the list of parts
            (void)hipStreamSynchronize(st);
            return hipErrorOutOfMemory;
        }
    }

    hipError_t run(const CopyPiece *pieces, int np, hipStream_t st, bool send) {
        std::lock_guard<std::mutex> lk(mu_);
        hipError_t e = np ? ready() : hipStreamSynchronize(st);
        std::vector<Part> parts[kSlots];   // what each slot under way holds for the caller
        size_t k = 0, used = 0;            // the slot being filled, its bytes
        // the slot is free again; what it held is the caller's
        auto take_back = [&](size_t s) {
            e = hipEventSynchronize(ev_[s]);
            if (e == hipSuccess && !send)
                for (const Part &p : parts[s]) std::memcpy(p.host, mem_ + s * kBytes + p.off, p.bytes);
            parts[s].clear();
        };
        auto next_slot = [&]() {
            e = hipEventRecord(ev_[k % kSlots], st);
            k++;
            used = 0;
            if (e == hipSuccess && k >= kSlots) take_back(k % kSlots);
        };
        for (int i = 0; i < np && e == hipSuccess; i++) {
            char *h = (char *)pieces[i].host, *d = (char *)pieces[i].dev;
            for (size_t left = pieces[i].bytes; left > 0 && e == hipSuccess;) {
                if (used >= kBytes) {
                    next_slot();
                    if (e != hipSuccess) break;
                }
                const size_t s = k % kSlots, n = std::min(left, kBytes - used);
                char *slot = mem_ + s * kBytes + used;
                if (send) std::memcpy(slot, h, n);
                e = send ? hipMemcpyAsync(d, slot, n, hipMemcpyHostToDevice, st)
                         : hipMemcpyAsync(slot, d, n, hipMemcpyDeviceToHost, st);
                parts[s].push_back({h, used, n});
                used = std::min(kBytes, used + ((n + 255) & ~(size_t)255));
                h += n;
                d += n;
                left -= n;
            }
        }
        if (e == hipSuccess && used > 0) next_slot();
        // the slots still under way, oldest first (a later call fills them anew)
        for (size_t s = k >= kSlots ? k - kSlots + 1 : 0; s < k && e == hipSuccess; s++) take_back(s % kSlots);
        if (e != hipSuccess && mem_) (void)hipStreamSynchronize(st);   // nothing writes to the slots any more
        return e;
    }
};

}  // namespace pf
