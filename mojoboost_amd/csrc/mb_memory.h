// The library's device memory: allocation, and the slabs that the calls on a
// dataset leave to one another; and the host memory of a fit's scores.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstdint>
#include <mutex>
#include <new>
#include <vector>

namespace mb {

// Device memory of the library's calls on a dataset. A call places its
// buffers in slabs (Arena) instead of allocating each one, and leaves the
// slabs to the dataset's next call: a training places some 100 buffers, and
// allocating and freeing them took 0.5 ms on a small table and 6 ms for ten
// classes on 300K x 50. Idle slabs belong to their dataset, are freed with
// it, total at most kIdleMost over the process, and are all freed when an
// allocation of the library's fails (device_malloc). Calls on one dataset at a
// time share nothing: a call takes every idle slab of its dataset, a second one
// beside it finds none.
struct Slab {
    uint8_t *p = nullptr;
    size_t size = 0;
    const void *owner = nullptr;
};

class SlabPool {
public:
    // no exception leaves these two: without host memory for the list, a call
    // starts with no slab, and a slab is freed instead of kept
    std::vector<Slab> take(const void *owner) noexcept {
        std::lock_guard<std::mutex> lock(mu_);
        std::vector<Slab> mine;
        try {
            mine.reserve(idle_.size());
        } catch (const std::bad_alloc &) {
            return mine;
        }
        size_t kept = 0;
        for (const Slab &s : idle_) {
            if (s.owner == owner) {
                mine.push_back(s);
                bytes_ -= s.size;
            } else {
                idle_[kept++] = s;
            }
        }
        idle_.resize(kept);
        return mine;
    }
    // the slabs must be idle on the device
    void give(std::vector<Slab> &slabs) noexcept {
        std::lock_guard<std::mutex> lock(mu_);
        bool room = true;
        try {
            idle_.reserve(idle_.size() + slabs.size());
        } catch (const std::bad_alloc &) {
            room = false;
        }
        for (const Slab &s : slabs) {
            if (room && s.owner && bytes_ + s.size <= kIdleMost) {
                idle_.push_back(s);
                bytes_ += s.size;
            } else {
                (void)hipFree(s.p);
            }
        }
        slabs.clear();
    }
    // frees an owner's idle slabs, or every one; the bytes freed
    size_t drop(const void *owner, bool all = false) {
        std::lock_guard<std::mutex> lock(mu_);
        size_t freed = 0;
        for (size_t i = idle_.size(); i-- > 0;)
            if (all || idle_[i].owner == owner) {
                (void)hipFree(idle_[i].p);
                freed += idle_[i].size;
                idle_.erase(idle_.begin() + (ptrdiff_t)i);
            }
        bytes_ -= freed;
        return freed;
    }

private:
    static constexpr size_t kIdleMost = (size_t)4 << 30;
    std::mutex mu_;
    std::vector<Slab> idle_;
    size_t bytes_ = 0;
};

// Never destroyed: the HIP runtime may be gone when static objects are.
inline SlabPool &slab_pool() {
    static SlabPool *pool = new SlabPool();
    return *pool;
}

// hipMalloc, a second time without the idle slabs where the first fails. Every
// device allocation of the library is made here.
inline hipError_t device_malloc(void **p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipSuccess) return e;
    (void)hipGetLastError();  // it is answered here, not at the next launch
    if (slab_pool().drop(nullptr, true) > 0) {
        e = hipMalloc(p, bytes);
        if (e != hipSuccess) (void)hipGetLastError();
    }
    return e;
}

// The buffers of one call, in the slabs its dataset's last call left and in
// new ones.
class Arena {
public:
    explicit Arena(const void *owner) : owner_(owner) {
        if (owner) slabs_ = slab_pool().take(owner);
    }
    Arena(const Arena &) = delete;
    Arena &operator=(const Arena &) = delete;
    ~Arena() {
        // as the frees did, wait for whatever still uses the buffers
        if (!slabs_.empty()) (void)hipDeviceSynchronize();
        slab_pool().give(slabs_);
    }
    hipError_t place(size_t bytes, void **at) noexcept {
        bytes = (std::max<size_t>(bytes, 1) + 255) & ~(size_t)255;
        try {
            slabs_.reserve(slabs_.size() + 1);
            used_.reserve(slabs_.size() + 1);
        } catch (const std::bad_alloc &) {
            return hipErrorOutOfMemory;
        }
        // first fit over the slabs' free ends
        used_.resize(slabs_.size(), 0);
        for (size_t i = 0; i < slabs_.size(); ++i)
            if (slabs_[i].size - used_[i] >= bytes) {
                *at = slabs_[i].p + used_[i];
                used_[i] += bytes;
                return hipSuccess;
            }
        Slab s;
        s.owner = owner_;
        // (without an owner nothing is kept, and 32 MB cost 30 us to allocate
        // and free)
        s.size = owner_ ? std::max(bytes, kSlab) : bytes;
        hipError_t e = device_malloc((void **)&s.p, s.size);
        if (e != hipSuccess && s.size > bytes) {
            s.size = bytes;
            e = device_malloc((void **)&s.p, s.size);
        }
        if (e != hipSuccess && free_unused()) {
            s.size = bytes;
            e = device_malloc((void **)&s.p, s.size);
        }
        if (e != hipSuccess) return e;
        slabs_.push_back(s);
        used_.push_back(bytes);
        *at = s.p;
        return hipSuccess;
    }

private:
    static constexpr size_t kSlab = (size_t)32 << 20;
    // the slabs taken over that hold nothing yet
    bool free_unused() {
        bool any = false;
        for (size_t i = slabs_.size(); i-- > 0;)
            if (used_[i] == 0) {
                (void)hipFree(slabs_[i].p);
                slabs_.erase(slabs_.begin() + (ptrdiff_t)i);
                used_.erase(used_.begin() + (ptrdiff_t)i);
                any = true;
            }
        return any;
    }
    const void *owner_;
    std::vector<Slab> slabs_;
    std::vector<size_t> used_;
};

// A fit's raw scores on the host: pinned from kPinBytes on (the copy from the
// device then runs at the link's rate, 84 MB in 1.6 ms against 5 into
// pageable memory after 14 of zeroing a vector), else ordinary memory,
// not zeroed first. The fits alive together pin at most kPinnedMost; scores
// past it are ordinary memory too.
class HostScores {
public:
    double *p = nullptr;
    size_t n = 0;
    void reserve(size_t count) {
        release();
        const size_t bytes = count * sizeof(double);
        if (bytes >= kPinBytes) {
            pinned_ = pinned_total().fetch_add(bytes) + bytes <= kPinnedMost &&
                      hipHostMalloc((void **)&p, bytes, hipHostMallocDefault) == hipSuccess;
            if (!pinned_) {
                (void)hipGetLastError();
                pinned_total() -= bytes;
                p = nullptr;
            }
        }
        if (!p) p = new double[count > 0 ? count : 1];
        n = count;
    }
    void release() {
        if (pinned_) {
            (void)hipHostFree(p);
            pinned_total() -= n * sizeof(double);
        } else {
            delete[] p;
        }
        p = nullptr;
        n = 0;
        pinned_ = false;
    }
    HostScores() = default;
    HostScores(const HostScores &) = delete;
    HostScores &operator=(const HostScores &) = delete;
    ~HostScores() { release(); }

private:
    static constexpr size_t kPinBytes = (size_t)1 << 20;
    static constexpr size_t kPinnedMost = (size_t)1 << 30;
    static std::atomic<size_t> &pinned_total() {
        static std::atomic<size_t> total{0};
        return total;
    }
    bool pinned_ = false;
};

}  // namespace mb
