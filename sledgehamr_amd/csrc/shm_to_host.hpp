// Transfers to pageable host memory through rings of pinned slots: the pool
// of rings and the copying threads.  Host code without HIP, so it can be
// checked where there is no GPU.
#pragma once

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <utility>
#include <vector>

namespace shm {

constexpr size_t kIoSlot = 8u << 20;   // bytes a producer fills at a time
constexpr int kIoSlots = 4;
constexpr size_t kIoUnit = 2u << 20;   // bytes a thread copies at a time
constexpr size_t kIoKeep = 4;

/** Pinning 32 MB takes milliseconds, so a ring outlives the call and the
 *  context that first needed it: calls take one from the process's pool and
 *  give it back, the pool keeps at most kIoKeep, and the last context of the
 *  process to close frees them.  Ring: bytes, device, reset(). */
template <class Ring>
class IoPool {
  public:
    void enter() {
        std::lock_guard<std::mutex> lk(mu_);
        ++users_;
    }
    void leave() {
        std::lock_guard<std::mutex> lk(mu_);
        if (--users_ == 0) {
            for (Ring &r : free_) r.reset();
            free_.clear();
        }
    }
    /** A kept ring of that size and device, or make(bytes, device). */
    template <class Make>
    Ring take(size_t bytes, int device, Make &&make) {
        {
            std::lock_guard<std::mutex> lk(mu_);
            for (size_t i = 0; i < free_.size(); ++i)
                if (free_[i].bytes == bytes && free_[i].device == device) {
                    const Ring r = free_[i];
                    free_.erase(free_.begin() + i);
                    return r;
                }
        }
        return make(bytes, device);
    }
    void give(Ring r) {
        std::lock_guard<std::mutex> lk(mu_);
        if (users_ > 0 && free_.size() < kIoKeep)
            free_.push_back(r);
        else
            r.reset();
    }

  private:
    std::mutex mu_;
    std::vector<Ring> free_;
    int users_ = 0;
};

/** A user of a pool for as long as it lives: as a member it leaves the pool
 *  also when its owner's constructor throws. */
template <class Pool>
class PoolUser {
  public:
    explicit PoolUser(Pool &p) : p_(p) { p_.enter(); }
    ~PoolUser() { p_.leave(); }
    PoolUser(const PoolUser &) = delete;
    PoolUser &operator=(const PoolUser &) = delete;

  private:
    Pool &p_;
};

/** Moves nbytes through kIoSlots slots of kIoSlot bytes into out.
 *  produce(offset, bytes, slot) enqueues what writes those bytes into a slot,
 *  wait(slot) returns when they are there, start(f) starts a thread that runs
 *  f or throws std::system_error.
 *  Pageable copies by the HIP runtime run at the pace of one thread that
 *  copies out of its staging buffer and takes the page faults of a freshly
 *  allocated array: 9.8 GB/s into numpy memory (13.7 ms for a 256^3
 *  component).  Here (38 GB/s, 3.5 ms) several threads share both (units of
 *  2 MB of the destination, so two threads rarely fault on one large page),
 *  while the device fills the next slots. */
template <class Produce, class Wait, class Start>
void copy_through_slots(char *out, size_t nbytes, const char *slots, Produce &&produce,
                        Wait &&wait, Start &&start) {
    static_assert(kIoSlot % kIoUnit == 0, "slots hold whole units");
    const size_t nchunk = (nbytes + kIoSlot - 1) / kIoSlot;
    const size_t upc = kIoSlot / kIoUnit;  // units per chunk
    const size_t nunit = (nbytes + kIoUnit - 1) / kIoUnit;
    std::vector<std::atomic<int>> left(nchunk);  // units of a chunk not copied yet
    for (size_t c = 0; c < nchunk; ++c)
        left[c] = (int)(std::min(nunit, (c + 1) * upc) - c * upc);
    std::atomic<size_t> ready{0}, unit{0};
    std::atomic<bool> stop{false};
    auto copy_unit = [&](size_t u) {
        const size_t c = u / upc, o = u * kIoUnit, n = std::min(kIoUnit, nbytes - o);
        std::memcpy(out + o, slots + (c % kIoSlots) * kIoSlot + (o - c * kIoSlot), n);
        left[c].fetch_sub(1, std::memory_order_release);
    };
    auto work = [&] {
        for (size_t u = unit++; u < nunit; u = unit++) {
            while (ready.load(std::memory_order_acquire) <= u / upc) {
                if (stop) return;
                std::this_thread::yield();
            }
            copy_unit(u);
        }
    };
    const unsigned hc = std::max(1u, std::thread::hardware_concurrency());
    const size_t nthr = std::min<size_t>({8, hc, std::max<size_t>(1, nunit / 2)});
    std::vector<std::thread> thr;
    struct Join {
        std::vector<std::thread> &t;
        std::atomic<bool> &stop;
        ~Join() {
            stop = true;
            for (std::thread &x : t) x.join();
        }
    } join{thr, stop};
    size_t queued = 0;
    for (size_t c = 0; c < nchunk; ++c) {
        // Fill every free slot, then wait for chunk c.
        for (; queued < nchunk && queued < c + kIoSlots; ++queued) {
            if (queued >= kIoSlots) {
                const size_t old = queued - kIoSlots;
                if (left[old].load(std::memory_order_acquire) > 0 && queued > c) break;
                while (left[old].load(std::memory_order_acquire) > 0) std::this_thread::yield();
            }
            const size_t o = queued * kIoSlot;
            produce(o, std::min(kIoSlot, nbytes - o), (int)(queued % kIoSlots));
        }
        wait((int)(c % kIoSlots));
        // The threads poll for the next chunk, so they start when the first
        // one is there: before it the device may still run whole steps.
        if (c == 0) {
            thr.reserve(nthr);
            try {
                for (size_t i = 0; i < nthr; ++i) thr.push_back(start(work));
            } catch (const std::system_error &) {
                // As many as the system gives.
            }
        }
        ready.store(c + 1, std::memory_order_release);
        // None: the caller copies.
        if (thr.empty())
            for (size_t u = c * upc; u < std::min(nunit, (c + 1) * upc); ++u) copy_unit(u);
    }
    for (std::thread &x : thr) x.join();
    thr.clear();
}

}  // namespace shm
