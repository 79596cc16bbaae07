// Scratch that one call holds while it enqueues its launches: a buffer per
// (device, stream), leased under a lock, so that the launches of two host
// threads on one stream cannot interleave between the one that writes the
// buffer and the one that reads it (on one stream the order of the calls is
// then the order of the work). A buffer is never recorded into a graph: a
// caller takes no lease while its stream is captured. So an outgrown or evicted
// buffer has no reader but work already queued, and is given back at once:
// Alloc::release waits for the device before it frees (as hipFree does).
// Bounded: at most max_streams buffers, the least recently used one evicted for
// another stream, and max_bytes in all (sizes are powers of two); a call that
// finds no room gets an empty lease.
//
// Host-only and independent of HIP: the allocator is a template parameter, so
// the rules are exercised on the CPU (tests/cpp/lease_pool_test.cpp).
#pragma once

#include <cstddef>
#include <list>
#include <mutex>

namespace smg {

template <class Alloc>
class LeasePool {
    struct Entry {
        int device;
        const void *stream;
        void *buf = nullptr;
        size_t cap = 0;
        unsigned long long tick = 0;
        int users = 0;   // leases held or waited for (under mu_)
        std::mutex mu;   // held with the lease
    };

public:
    explicit LeasePool(size_t max_streams, size_t max_bytes, Alloc a = Alloc())
        : alloc_(a), max_streams_(max_streams), max_bytes_(max_bytes) {}
    ~LeasePool() {
        for (Entry &e : entries_)
            if (e.buf) alloc_.release(e.device, e.buf);
    }
    LeasePool(const LeasePool &) = delete;
    LeasePool &operator=(const LeasePool &) = delete;

    class Lease {
    public:
        Lease() = default;
        Lease(Lease &&o) : p_(o.p_), e_(o.e_) { o.p_ = nullptr; }
        Lease &operator=(Lease &&o) {
            if (this != &o) {
                drop();
                p_ = o.p_;
                e_ = o.e_;
                o.p_ = nullptr;
            }
            return *this;
        }
        ~Lease() { drop(); }
        void *buf() const { return p_ ? e_->buf : nullptr; }

    private:
        friend class LeasePool;
        Lease(LeasePool *p, Entry *e) : p_(p), e_(e) {}
        void drop() {
            if (!p_) return;
            e_->mu.unlock();
            std::lock_guard<std::mutex> lk(p_->mu_);
            e_->users--;
            p_ = nullptr;
        }
        LeasePool *p_ = nullptr;
        Entry *e_ = nullptr;
    };

    // A buffer of at least `bytes` for work on (device, stream), held until the
    // lease ends; an empty lease if there is no room or no memory for it.
    Lease take(int device, const void *stream, size_t bytes) {
        Entry *e = nullptr;
        {
            std::lock_guard<std::mutex> lk(mu_);
            for (Entry &x : entries_)
                if (x.device == device && x.stream == stream) e = &x;
            if (!e) {
                if (entries_.size() >= max_streams_ && !evict(nullptr)) return Lease();
                entries_.emplace_back();
                e = &entries_.back();
                e->device = device;
                e->stream = stream;
            }
            e->users++;
            e->tick = ++tick_;
        }
        e->mu.lock();
        Lease l(this, e);
        if (e->cap < bytes && !grow(*e, bytes)) return Lease();
        return l;
    }

    size_t bytes() const { std::lock_guard<std::mutex> lk(mu_); return bytes_; }
    size_t streams() const { std::lock_guard<std::mutex> lk(mu_); return entries_.size(); }

private:
    bool grow(Entry &e, size_t bytes) {
        size_t cap = (size_t)1 << 20;
        while (cap < bytes) cap <<= 1;
        std::lock_guard<std::mutex> lk(mu_);
        if (cap > max_bytes_) return false;
        while (bytes_ - e.cap + cap > max_bytes_)
            if (!evict(&e)) return false;
        if (e.buf) alloc_.release(e.device, e.buf);
        bytes_ -= e.cap;
        e.cap = 0;
        e.buf = alloc_.acquire(e.device, cap);
        if (!e.buf) return false;
        e.cap = cap;
        bytes_ += cap;
        return true;
    }
    // The least recently used entry that no call holds, given back (under mu_).
    bool evict(const Entry *keep) {
        auto at = entries_.end();
        for (auto i = entries_.begin(); i != entries_.end(); ++i)
            if (i->users == 0 && &*i != keep && (at == entries_.end() || i->tick < at->tick)) at = i;
        if (at == entries_.end()) return false;
        if (at->buf) alloc_.release(at->device, at->buf);
        bytes_ -= at->cap;
        entries_.erase(at);
        return true;
    }

    Alloc alloc_;
    const size_t max_streams_, max_bytes_;
    mutable std::mutex mu_;
    std::list<Entry> entries_;
    unsigned long long tick_ = 0;
    size_t bytes_ = 0;
};

}  // namespace smg
