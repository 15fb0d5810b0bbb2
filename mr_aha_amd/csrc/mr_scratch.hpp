// Lists behind the scratch blocks kept between calls (mr_hip.hpp), without the
// device: `Dev` supplies the three calls that touch it,
//   static int device();                       current device, or negative
//   static void *alloc(size_t bytes);          on the current device, or null
//   static void release(int dev, void *p);     back to device `dev`
// so the same lists run against a plain allocator on the host.
//
// A block belongs to one caller from get() to put(), so threads and streams
// never share one; only the list is guarded. put() allocates nothing and
// throws nothing: it runs in destructors.
#pragma once

#include <cstddef>
#include <mutex>
#include <new>
#include <vector>

template <class Dev> class mr_scratch {
public:
    // max_idle: bytes kept idle at most; max_age: requests after which an idle
    // block goes back to the device
    mr_scratch(size_t max_idle, unsigned long long max_age) : max_idle_(max_idle), max_age_(max_age) {}

    // A block of at least `bytes` (rounded up to megabytes, and up to an eighth
    // more) on the current device, or null.
    void *get(size_t bytes)
    {
        if (bytes == 0) bytes = 1;
        // whole megabytes above one, so that slightly different requests match
        if (bytes > (1u << 20)) bytes = (bytes + (1u << 20) - 1) & ~(size_t)((1u << 20) - 1);
        const int dev = Dev::device();
        if (dev < 0) return nullptr;
        {
            std::lock_guard<std::mutex> lk(mu_);
            ++tick_;
            drop([&](const block &b) { return tick_ - b.tick > max_age_; });
            block *best = nullptr;
            for (block &b : blocks_)
                if (b.idle && b.dev == dev && b.bytes >= bytes && b.bytes - bytes <= bytes / 8 &&
                    (!best || b.bytes < best->bytes))
                    best = &b;
            if (best) {
                best->idle = false;
                return best->p;
            }
        }
        void *p = Dev::alloc(bytes);
        if (!p && release_idle(dev) > 0) p = Dev::alloc(bytes);
        if (!p) return nullptr;
        std::lock_guard<std::mutex> lk(mu_);
        try {
            blocks_.push_back(block{p, bytes, dev, 0, false});
        } catch (const std::bad_alloc &) {
            Dev::release(dev, p);
            return nullptr;
        }
        return p;
    }

    // Hand a block back (null, and blocks that were forgotten, are ignored).
    void put(void *p)
    {
        if (!p) return;
        std::lock_guard<std::mutex> lk(mu_);
        for (block &b : blocks_)
            if (b.p == p && !b.idle) {
                b.idle = true;
                b.tick = tick_;
                b.seq = ++seq_;
                break;
            }
        // over the limit: the blocks idle longest go first
        size_t total = 0;
        for (const block &b : blocks_) total += b.idle ? b.bytes : 0;
        while (total > max_idle_) {
            const block *old = nullptr;
            for (const block &b : blocks_)
                if (b.idle && (!old || b.seq < old->seq)) old = &b;
            const void *q = old->p;
            total -= old->bytes;
            drop([&](const block &b) { return b.p == q; });
        }
    }

    // Give the idle blocks of `dev` back to it; the bytes given back.
    size_t release_idle(int dev)
    {
        std::lock_guard<std::mutex> lk(mu_);
        return drop([&](const block &b) { return b.dev == dev; });
    }

    size_t idle_bytes(int dev)
    {
        std::lock_guard<std::mutex> lk(mu_);
        size_t n = 0;
        for (const block &b : blocks_) n += (b.idle && b.dev == dev) ? b.bytes : 0;
        return n;
    }

    // Times the memory of `dev` was forgotten.
    unsigned epoch(int dev)
    {
        std::lock_guard<std::mutex> lk(mu_);
        return epoch_[slot(dev)];
    }

    // The memory of `dev` no longer exists (device reset): drop every block of
    // it, in use or idle, without touching the device. `since`: the epoch in
    // which the caller's memory was taken; a later one means that its loss is
    // known already and the blocks listed now are newer. True if it was not.
    bool forget(int dev, unsigned since)
    {
        std::lock_guard<std::mutex> lk(mu_);
        unsigned &e = epoch_[slot(dev)];
        if (e != since) return false;
        ++e;
        size_t n = 0;
        for (const block &b : blocks_)
            if (b.dev != dev) blocks_[n++] = b;
        blocks_.resize(n);
        return true;
    }

private:
    struct block {
        void *p = nullptr;
        size_t bytes = 0;
        int dev = -1;
        unsigned long long tick = 0;   // request count when it became idle
        bool idle = false;
        unsigned long long seq = 0;    // order in which blocks became idle
    };

    static int slot(int dev) { return dev & 63; }

    // Return the idle blocks picked by `gone` to their devices (lock held).
    template <class F> size_t drop(F gone)
    {
        size_t n = 0, bytes = 0;
        for (const block &b : blocks_) {
            if (b.idle && gone(b)) {
                Dev::release(b.dev, b.p);
                bytes += b.bytes;
            } else {
                blocks_[n++] = b;
            }
        }
        blocks_.resize(n);
        return bytes;
    }

    const size_t max_idle_;
    const unsigned long long max_age_;
    std::mutex mu_;
    std::vector<block> blocks_;
    unsigned epoch_[64] = {};
    unsigned long long tick_ = 0, seq_ = 0;
};
