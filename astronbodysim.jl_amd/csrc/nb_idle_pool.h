// nb_idle_pool.h -- objects of a device that wait for their next use.
#pragma once
#include <stdint.h>

#include <mutex>

namespace nb {

// At most PER_DEVICE idle objects of each device (B has `int dev` and `B *next`),
// while anyone holds the pool.  The bound is per device: one of four for the whole
// process left the fifth and later GPUs of a node to allocate and free 8 MiB of
// pinned memory for every download.
template <typename B, int PER_DEVICE>
class IdlePool {
public:
    // An idle object of the device, or nullptr.
    B *take(int dev) {
        std::lock_guard<std::mutex> lock(mutex_);
        for (B **p = &idle_; *p; p = &(*p)->next)
            if ((*p)->dev == dev) {
                B *b = *p;
                *p = b->next;
                return b;
            }
        return nullptr;
    }
    // Whether b stays here; if not, the caller frees it.
    bool give(B *b) {
        std::lock_guard<std::mutex> lock(mutex_);
        int same = 0;
        for (const B *p = idle_; p; p = p->next) same += p->dev == b->dev;
        if (held_ <= 0 || same >= PER_DEVICE) return false;
        b->next = idle_;
        idle_ = b;
        return true;
    }
    void hold() {
        std::lock_guard<std::mutex> lock(mutex_);
        ++held_;
    }
    // The idle objects for the caller to free (by next), once nobody holds the pool.
    B *release() {
        std::lock_guard<std::mutex> lock(mutex_);
        if (--held_ > 0) return nullptr;
        B *b = idle_;
        idle_ = nullptr;
        return b;
    }

private:
    std::mutex mutex_;
    B *idle_ = nullptr;
    int64_t held_ = 0;
};

}  // namespace nb
