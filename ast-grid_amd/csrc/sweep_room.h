// Room for sweeps whose workgroups wait for each other.
//
// A tile of the tiled sweeps waits for values of other tiles, so all tiles of a
// launch have to be resident together: one compute unit each. One launch always
// has room, but two solves at once (contexts of two threads, each on its own
// stream) can be given half the device each, and then neither goes on until its
// waits end after 3 s. A solve therefore enters with the compute units that its
// sweeps rely on and waits, in the order of arrival, while those of the solves
// inside leave too few; solves that fit side by side run side by side.
#pragma once

#include <condition_variable>
#include <mutex>

namespace astg {

class SweepRoom {
public:
    // want: compute units relied on (at least 1), cap: those of the device.
    void enter(int want, int cap) {
        std::unique_lock<std::mutex> l(m_);
        const unsigned long long me = next_++;
        cv_.wait(l, [&] { return me == serving_ && (used_ == 0 || used_ + want <= cap); });
        ++serving_;
        used_ += want;
        cv_.notify_all();
    }
    void leave(int want) {
        std::lock_guard<std::mutex> l(m_);
        used_ -= want;
        cv_.notify_all();
    }

private:
    std::mutex m_;
    std::condition_variable cv_;
    unsigned long long next_ = 0, serving_ = 0;
    int used_ = 0;
};

// For the time of a solve; want 0: nothing is relied on.
class SweepLease {
public:
    SweepLease(SweepRoom& room, int want, int cap) : room_(room), want_(want) {
        if (want_ > 0) room_.enter(want_, cap);
    }
    ~SweepLease() {
        if (want_ > 0) room_.leave(want_);
    }
    SweepLease(const SweepLease&) = delete;
    SweepLease& operator=(const SweepLease&) = delete;

private:
    SweepRoom& room_;
    int want_;
};

}  // namespace astg
