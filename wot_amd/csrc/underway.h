// The solves under way on each GPU.  Not part of the C ABI.
#pragma once
#include <atomic>

#include <hip/hip_runtime.h>

namespace wotk {

constexpr int kMaxDevices = 64;

// One solve of this process, from its first launch to its last wait.  A persistent launch has its CUs
// to itself, and two at once could each hold CUs that the other waits for, while the launched sweeps
// of several threads fill each other's gaps: per solve and iteration, 1 / 2 / 8 threads at once,
// launched 8.4 / 4.4 / 2.4 us, resident 5.2 one after the other, at 300 x 400; 15.0 / 9.1 / 7.1 and
// 11.1 at 2000 x 2500.  So a solve is resident only if no other is under way where it starts; its
// bits are the same either way.
class UnderWay {
public:
    UnderWay() {
        if (hipGetDevice(&dev_) != hipSuccess || dev_ < 0 || dev_ >= kMaxDevices) dev_ = -1;
        alone_ = dev_ >= 0 && count_[dev_].fetch_add(1) == 0;
    }
    ~UnderWay() {
        if (dev_ >= 0) count_[dev_].fetch_sub(1);
    }
    UnderWay(const UnderWay &) = delete;
    UnderWay &operator=(const UnderWay &) = delete;
    bool alone() const { return alone_; }

private:
    inline static std::atomic<int> count_[kMaxDevices] = {};
    int dev_ = -1;
    bool alone_ = false;
};

}  // namespace wotk
