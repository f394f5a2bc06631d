// sf_grid_gate.h -- which grid-mode launches of a device may run at the same time.
#pragma once

#include <condition_variable>
#include <cstdint>
#include <mutex>

namespace sf {

// The workgroups of a grid-mode launch wait for each other, so all of them must be resident.  Two
// launches at once (captured steps on two threads) could each hold a part of the chip and wait for the
// rest until the time limit: a workgroup of the resident passes has 12 or 16 waves of 128 VGPRs and
// fills a CU, and 128^2 nodes already take 192 of them.  A workgroup takes at most one CU whatever its
// waves and registers, so launches whose workgroups together number no more than the CUs always all get
// in.  enter(n) waits until n more do, in order of arrival, so that a large launch is not passed by small
// ones for ever.  One gate per device.
class GridGate {
public:
    void enter(int n, int cus)
    {
        std::unique_lock<std::mutex> lock(m_);
        const uint64_t mine = next_++;
        cv_.wait(lock, [&] { return turn_ == mine && (used_ == 0 || used_ + n <= cus); });
        used_ += n;
        ++turn_;
        cv_.notify_all();
    }
    void leave(int n)
    {
        std::lock_guard<std::mutex> lock(m_);
        used_ -= n;
        cv_.notify_all();
    }

private:
    std::mutex m_;
    std::condition_variable cv_;
    int used_ = 0;
    uint64_t next_ = 0, turn_ = 0;  // tickets given out, and the one whose turn it is
};

}  // namespace sf
