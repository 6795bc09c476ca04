// cu_budget.h -- the compute units that one-launch solves (resident.hip) hold on a device.
#pragma once

#include <condition_variable>
#include <cstdint>
#include <mutex>

namespace shk {

// Workgroups of resident launches in flight per device: their sum never exceeds the CUs, so
// that every launch gets all of its workgroups onto the chip.  Requests are served in the
// order they come: one that would fit waits behind a larger one, or small solves of several
// threads could keep a large one out for good.
class CuBudget {
    std::mutex m_;
    std::condition_variable cv_;
    int used_ = 0;
    uint64_t next_ = 0, serving_ = 0;

public:
    void acquire(int blocks, int cus) {
        std::unique_lock<std::mutex> lk(m_);
        const uint64_t ticket = next_++;
        cv_.wait(lk, [&] { return serving_ == ticket && used_ + blocks <= cus; });
        used_ += blocks;
        ++serving_;
        cv_.notify_all();
    }
    void release(int blocks) {
        {
            std::lock_guard<std::mutex> lk(m_);
            used_ -= blocks;
        }
        cv_.notify_all();
    }
};

}  // namespace shk
