// coop.hpp — admission of kernels whose workgroups wait for each other (a GMRES solve of several
// workgroups, the panels of a large LU).  Such a kernel makes progress once all its workgroups run, and
// two that each hold a part of the CUs wait for each other until their bound.  A GMRES workgroup fills its
// CU (149 KB of LDS), so the kernels in flight on a device may take at most its CUs less a margin
// together: the last one to start then always finds its CUs.
#pragma once
#include <algorithm>
#include <condition_variable>
#include <cstdint>
#include <mutex>

namespace lsx {

constexpr int COOP_MARGIN = 16;  // CUs never reserved: panels of up to 16 workgroups go unannounced
inline int coop_cus(int num_cus) { return std::max(64, num_cus - COOP_MARGIN); }

// Workgroups in flight on one device, granted in the order of the requests (so that a wide solve is not
// overtaken for ever).  A request for more than the total takes the whole of it.
class CoopBudget {
  public:
    void acquire(int k, int total) {
        std::unique_lock<std::mutex> lk(mu_);
        const uint64_t me = next_++;
        cv_.wait(lk, [&] { return me == turn_ && used_ + std::min(k, total) <= total; });
        used_ += std::min(k, total);
        turn_ += 1;
        cv_.notify_all();
    }
    void release(int k, int total) {
        std::lock_guard<std::mutex> lk(mu_);
        used_ -= std::min(k, total);
        cv_.notify_all();
    }

  private:
    std::mutex mu_;
    std::condition_variable cv_;
    uint64_t next_ = 0, turn_ = 0;
    int used_ = 0;
};

// The budget of a device, shared by every context, handle and server of the process.
inline CoopBudget& coop_budget(int device) {
    static CoopBudget b[64];
    return b[device & 63];
}

// k workgroups of a device from take() until the hold ends, which must be after the kernel's end.
// Nothing is taken for a kernel of one workgroup (it waits for nobody).
class CoopHold {
  public:
    CoopHold() = default;
    CoopHold(const CoopHold&) = delete;
    CoopHold& operator=(const CoopHold&) = delete;
    ~CoopHold() {
        if (b_) b_->release(k_, total_);
    }
    void take(int device, int num_cus, int k) {
        if (b_ || k <= 1) return;
        total_ = coop_cus(num_cus);
        k_ = k;
        coop_budget(device).acquire(k_, total_);
        b_ = &coop_budget(device);
    }

  private:
    CoopBudget* b_ = nullptr;
    int k_ = 0, total_ = 0;
};

}  // namespace lsx
