// resident_ticket.h -- the compute units that resident kernels of this process hold, per device.
//
// A resident kernel ends only if all of its blocks run at the same time, and almost every
// instance needs a compute unit for each (its registers leave no room for a second block).  Blocks
// of two such kernels that cannot all run would wait for each other until their waits run out,
// so a launch that does not fit beside those in flight is not made.
//
// Blocks go to the XCDs in turn, so b blocks take up to ceil(b / 8) compute units of each: that is
// what is counted.  (Counted in blocks, 132 and 124 of them would fit 256 units; four XCDs would
// get 17 + 16 for their 32.)
#pragma once

#include <mutex>

namespace prism_hip {

constexpr int XCDS = 8;

class ResidentTicket {
    struct Device {
        std::mutex use;
        int held{0};  // compute units of an XCD
    };
    static Device& device(int i) {
        static Device d[64];
        return d[i & 63];
    }
    Device* at_{nullptr};
    int share_{0};

public:
    // True when a kernel of `blocks` blocks fits beside those in flight on the device (one that
    // is alone always does: its plan has no more blocks than compute units).
    bool take(int dev, int blocks, int n_cu) {
        give();
        const int share = (blocks + XCDS - 1) / XCDS;
        Device& d = device(dev);
        std::lock_guard<std::mutex> lock(d.use);
        if (d.held > 0 && d.held + share > n_cu / XCDS) return false;
        d.held += share;
        at_ = &d;
        share_ = share;
        return true;
    }
    void give() {
        if (!at_) return;
        std::lock_guard<std::mutex> lock(at_->use);
        at_->held -= share_;
        at_ = nullptr;
    }
    ResidentTicket() = default;
    ResidentTicket(const ResidentTicket&) = delete;
    ResidentTicket& operator=(const ResidentTicket&) = delete;
    ~ResidentTicket() { give(); }
};

}  // namespace prism_hip
