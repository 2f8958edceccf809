// resident_ticket.h -- the compute units that resident kernels of this process hold, per device.
//
// A resident kernel ends only if all of its blocks run at the same time, and almost every
// instance needs a compute unit for each (its registers leave no room for a second block).  Blocks
// of two such kernels that cannot all run would wait for each other until their waits run out,
// so a launch that does not fit beside those in flight is not made.  Where the launches of the
// single kernels give the same bits the caller takes those for a chunk of iterations (four
// threads, 100,000 rows FP64: 298 us a solve, and 434 us where they take turns); elsewhere it waits
// for its turn, in the order of asking, for a launch of 128 iterations (1 to 4 ms) or two, or a
// solve's bits would depend on what other threads did meanwhile (four threads, 262,144 rows:
// 683 us a solve, and 716 us without turns).
//
// Blocks go to the XCDs in turn, so b blocks take up to ceil(b / 8) compute units of each: that is
// what is counted.  (Counted in blocks, 132 and 124 of them would fit 256 units; four XCDs would
// get 17 + 16 for their 32.)
#pragma once

#include <algorithm>
#include <condition_variable>
#include <mutex>

namespace prism_hip {

constexpr int XCDS = 8;

class ResidentTicket {
    struct Device {
        std::mutex use;
        std::condition_variable turn;
        int held{0};  // compute units of an XCD
        unsigned long long asked{0}, served{0};
    };
    static Device& device(int i) {
        static Device d[64];
        return d[i & 63];
    }
    Device* at_{nullptr};
    int share_{0};

public:
    // Compute units of an XCD that `blocks` blocks take, and whether that many fit beside `held`
    // (a kernel alone always does: its plan has no more blocks than compute units).
    static int share(int blocks) { return (blocks + XCDS - 1) / XCDS; }
    static bool fits(int held, int share, int n_cu) { return held == 0 || held + share <= n_cu / XCDS; }

    // False when the launch is not to be made now (never with `wait`).
    bool take(int dev, int blocks, int n_cu, bool wait) {
        give();
        const int want = share(blocks);
        Device& d = device(dev);
        std::unique_lock<std::mutex> lock(d.use);
        // who does not wait does not pass those who do
        if (!wait && (d.asked != d.served || !fits(d.held, want, n_cu))) return false;
        const unsigned long long mine = d.asked++;
        d.turn.wait(lock, [&] { return mine == d.served && fits(d.held, want, n_cu); });
        ++d.served;
        d.held += want;
        at_ = &d;
        share_ = want;
        d.turn.notify_all();
        return true;
    }
    void give() {
        if (!at_) return;
        std::lock_guard<std::mutex> lock(at_->use);
        at_->held -= share_;
        at_->turn.notify_all();
        at_ = nullptr;
    }
    ResidentTicket() = default;
    ResidentTicket(const ResidentTicket&) = delete;
    ResidentTicket& operator=(const ResidentTicket&) = delete;
    ~ResidentTicket() { give(); }
};

// When a context takes resident kernels again after a wait that ran out: their blocks do not
// run together then, because another process (whose kernels the ticket does not see) holds compute
// units, and the next solves would lose the same time, up to 2^20 polls (several tenths
// of a second) for a solve of milliseconds.  They stay off for 8 times the time lost, twice as long
// each further time in a row: at most a ninth of the time goes into such waits.  Times in
// seconds, of one steady clock.
class ResidentRest {
    std::mutex use_;
    double until_{0.0}, factor_{FIRST};

public:
    static constexpr double FIRST = 8.0, MOST = 1024.0;
    bool over(double now) {
        std::lock_guard<std::mutex> lock(use_);
        return now >= until_;
    }
    void ranOut(double lost, double now) {
        std::lock_guard<std::mutex> lock(use_);
        until_ = now + factor_ * lost;
        factor_ = std::min(2.0 * factor_, MOST);
    }
    void endedWell() {
        std::lock_guard<std::mutex> lock(use_);
        factor_ = FIRST;
    }
};

}  // namespace prism_hip
