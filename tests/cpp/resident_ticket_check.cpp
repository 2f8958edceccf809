// Which resident kernels may be in flight together (prism_amd/csrc/resident_ticket.h): the blocks of
// every set that is let in, dealt to the XCDs in turn from any one on, fit their compute
// units; the others wait, and are served in the order of asking, or are told that they do not fit.
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <thread>
#include <vector>

#include "../../prism_amd/csrc/resident_ticket.h"

using prism_hip::ResidentTicket;
using prism_hip::XCDS;

static void check(bool ok, const char* what, int a, int b) {
    if (ok) return;
    std::printf("FAILED: %s (%d, %d)\n", what, a, b);
    std::exit(1);
}

static void settle() { std::this_thread::sleep_for(std::chrono::milliseconds(50)); }

int main() {
    const int cu = 256;
    for (int a = 1; a <= cu; ++a)
        for (int b = 1; b <= cu; ++b) {
            const bool both = ResidentTicket::fits(ResidentTicket::share(a), ResidentTicket::share(b), cu);
            // most blocks that an XCD of 32 units can get
            const int worst = (a + XCDS - 1) / XCDS + (b + XCDS - 1) / XCDS;
            check(!both || worst <= cu / XCDS, "more blocks than an XCD has units", a, b);
            check(both || worst > cu / XCDS, "refused though it fits", a, b);
            check(ResidentTicket::fits(0, ResidentTicket::share(a), b), "a kernel alone is refused", a, b);
        }
    {
        // 132 and 124 blocks want 17 + 16 of 32 units: the second waits, and what asks after it
        // (small enough to go at once) does not pass it
        ResidentTicket first;
        check(first.take(0, 132, cu, false), "a kernel alone is refused", 132, 0);
        std::atomic<int> order{0};
        int big = 0, small = 0, elsewhere = 0;
        std::thread t([&] {
            ResidentTicket s;
            s.take(0, 124, cu, true);
            big = ++order;
            settle();
        });
        settle();
        std::thread u([&] {
            ResidentTicket s;
            s.take(0, 8, cu, true);
            small = ++order;
        });
        settle();
        check(order == 0, "let in beside 132 blocks", 132, 124);
        ResidentTicket other;
        check(!other.take(0, 8, cu, false), "passed those who wait", 8, 0);
        std::thread v([&] {
            ResidentTicket s;
            s.take(1, cu, cu, true);
            elsewhere = 1;
        });
        v.join();
        check(elsewhere == 1, "another device's kernels are counted", 1, 0);
        first.give();
        t.join();
        u.join();
        check(big == 1 && small == 2, "order of asking", big, small);
        check(first.take(0, cu, cu, false) && !other.take(0, 1, cu, false), "a full device", cu, 1);
        check(first.take(0, cu, cu, false), "taken again: its first units are given back", cu, 0);
    }
    {
        // never more than the units of an XCD at once
        std::atomic<int> held{0}, worst{0}, rounds{0};
        std::vector<std::thread> ts;
        for (int k = 0; k < 6; ++k)
            ts.emplace_back([&, k] {
                ResidentTicket s;
                for (int i = 0; i < 500; ++i) {
                    const int blocks = 1 + (37 * i + 91 * k) % cu, units = ResidentTicket::share(blocks);
                    if (!s.take(2, blocks, cu, i % 3 != 0)) continue;
                    const int h = held += units;
                    if (h > worst) worst = h;
                    held -= units;
                    s.give();
                    if (i % 3) ++rounds;
                }
            });
        for (auto& t : ts) t.join();
        check(rounds == 6 * 333 && worst <= cu / XCDS, "units held at once", rounds, worst);
    }
    {
        // waits that run out after 0.4 s each, in a process that solves without a pause
        prism_hip::ResidentRest rest;
        check(rest.over(0.0), "off at the start", 0, 0);
        double now = 100.0, lost = 0.0;
        int waits = 0;
        while (now < 1100.0) {
            if (rest.over(now)) {
                now += 0.4;
                lost += 0.4;
                ++waits;
                rest.ranOut(0.4, now);
                check(!rest.over(now) && !rest.over(now + 3.1), "on again at once", waits, 0);
            }
            now += 0.005;  // a solve
            check(lost <= 0.4 + (now - 100.0) / 9.0, "time lost", waits, (int)now);
        }
        check(waits >= 5 && waits <= 10, "waits in 1000 s", waits, 0);
        rest.endedWell();
        rest.ranOut(0.4, 5000.0);
        check(!rest.over(5003.1) && rest.over(5003.3), "the first rest again", 0, 0);
    }
    std::puts("ok");
}
