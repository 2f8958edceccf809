// Which resident kernels may be in flight together (prism_amd/csrc/resident_ticket.h): the blocks of
// every set that is let in, dealt to the XCDs in turn from any one on, fit their compute units.
#include <cstdio>
#include <cstdlib>

#include "../../prism_amd/csrc/resident_ticket.h"

using prism_hip::ResidentTicket;
using prism_hip::XCDS;

static void check(bool ok, const char* what, int a, int b) {
    if (ok) return;
    std::printf("FAILED: %s (%d, %d)\n", what, a, b);
    std::exit(1);
}

int main() {
    const int cu = 256;
    for (int a = 1; a <= cu; ++a)
        for (int b = 1; b <= cu; ++b) {
            ResidentTicket s, t;
            check(s.take(0, a, cu), "a kernel alone is refused", a, 0);
            const bool both = t.take(0, b, cu);
            // most blocks that an XCD of 32 units can get
            const int worst = (a + XCDS - 1) / XCDS + (b + XCDS - 1) / XCDS;
            check(!both || worst <= cu / XCDS, "more blocks than an XCD has units", a, b);
            check(both || worst > cu / XCDS, "refused though it fits", a, b);
            ResidentTicket other;
            check(other.take(1, cu, cu), "another device's kernels are counted", a, b);
        }
    {
        ResidentTicket s, t;
        check(s.take(0, 132, cu) && !t.take(0, 124, cu), "17 + 16 of 32 units", 132, 124);
        s.give();
        check(t.take(0, 124, cu), "units given back are not free", 132, 124);
        check(t.take(0, cu, cu), "a ticket taken again keeps its first units", cu, 0);
    }
    ResidentTicket t;
    check(t.take(0, 7, 6), "a device of few units, alone", 7, 6);
    std::puts("ok");
}
