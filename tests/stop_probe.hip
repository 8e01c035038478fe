// Host program for tests/test_stop_flag.py: runs the basic scheme's stop
// decision on a control block and prints which passes take part before it,
// after it (the rest of the launch that decided) and after the next z pass.
#include "../mat3d_amd/csrc/m3d_basic.hpp"
#include "../mat3d_amd/csrc/m3d_flex.hpp"

#include <cstdio>
#include <cstring>

using namespace m3d;

// the inverse and the forward y pass, run-time and compile-time lengths
static void passes(const Ctl& c)
{
    std::printf("%d%d%d%d", flex::active(c, BUF_MAIN), flex::active(c, BUF_K), fast::xy_active<BUF_MAIN>(c),
                fast::xy_active<BUF_K>(c));
}

int main()
{
    for (int why = 0; why < 4; ++why) { // goes on, converged, cap, constitutive update failed
        Ctl c;
        std::memset(&c, 0, sizeof c);
        c.it = 5;
        c.cap = why == 2 ? 4 : 100;
        c.err = why == 3;
        c.deq = c.dsum = why == 1 ? 1e-8 : 1.0;
        c.tol_f = c.tol_eq = 1e-6;
        passes(c);
        bstop_rule(c);
        std::printf(" ");
        passes(c);
        const bool other = bz_skip(c, false);
        std::printf(" %d ", other);
        passes(c);
        const bool first = bz_skip(c, true);
        std::printf(" %d ", first);
        passes(c);
        std::printf(" %d\n", c.done);
    }
}
