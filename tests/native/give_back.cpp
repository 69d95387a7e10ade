// A point list whose grid takes more than 4 GiB gives the workspace back when
// the object is finalized; a small list's stays.
#include <cstdio>
#include <string>
#include <vector>

#include "device_budget.hpp"
#include "scarf3d.h"
#include "scarf3d_srm.h"

namespace {

int bad = 0;

void list(int n, real box, real dh, int nharm, bool large)
{
    std::vector<real> p[3], field(n, real(0));
    unsigned s = 12345;
    for (int q = 0; q < 3; ++q)
        for (int i = 0; i < n; ++i) {
            s = s * 1664525u + 1013904223u;
            p[q].push_back(real((s >> 8) / 16777216.0 * box));
        }
    scarf_opt o;
    scarf_opt_init(&o);
    o.method = 1;
    o.hurst = real(0.3);
    const real cl[3] = {300, 250, 200};
    real stats[8];
    scarf_nocart_initialize(3, n, p[0].data(), p[1].data(), p[2].data(), dh, 0, cl, real(0.05), &o);
    scarf_set_nharm(nharm);
    scarf_set_kernel(SCARF_KERNEL_AUTO);
    scarf_execute(1, field.data(), stats);
    const std::string err = scarf_last_error();
    const size_t before = scarf::device_budget().held();
    scarf_finalize();
    const size_t after = scarf::device_budget().held();
    const size_t gib = size_t(1) << 30;
    const bool ok = err.empty() && (large ? before > 4 * gib && after < gib : before < gib && after == before);
    bad += !ok;
    std::printf("%d points: %zu held, %zu after %s\n", n, before, after, err.c_str());
}

}  // namespace

int main()
{
    list(20000, 2000, 40, 1900, false);
    list(2000000, 5000, 10, 60000, true);
    list(2000000, 5000, 10, 60000, true);
    list(20000, 2000, 40, 1900, false);
    std::printf("%d bad\n", bad);
    return bad != 0;
}
