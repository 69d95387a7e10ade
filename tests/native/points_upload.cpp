// A point list with room for its FP64 coordinates but not for the raw ones
// beside them: the field of the same call with room for both.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <string>
#include <vector>

#include "scarf3d.h"
#include "scarf3d_srm.h"

namespace {

std::vector<real> list(const std::vector<real> (&p)[3], int nd, int nharm, int kernel, real (&stats)[8], std::string &err)
{
    scarf_opt o;
    scarf_opt_init(&o);
    o.method = 1;
    o.hurst = real(0.3);
    const real cl[3] = {300, 250, 200};
    std::vector<real> field(p[0].size(), real(0));
    scarf_nocart_initialize(nd, int(p[0].size()), p[0].data(), p[1].data(), nd == 3 ? p[2].data() : nullptr, real(40), 0, cl,
                            real(0.05), &o);
    scarf_set_nharm(nharm);
    scarf_set_kernel(kernel);
    scarf_execute(3, field.data(), stats);
    err = scarf_last_error();
    scarf_finalize();
    return field;
}

}  // namespace

int main()
{
    int bad = 0;
    const int n = 30011, nharm = 900, np = 960;
    std::vector<real> p[3];
    for (int q = 0; q < 3; ++q)
        for (int i = 0; i < n; ++i) p[q].push_back(real((i * (7919LL + 104 * q) % 20011) * (0.1 - 0.02 * q)));
    const int direct = sizeof(real) == 4 ? SCARF_KERNEL_DIRECT_F32 : SCARF_KERNEL_DIRECT_F64;
    // field, record, FP64 coordinates, the direct sum's partials
    const size_t room = n * sizeof(real) + 5 * np * sizeof(double) + 3 * sizeof(double) * size_t(n) +
                        3 * sizeof(double) * ((n + 255) / 256);
    for (const int nd : {3, 2}) {
        real at[8], free[8];
        std::string err;
        setenv("SCARF_DEVICE_MEMORY_LIMIT", std::to_string(room).c_str(), 1);
        const std::vector<real> a = list(p, nd, nharm, direct, at, err);
        std::printf("%dD at the limit: %s\n", nd, err.empty() ? "runs" : err.c_str());
        bad += !err.empty();
        unsetenv("SCARF_DEVICE_MEMORY_LIMIT");
        const std::vector<real> b = list(p, nd, nharm, direct, free, err);
        const bool same = a == b && std::equal(at, at + 4, free);
        std::printf("%dD: %s\n", nd, same ? "the same field" : "another field");
        bad += !err.empty() || !same;
    }
    std::printf("%d bad\n", bad);
    return bad != 0;
}
