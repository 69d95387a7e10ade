// The transform's workspace over shapes and harmonic counts: beyond the tables
// per harmonic and one round of its fewest planes it stays below 448 MiB, also
// for thin blocks of many planes and many harmonics, and every plane is in a
// round.
#include <algorithm>
#include <cstdio>

#include "srm_transform.hpp"

int main()
{
    int bad = 0, plans = 0;
    for (const bool f64 : {false, true})
        for (int nx : {1, 7, 30, 100, 301, 1024, 4000})
            for (int ny : {1, 8, 30, 257, 1024, 2000})
                for (int nz : {1, 9, 129, 2000, 16384, 1000000})
                    for (int np : {64, 5056, 30016, 300032, 1000000}) {
                        scarf::Geometry g;
                        g.structured = true;
                        g.nx = nx;
                        g.ny = ny;
                        g.nz = nz;
                        g.ds = 10.0;
                        scarf::TransformPlan p;
                        if (!scarf::transform_plan(g, np, f64, p)) continue;
                        ++plans;
                        const size_t size = f64 ? 16 : 8, cls = f64 ? 16 : 8;
                        const size_t tables = size_t(np) * (8 + (2 * cls + 16) * 8) + (p.l / cls) * (p.m + 2) * sizeof(int) +
                                              (4 * size_t(p.l) + 4 * size_t(p.m)) * size + 8 * (size_t(nx) + ny) + 16384;
                        const size_t round = 8 * size_t(p.zb) * (size_t(p.columns) * ny + np) * size;
                        const size_t most = tables + std::max(round, size_t(448) << 20);
                        if (p.bytes > most || p.slab < 1 || p.slab % p.zb != 0) {
                            std::printf("f64 %d %d x %d x %d, %d harmonics: %zu bytes, %d planes a round\n", int(f64), nx, ny,
                                        nz, np, p.bytes, p.slab);
                            ++bad;
                        }
                    }
    std::printf("%d plans, %d bad\n", plans, bad);
    return bad != 0;
}
