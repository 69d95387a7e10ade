// The interpolation's launches of a point list: consecutive, every point in
// one of them, no launch with 2^32 threads or more (what HIP takes at most),
// up to the largest list that the plan accepts.
#include <cstdio>

#include "srm_points.hpp"

int main()
{
    int bad = 0;
    for (const bool f64 : {false, true}) {
        const long taps = f64 ? 16 : 8, per_block = scarf::kPointsThreads / taps;
        const long part = scarf::kPointsBlocks * per_block;
        for (long n : {1L, per_block, per_block + 1, part - 1, part, part + 1, 2 * part + 5, (1L << 28) - 1, 1L << 28,
                       (1L << 29) - 1, 1L << 29, 0x7fffffffL}) {
            long next = 0;
            for (const scarf::PointsLaunch &l : scarf::points_launches(n, f64)) {
                const bool ok = l.first == next && l.blocks > 0 && long(l.blocks) * scarf::kPointsThreads < (1L << 32) &&
                                l.first + (long(l.blocks) - 1) * per_block < n;
                if (!ok) {
                    std::printf("f64 %d, %ld points: launch from %ld, %u blocks\n", int(f64), n, l.first, l.blocks);
                    ++bad;
                }
                next = l.first + long(l.blocks) * per_block;
            }
            if (next < n) {
                std::printf("f64 %d, %ld points: %ld covered\n", int(f64), n, next);
                ++bad;
            }
            // the plan takes such a list: its grid does not grow with the points
            const double lo[3] = {0, 0, 0}, hi[3] = {1000, 900, 800}, wmax[3] = {0.1, 0.1, 0.1};
            scarf::PointsPlan p;
            if (!scarf::points_plan(lo, hi, wmax, false, n, 4096, f64, p)) {
                std::printf("f64 %d, %ld points: no plan\n", int(f64), n);
                ++bad;
            }
        }
    }
    std::printf("%d bad\n", bad);
    return bad != 0;
}
