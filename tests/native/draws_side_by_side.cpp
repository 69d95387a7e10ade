// The rule that takes an ensemble's draws side by side or one after the other:
// by its own estimates no slower than all draws the one way or all the other
// (within the quarter it leaves for uneven draws), over many mixed sets.
#include <algorithm>
#include <cstdio>
#include <random>
#include <vector>

#include "srm_host.hpp"

using scarf::DrawCost;

namespace {

double time_of(const std::vector<DrawCost> &c, const std::vector<char> &side, int threads)
{
    double one_by_one = 0, together = 0, longest = 0;
    int k = 0;
    for (size_t m = 0; m < c.size(); ++m) {
        if (!side[m]) one_by_one += c[m].screened;
        else {
            together += c[m].alone;
            longest = std::max(longest, c[m].alone);
            ++k;
        }
    }
    return one_by_one + (k ? std::max(longest, together / std::min(k, threads)) : 0.0);
}

}  // namespace

int main()
{
    int bad = 0;
    std::mt19937 rng(7);
    auto setup = [](double acceptance) {
        scarf::SrmSetup s;
        s.kmin = 0.0;
        s.kmax = 1.0;
        s.cnst = 1.0;
        s.band = acceptance;
        return s;
    };
    for (int set = 0; set < 4000; ++set) {
        const int n = 1 + int(rng() % 100), threads = 1 + int(rng() % 16);
        const bool alike = set % 2 == 0;
        std::vector<DrawCost> c;
        for (int m = 0; m < n; ++m) {
            if (alike && m > 0) {
                c.push_back(c[0]);
                continue;
            }
            const double share = std::pow(10.0, -3.0 * (rng() % 1000) / 1000.0);
            c.push_back(scarf::draw_cost(int(std::pow(10.0, 1.5 + 3.0 * (rng() % 1000) / 1000.0)), setup(share)));
        }
        const std::vector<char> side = scarf::draws_side_by_side(c, threads);
        const double t = time_of(c, side, threads), none = time_of(c, std::vector<char>(n, 0), threads),
                     all = time_of(c, std::vector<char>(n, 1), threads);
        if (t > 1.26 * std::min(none, all) || t > none * 1.001) {
            std::printf("set %d: %d members, %d threads: %.3f ms, screened %.3f, side by side %.3f\n", set, n, threads, t,
                        none, all);
            ++bad;
        }
    }
    // many short draws go side by side, long ones and a lone one do not
    const std::vector<DrawCost> shorts(64, scarf::draw_cost(150, setup(0.05)));
    const std::vector<DrawCost> longs(16, scarf::draw_cost(16000, setup(0.004)));
    const std::vector<DrawCost> one(1, scarf::draw_cost(400, setup(0.05)));
    for (const auto &[c, want] : {std::make_pair(shorts, 64), std::make_pair(longs, 0), std::make_pair(one, 0)}) {
        const std::vector<char> side = scarf::draws_side_by_side(c, 16);
        const int got = int(std::count(side.begin(), side.end(), 1));
        if (got != want) {
            std::printf("%zu draws of %.3f ms: %d side by side\n", c.size(), c[0].alone, got);
            ++bad;
        }
    }
    std::printf("%d bad\n", bad);
    return bad != 0;
}
