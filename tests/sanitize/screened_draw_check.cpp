// The draw with its trials screened elsewhere (HarmonicSampler::create_rows
// with a TrialScreen), here by a host screen: Yarn2 and the bins' limits, with
// the verdict of a 64-bit test and a margin, some pairs left open and some
// rejected. Its rows must equal build_table's of the unscreened draw bit for
// bit, whatever the cuts of the walk, the block sizes, the number of threads,
// and wherever the screen gives up. Built by tests/test_sanitize_screen.py
// with AddressSanitizer and UndefinedBehaviorSanitizer.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "srm_host.hpp"
#include "yarn2.hpp"

using namespace scarf;

namespace {

class HostScreen : public TrialScreen {
public:
    long fail_after = -1;   // blocks screened before the screen gives up
    long at_most = 0;       // pairs of a block, fewer than asked for
    unsigned open = 0;      // every open-th pair is left to the draw
    long blocks = 0, held = 0, rejected = 0, unsure = 0;

    bool screen(int seed, long first, long count, const TrialTest &t, const uint32_t *limit, int bins,
                TrialBlock &out) override
    {
        if (fail_after >= 0 && blocks >= fail_after) return false;
        ++blocks;
        if (at_most > 0) count = std::min(count, at_most);
        Yarn2 g;
        g.seed(static_cast<unsigned long>(seed));
        g.discard(2 * static_cast<uint64_t>(first));
        std::vector<uint32_t> v(2 * static_cast<size_t>(count + 3));
        for (uint32_t &x : v) x = static_cast<uint32_t>(g());
        pairs_.clear();
        raw_.clear();
        const uint64_t width = (uint64_t(1) << 31) / static_cast<uint64_t>(bins);
        for (long p = 0; p < count; ++p) {
            const uint32_t *r = v.data() + 2 * p;
            if (r[1] >= limit[r[0] / width]) continue;
            const uint32_t how = verdict(t, r[0], r[1], first + p);
            pairs_.push_back(static_cast<uint32_t>(p) | how << 30);
            raw_.insert(raw_.end(), r, r + TrialBlock::kRaw);
            ++held;
            rejected += how == TrialBlock::kReject;
            unsure += how == TrialBlock::kUnsure;
        }
        out.start = first;
        out.end = first + count;
        out.pairs = pairs_.data();
        out.raw = raw_.data();
        out.total = pairs_.size();
        return true;
    }

private:
    uint32_t verdict(const TrialTest &t, uint32_t v0, uint32_t v1, long pair) const
    {
        if (open > 0 && pair % open == 0) return TrialBlock::kUnsure;
        double u, r1;
        if (t.f64) {
            const double p = Yarn2::to_uniform01(v0) * t.range;
            u = p + t.kmin;
            r1 = Yarn2::to_uniform01(v1);
        } else {
            const float p = static_cast<float>(Yarn2::to_uniform01(v0)) * static_cast<float>(t.range);
            u = p + static_cast<float>(t.kmin);
            r1 = static_cast<float>(Yarn2::to_uniform01(v1));
        }
        double a = t.acf == 0 ? std::pow(1.0 + u * u, -t.nu) : std::exp(-0.25 * u * u);
        a *= (t.ndim == 3 ? u * u : u) * t.cnst;
        const double margin = t.f64 ? 1e-10 : 2e-5;
        if (r1 < a * (1.0 - margin) && a > 1e-30) return u > t.kc ? TrialBlock::kDrop : TrialBlock::kKeep;
        if (r1 > a * (1.0 + margin) + 1e-30) return TrialBlock::kReject;
        return TrialBlock::kUnsure;
    }
    std::vector<uint32_t> pairs_, raw_;
};

SrmConfig grid(int nd, int n, double ds, double dh, int acf, double cl, double hurst, int nharm, double alpha = 0)
{
    SrmConfig c;
    c.nd = nd;
    c.structured = true;
    for (int i = 0; i < 3; ++i) {
        c.fs[i] = 1;
        c.fe[i] = i < nd ? n : 1;
        c.cl[i] = i < nd ? cl * (1.0 - 0.1 * i) : 0;
        c.nc[i] = 0;
        c.fc[i] = i < nd ? (n - 1) * ds : 0;
    }
    c.ds = ds;
    c.dh = dh;
    c.acf = acf;
    c.sigma = 0.05;
    c.hurst = hurst;
    c.alpha = alpha;
    c.method = 1;
    c.nharm = nharm;
    return c;
}

template <class Real>
int check(const char *name, const SrmConfig &c)
{
    SrmSetup s;
    std::string err;
    if (srm_setup<Real>(c, s, err) != 0) {
        std::printf("%s: %s\n", name, err.c_str());
        return 1;
    }
    struct Way {
        int cut, threads;
        long block, fail_after, at_most;
        unsigned open;
    };
    const Way ways[] = {{1 << 30, 1, 0, -1, 0, 0},  {1 << 30, 4, 0, -1, 0, 3}, {7, 3, 0, -1, 0, 1},
                        {128, 4, 37, -1, 0, 5},     {64, 2, 0, 2, 501, 2},     {1 << 30, 4, 2049, 3, 0, 0},
                        {1 << 30, 1, 0, 0, 0, 0},   {100, 2, 0, -1, 97, 4}};
    int bad = 0;
    for (int seed : {1234, 77, 2000000011}) {
        std::unique_ptr<HarmonicSampler> plain = HarmonicSampler::create<Real>(c, s, seed, 2);
        plain->draw_until(1 << 30);
        const HarmonicTable t = build_table(s, plain->draw());
        const std::vector<double> *want[5] = {&t.wx, &t.wy, &t.wz, &t.phase, &t.amp};
        for (const Way &w : ways) {
            HostScreen screen;
            screen.fail_after = w.fail_after;
            screen.at_most = w.at_most;
            screen.open = w.open;
            std::unique_ptr<HarmonicSampler> d =
                HarmonicSampler::create_rows<Real>(c, s, seed, &screen, w.threads, w.block);
            int kept = 0;
            bool same = true;
            for (long until = w.cut; !d->finished(); until += w.cut) {
                const int now = d->draw_until(static_cast<int>(std::min<long>(until, 1 << 30)));
                const HarmonicRows r = d->rows(kept, now);
                for (int f = 0; f < 5 && now > kept; ++f)
                    same = same && now <= t.count() &&
                           std::memcmp(r.field[f], want[f]->data() + kept, size_t(now - kept) * sizeof(double)) == 0;
                kept = now;
            }
            same = same && kept == t.count();
            if (!same || (screen.blocks == 0 && w.fail_after != 0)) {
                std::printf("%s seed %d cut %d threads %d block %ld: %d of %d kept, %s, %ld blocks\n", name, seed, w.cut,
                            w.threads, w.block, kept, t.count(), same ? "the same" : "other harmonics", screen.blocks);
                ++bad;
            }
            std::printf("%s %d: %ld blocks, %ld held, %ld rejected, %ld open\n", name, seed, screen.blocks, screen.held,
                        screen.rejected, screen.unsure);
        }
    }
    return bad;
}

}  // namespace

int main()
{
    int bad = 0;
    bad += check<float>("vk", grid(3, 64, 20.0, 20.0, 0, 5000.0, 0.1, 900));
    bad += check<double>("vk_rotated", grid(3, 64, 20.0, 8.0, 0, 3000.0, 0.3, 600, 30.0));
    bad += check<float>("gauss", grid(3, 60, 100.0, 100.0, 1, 300.0, 0.0, 1500));  // the maximum inside the band
    bad += check<double>("gauss_d", grid(3, 40, 50.0, 50.0, 1, 300.0, 0.0, 700));
    bad += check<float>("plane", grid(2, 50, 30.0, 30.0, 0, 150.0, 0.3, 1500));
    bad += check<float>("dropped", grid(3, 20, 40.0, 10.0, 0, 200.0, 0.1, 1500));  // harmonics above kc
    bad += check<double>("dropped_d", grid(2, 20, 40.0, 10.0, 0, 200.0, 0.1, 900));
    std::printf("%d bad\n", bad);
    return bad != 0;
}
