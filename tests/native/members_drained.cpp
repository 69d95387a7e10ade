// Device::run_members ends with no work in flight when a member's draw throws,
// fails, or brings more harmonics than its plan holds, while the members before
// it run; the next call is whole again.
#include <cstdio>
#include <stdexcept>
#include <string>
#include <vector>

#include <hip/hip_runtime.h>

#include "srm_device.hpp"

int main()
{
    using namespace scarf;
    Device dev;
    std::string err;
    if (!dev.ensure(err)) {
        std::printf("%s\n", err.c_str());
        return 2;
    }
    const int nharm = 20000, count = 3;
    std::vector<double> w(nharm), amp(nharm, 1.0), zero(nharm + 64, 0.0);
    for (int l = 0; l < nharm; ++l) w[l] = 1e-3 * (1 + l % 97);
    std::vector<Device::Member> members(count);
    for (Device::Member &m : members) {
        m.g.structured = true;
        m.g.nx = m.g.ny = 512;
        m.g.nz = 256;
        m.g.ds = 10.0;
        m.nharm = nharm;
        m.scaling = 1.0;
        m.sigma = 1.0;
        if (hipMalloc(&m.d_field, size_t(512) * 512 * 256 * sizeof(float)) != hipSuccess) return 2;
    }
    if (!dev.reserve_members<float>(members)) return 2;
    int bad = 0;
    double st0 = 0;
    for (const char *how : {"whole", "throws", "fails", "too many", "whole again"}) {
        const std::string h = how;
        const bool whole = h[0] == 'w';
        const Device::MemberDraw draw = [&](int m, HarmonicRows &rows, std::string &e) {
            rows.field[0] = rows.field[1] = rows.field[2] = w.data();
            rows.field[3] = zero.data();
            rows.field[4] = amp.data();
            rows.n = nharm;
            if (m < 2 || whole) return true;
            if (h == "throws") throw std::bad_alloc();
            if (h == "too many") {
                for (const double *&f : rows.field) f = zero.data();
                rows.n = nharm + 1;
                return true;
            }
            e = "no draw";
            return false;
        };
        std::vector<double> stats;
        double ms = 0;
        bool ran = false;
        try {
            ran = dev.run_members<float>(members, draw, stats, ms, err);
        } catch (const std::bad_alloc &) {
        }
        const hipError_t left = hipStreamQuery(dev.stream());
        if (h == "whole") st0 = stats[2];
        const bool ok = ran == whole && left == hipSuccess && (!whole || (stats.size() == 6 * count && stats[2] == st0));
        std::printf("%s: %s, %s\n", how, ran ? "ran" : "ended", hipGetErrorString(left));
        bad += !ok;
    }
    std::printf("%d bad\n", bad);
    return bad != 0;
}
