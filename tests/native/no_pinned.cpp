// Realizations in a process that is refused pinned host memory of any size
// worth the name: this program's own hipHostMalloc takes the place of the
// runtime's and passes small requests on.
//   usage: no_pinned <1: refuse, 0: pass everything on>   prints a hash per field
#include <dlfcn.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include <hip/hip_runtime.h>

#include "scarf3d.h"
#include "scarf3d_srm.h"

static bool refuse = false;
static int refused = 0;

extern "C" __attribute__((visibility("default"))) hipError_t hipHostMalloc(void **ptr, size_t bytes, unsigned int flags)
{
    using Call = hipError_t (*)(void **, size_t, unsigned int);
    static const Call next = reinterpret_cast<Call>(dlsym(RTLD_NEXT, "hipHostMalloc"));
    if (refuse && bytes > 1024) {
        ++refused;
        *ptr = nullptr;
        return hipErrorOutOfMemory;
    }
    return next(ptr, bytes, flags);
}

namespace {

int bad = 0;

void tell(const char *what, const std::vector<real> &f, const char *err)
{
    uint64_t h = 1469598103934665603ull;
    const unsigned char *b = reinterpret_cast<const unsigned char *>(f.data());
    for (size_t i = 0; i < f.size() * sizeof(real); ++i) h = (h ^ b[i]) * 1099511628211ull;
    double s = 0;
    for (real v : f) s += double(v) * v;
    std::printf("%s: %016llx %s\n", what, static_cast<unsigned long long>(h), *err ? err : s > 0 ? "field" : "no field");
    std::fflush(stdout);
    bad += *err != 0 || !(s > 0);
}

void grid(const char *what, const int (&n)[3], int method, int nharm, int kernel)
{
    scarf_opt o;
    scarf_opt_init(&o);
    o.method = method;
    o.hurst = real(0.3);
    const int fs[3] = {1, 1, 1};
    const real cl[3] = {300, 250, 200};
    std::vector<real> field(size_t(n[0]) * n[1] * n[2], real(0));
    real stats[8];
    scarf_cart_initialize(3, fs, n, real(50), 0, cl, real(0.05), &o);
    scarf_set_nharm(nharm);
    scarf_set_kernel(kernel);
    scarf_execute(7, field.data(), stats);
    tell(what, field, scarf_last_error());
    scarf_finalize();
}

void points(const char *what, int method, int nharm)
{
    scarf_opt o;
    scarf_opt_init(&o);
    o.method = method;
    o.hurst = real(0.3);
    const int n = 20000;
    std::vector<real> p[3], field(n, real(0));
    for (int q = 0; q < 3; ++q)
        for (int i = 0; i < n; ++i) p[q].push_back(real((i * (7919LL + 104 * q) % 20011) * (0.1 - 0.02 * q)));
    const real cl[3] = {300, 250, 200};
    real stats[8];
    scarf_nocart_initialize(3, n, p[0].data(), p[1].data(), p[2].data(), real(40), 0, cl, real(0.05), &o);
    scarf_set_nharm(nharm);
    scarf_set_kernel(SCARF_KERNEL_AUTO);
    scarf_execute(3, field.data(), stats);
    tell(what, field, scarf_last_error());
    scarf_finalize();
}

void ensemble(const char *what, int nharm)
{
    std::vector<scarf_member> members(4);
    std::vector<real *> fields;
    std::vector<size_t> count;
    for (size_t m = 0; m < members.size(); ++m) {
        scarf_member &s = members[m];
        std::memset(&s, 0, sizeof s);
        s.nd = 3;
        for (int q = 0; q < 3; ++q) {
            s.fs[q] = 1;
            s.fe[q] = 40 + 3 * int(m) - 5 * q;
            s.cl[q] = real(300 - 50 * q);
        }
        s.ds = 50;
        s.hurst = real(0.3);
        s.sigma = real(0.05);
        s.nharm = nharm + 64 * int(m);
        s.seed = int(m) + 1;
        count.push_back(size_t(s.fe[0]) * s.fe[1] * s.fe[2]);
        void *ptr = nullptr;
        if (hipMalloc(&ptr, count.back() * sizeof(real)) != hipSuccess) std::exit(2);
        fields.push_back(static_cast<real *>(ptr));
    }
    std::vector<real> stats(8 * members.size());
    const int rc = scarf_ensemble_execute(int(members.size()), members.data(), fields.data(), stats.data(), 0);
    for (size_t m = 0; m < members.size(); ++m) {
        std::vector<real> f(count[m], real(0));
        if (rc == 0 && hipMemcpy(f.data(), fields[m], count[m] * sizeof(real), hipMemcpyDeviceToHost) != hipSuccess)
            std::exit(2);
        tell(what, f, rc == 0 ? "" : scarf_last_error());
    }
}

}  // namespace

int main(int argc, char **argv)
{
    refuse = argc > 1 && std::atoi(argv[1]) != 0;
    grid("grid", {40, 30, 20}, 1, 2000, SCARF_KERNEL_AUTO);
    grid("grid of few harmonics", {40, 30, 20}, 1, 60, SCARF_KERNEL_AUTO);
    grid("streamed draw", {64, 40, 12}, 1, 3000, SCARF_KERNEL_MFMA_BF16X3);
    grid("large field", {170, 150, 120}, 1, 1500, SCARF_KERNEL_AUTO);
    points("points", 1, 1900);
    points("points again", 1, 1900);
    points("fim points", 0, 1);
    grid("fim", {33, 37, 45}, 0, 1, SCARF_KERNEL_AUTO);
    ensemble("ensemble", 1500);
    ensemble("ensemble of few harmonics", 64);
    std::fprintf(stderr, "%d refused\n", refused);
    if (refuse && refused == 0) ++bad;
    return bad != 0;
}
