// A device that is full but for 64 KiB when an ensemble, a tile timing or an
// FFT plan asks for its buffers, while the library keeps workspaces of calls
// before: this program's own hipMalloc and hipFree count, and refuse what the
// room would not hold.
//   usage: full_device <1: full, 0: room for everything>   prints a hash per field
#include <dlfcn.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

#include <hip/hip_runtime.h>

#include "scarf3d.h"
#include "scarf3d_srm.h"

static std::mutex guard;
static std::map<void *, size_t> sizes;
static size_t live = 0, room = ~size_t(0);
static int refused = 0;

extern "C" __attribute__((visibility("default"))) hipError_t hipMalloc(void **ptr, size_t bytes)
{
    using Call = hipError_t (*)(void **, size_t);
    static const Call next = reinterpret_cast<Call>(dlsym(RTLD_NEXT, "hipMalloc"));
    std::lock_guard<std::mutex> lock(guard);
    if (bytes > room || live > room - bytes) {
        ++refused;
        *ptr = nullptr;
        return hipErrorOutOfMemory;
    }
    const hipError_t e = next(ptr, bytes);
    if (e == hipSuccess) {
        sizes[*ptr] = bytes;
        live += bytes;
    }
    return e;
}

extern "C" __attribute__((visibility("default"))) hipError_t hipFree(void *ptr)
{
    using Call = hipError_t (*)(void *);
    static const Call next = reinterpret_cast<Call>(dlsym(RTLD_NEXT, "hipFree"));
    std::lock_guard<std::mutex> lock(guard);
    const auto it = sizes.find(ptr);
    if (it != sizes.end()) {
        live -= it->second;
        sizes.erase(it);
    }
    return next(ptr);
}

namespace {

int bad = 0;
bool full = false;

void fill_device() { room = full ? live + (size_t(64) << 10) : ~size_t(0); }
void empty_device() { room = ~size_t(0); }

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

void grid(const char *what, const int (&n)[3], int method, int kernel, bool in_full)
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
    scarf_set_nharm(2000);
    scarf_set_kernel(kernel);
    if (in_full) fill_device();
    scarf_execute(7, field.data(), stats);
    empty_device();
    tell(what, field, scarf_last_error());
    scarf_finalize();
}

// a workspace of 137 MB (float) that the library keeps; the tile timing of an
// ensemble takes 105 MB
void keep_workspace() { grid("grid", {512, 512, 90}, 1, SCARF_KERNEL_AUTO, false); }

void ensemble()
{
    scarf_member members[2];
    real *fields[2];
    const size_t count = size_t(160) * 90 * 60;
    for (int m = 0; m < 2; ++m) {
        scarf_member &s = members[m];
        std::memset(&s, 0, sizeof s);
        s.nd = 3;
        const int fe[3] = {160, 90, 60};
        for (int q = 0; q < 3; ++q) {
            s.fs[q] = 1;
            s.fe[q] = fe[q];
            s.cl[q] = real(300 - 50 * q);
        }
        s.ds = 50;
        s.hurst = real(0.3);
        s.sigma = real(0.05);
        s.nharm = 1500;
        s.seed = m + 1;
        void *ptr = nullptr;
        if (hipMalloc(&ptr, count * sizeof(real)) != hipSuccess) std::exit(2);
        fields[m] = static_cast<real *>(ptr);
    }
    real stats[16];
    fill_device();
    const int rc = scarf_ensemble_execute(2, members, fields, stats, SCARF_KERNEL_MFMA_BF16X3);
    empty_device();
    for (int m = 0; m < 2; ++m) {
        std::vector<real> f(count, real(0));
        if (rc == 0 && hipMemcpy(f.data(), fields[m], count * sizeof(real), hipMemcpyDeviceToHost) != hipSuccess)
            std::exit(2);
        tell("ensemble", f, rc == 0 ? "" : scarf_last_error());
        (void)hipFree(fields[m]);
    }
}

}  // namespace

int main(int argc, char **argv)
{
    full = argc > 1 && std::atoi(argv[1]) != 0;
    keep_workspace();
    ensemble();
    if (sizeof(real) == 4) {  // the named grid kernels are the float library's
        keep_workspace();
        grid("timed tiles", {150, 140, 130}, 1, SCARF_KERNEL_MFMA_BF16X3, true);
    }
    grid("fim", {148, 158, 166}, 0, SCARF_KERNEL_AUTO, false);
    keep_workspace();
    grid("fim of another size", {142, 138, 148}, 0, SCARF_KERNEL_AUTO, true);
    std::fprintf(stderr, "%d refused\n", refused);
    if (full && refused == 0) ++bad;
    return bad != 0;
}
