// Point-list SRM through a grid (see srm_points.hpp).
#include "srm_points.hpp"

#include <algorithm>
#include <cmath>

#include "kaiser_bessel.hpp"
#include "srm_stats.hpp"

namespace scarf {
namespace {

constexpr double kPi = 3.14159265358979323846;
// taps and oversampling of the interpolated grid: kernel errors of 2e-8 and
// 1e-15 of the field. FP64 lists keep what the roundings of the phases and
// positions leave out, as the transform does: 2000 points x 250 harmonics
// 3.2e-15 in the 2-norm, 50000 x 4000 3.1e-15 (6.6e-15 and 6.0e-15 without; the
// direct FP64 sum 3.3e-15 and 3.6e-15)
template <class Real>
constexpr int kTaps = sizeof(Real) == 4 ? 8 : 16;
constexpr double oversampling(bool f64) { return f64 ? 2.0 : 2.5; }
template <class Real>
constexpr int kTerms = sizeof(Real) == 4 ? 40 : 60;  // of I0 for their beta
constexpr int kMomentBlocks = 1024;

struct GridArgs {
    double h[3], x0[3], ih[3], beta;
    int n[3];
    int flat;
    int bin, bins[3];
};

// The record for the grid: wavenumbers per cell, phases at the grid's origin,
// amplitudes over the kernel's transform.
template <class Real>
__global__ __launch_bounds__(256) void points_record(const double *__restrict__ harm, double *__restrict__ out, int np_,
                                                     GridArgs a)
{
    constexpr int W = kTaps<Real>;
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= np_) return;
    double phase = harm[3 * long(np_) + n], amp = harm[4 * long(np_) + n];
    Turns at = turns(phase, 1.0);
    for (int d = 0; d < 3; ++d) {
        const double w = harm[d * long(np_) + n], t = w * a.h[d];
        out[d * long(np_) + n] = t;
        if constexpr (sizeof(Real) == 8) {
            const Turns more = turns(w, a.x0[d]);
            at.hi += more.hi;
            at.hi -= rint(at.hi);
            at.lo += more.lo;
            phase = 2.0 * kPi * (at.hi + at.lo);
        } else {
            phase += w * a.x0[d];
        }
        if (d < 2 || !a.flat) amp *= kaiser_bessel_inverse(t, W, a.beta);
    }
    out[3 * long(np_) + n] = phase;
    out[4 * long(np_) + n] = amp;
}

// first tap of coordinate u (cells from the origin), inside the grid also for
// a coordinate that is not a number
template <int W>
__device__ inline int first_tap(double u, int n)
{
    return min(max(int(ceil(u - 0.5 * W)), 0), n - W);
}

template <class Real>
__device__ inline long bin_of(const GridArgs &a, const double *__restrict__ pts, long npts, long i)
{
    constexpr int W = kTaps<Real>;
    int b[3];
    for (int d = 0; d < 3; ++d)
        b[d] = d == 2 && a.flat ? 0 : first_tap<W>((pts[d * npts + i] - a.x0[d]) * a.ih[d], a.n[d]) / a.bin;
    return (long(b[2]) * a.bins[1] + b[1]) * a.bins[0] + b[0];
}

__global__ __launch_bounds__(256) void points_clear(int *__restrict__ count, long n)
{
    for (long q = blockIdx.x * 256L + threadIdx.x; q < n; q += gridDim.x * 256L) count[q] = 0;
}

template <class Real>
__global__ __launch_bounds__(256) void points_count(GridArgs a, const double *__restrict__ pts, long npts,
                                                    int *__restrict__ count)
{
    for (long i = blockIdx.x * 256L + threadIdx.x; i < npts; i += gridDim.x * 256L)
        atomicAdd(&count[bin_of<Real>(a, pts, npts, i)], 1);
}

// counts to first places, in one block
__global__ __launch_bounds__(1024) void points_scan(int *__restrict__ count, long n)
{
    __shared__ int sums[16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int running = 0;
    constexpr int V = 8;  // bins per thread and round
    for (long q0 = 0; q0 < n; q0 += 1024 * V) {
        const long q = q0 + threadIdx.x * long(V);
        int c[V], tot = 0;
#pragma unroll
        for (int v = 0; v < V; ++v) {
            c[v] = q + v < n ? count[q + v] : 0;
            tot += c[v];
        }
        int inc = tot;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int o = __shfl_up(inc, off);
            if (lane >= off) inc += o;
        }
        __syncthreads();
        if (lane == 63) sums[wave] = inc;
        __syncthreads();
        int at = running + inc - tot;
        for (int w = 0; w < 16; ++w) {
            if (w < wave) at += sums[w];
            running += sums[w];
        }
#pragma unroll
        for (int v = 0; v < V; ++v)
            if (q + v < n) {
                count[q + v] = at;
                at += c[v];
            }
    }
}

// The order within a bin is whatever the atomics give: every point's value is
// its own.
template <class Real>
__global__ __launch_bounds__(256) void points_order(GridArgs a, const double *__restrict__ pts, long npts,
                                                    int *__restrict__ count, int *__restrict__ perm)
{
    for (long i = blockIdx.x * 256L + threadIdx.x; i < npts; i += gridDim.x * 256L)
        perm[atomicAdd(&count[bin_of<Real>(a, pts, npts, i)], 1)] = int(i);
}

// W lanes per point, one per tap: a lane evaluates its tap of each axis and
// walks the W x W rows at its column, so that a load reads the W consecutive
// values of 64 / W rows. Bound by the vector memory pipe (double: 17 clocks
// for a load's four unaligned 128-byte rows): 2M points take 0.29 ms in float
// and 3.5 ms in double. A thread per point, 64 unrelated addresses to a load,
// took 0.31 and, with 14 taps, two thirds of the products, 3.8 ms. Visited by
// bins, points share lines and the grid is read from HBM about once.
template <class Real>
__global__ __launch_bounds__(kPointsThreads) void points_interpolate(GridArgs a, const Real *__restrict__ grid,
                                                                     const double *__restrict__ pts, long first,
                                                                     long npts, const int *__restrict__ perm,
                                                                     Real *__restrict__ field)
{
    constexpr int W = kTaps<Real>;
    const int tap = threadIdx.x % W;
    const long s = first + blockIdx.x * long(kPointsThreads / W) + threadIdx.x / W;
    const long i = s < npts ? (perm ? perm[s] : s) : 0;  // spare lanes repeat a point
    const double e_beta = exp(-a.beta);
    double t[3] = {1.0, 1.0, 1.0};
    int k[3] = {0, 0, 0};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if (d == 2 && a.flat) break;
        const double x = pts[d * npts + i], dx = x - a.x0[d], u = dx * a.ih[d];
        double rest = 0.0;  // what u leaves out
        if constexpr (sizeof(Real) == 8) {
#pragma clang fp contract(off)
            const double minus = dx - x, lost = (x - (dx - minus)) - (a.x0[d] + minus);  // of dx
            rest = (fma(-u, a.h[d], dx) + lost) * a.ih[d];
        }
        k[d] = first_tap<W>(u, a.n[d]);
        t[d] = kaiser_bessel<kTerms<Real>, sizeof(Real) == 8>(k[d] + tap - u - rest, W, a.beta, e_beta);
        if (u != u) t[d] = u;  // not a number: neither is the value
    }
    Real ty[W];
#pragma unroll
    for (int q = 0; q < W; ++q) ty[q] = static_cast<Real>(__shfl(t[1], q, W));
    double sum = 0.0;
    const int planes = a.flat ? 1 : W;
    const Real *g = grid + (size_t(k[2]) * a.n[1] + k[1]) * a.n[0] + k[0] + tap;
    for (int z = 0; z < planes; ++z, g += size_t(a.n[0]) * a.n[1]) {
        Real v[W], p = Real(0);
#pragma unroll
        for (int q = 0; q < W; ++q) v[q] = g[size_t(q) * a.n[0]];
#pragma unroll
        for (int q = 0; q < W; ++q) p = fma(v[q], ty[q], p);
        sum = fma(static_cast<double>(p), a.flat ? 1.0 : __shfl(t[2], z, W), sum);
    }
    sum *= t[0];
#pragma unroll
    for (int off = W / 2; off >= 1; off >>= 1) sum += __shfl_xor(sum, off, W);
    if (tap == 0 && s < npts) field[i] = static_cast<Real>(sum);
}

// moments of the values in the caller's order, about each thread's first
template <class Real>
__global__ __launch_bounds__(256) void points_moments(const Real *__restrict__ v, long n, double *__restrict__ part)
{
    const long stride = gridDim.x * 256L, first = blockIdx.x * 256L + threadIdx.x;
    double s1 = 0.0, s2 = 0.0, cnt = 0.0;
    const double pivot = first < n ? static_cast<double>(v[first]) : 0.0;
    for (long i = first; i < n; i += stride) {
        const double d = static_cast<double>(v[i]) - pivot;
        s1 += d;
        s2 = fma(d, d, s2);
        cnt += 1.0;
    }
    Moments m{cnt, 0.0, 0.0};
    if (cnt > 0.0) {
        m.mean = pivot + s1 / cnt;
        m.m2 = s2 - s1 * (s1 / cnt);
    }
    block_moments(m, part + 3 * blockIdx.x);
}

}  // namespace

std::vector<PointsLaunch> points_launches(long npts, bool f64)
{
    const long per_block = kPointsThreads / (f64 ? kTaps<double> : kTaps<float>);
    std::vector<PointsLaunch> out;
    for (long first = 0; first < npts; first += kPointsBlocks * per_block)
        out.push_back({first, static_cast<unsigned>(std::min(kPointsBlocks, (npts - first + per_block - 1) / per_block))});
    return out;
}

bool points_plan(const double lo[3], const double hi[3], const double wmax[3], bool flat, long npts, int np_, bool f64,
                 PointsPlan &p)
{
    p = PointsPlan{};
    const size_t size = f64 ? 8 : 4;
    p.w = f64 ? kTaps<double> : kTaps<float>;
    const double over = oversampling(f64);
    p.beta = 0.995 * kPi * p.w * (1.0 - 0.5 / over);
    p.flat = flat;
    p.npts = npts;
    p.np_ = np_;
    if (npts < 1 || npts > 0x7fffffffL) return false;
    int n[3] = {1, 1, 1};
    double cells = 1.0;
    for (int d = 0; d < (flat ? 2 : 3); ++d) {
        const double span = hi[d] - lo[d];
        if (!std::isfinite(span) || !(span >= 0.0) || !std::isfinite(wmax[d])) return false;
        p.h[d] = wmax[d] > 0.0 ? kPi / (over * wmax[d]) : std::max(span, 1.0);
        const double steps = std::ceil(span / p.h[d]);
        if (!(steps < 16384.0)) return false;
        // a step to spare on both sides: a coordinate's rounding stays inside
        n[d] = static_cast<int>(steps) + p.w + 3;
        p.x0[d] = lo[d] - (p.w / 2 + 1) * p.h[d];
        cells *= n[d];
    }
    if (cells * size > double(size_t(16) << 30)) return false;
    p.g.nx = n[0];
    p.g.ny = n[1];
    p.g.nz = n[2];
    p.g.ds = 1.0;
    if (!transform_plan(p.g, np_, f64, p.grid)) return false;
    // a grid that stays in the L2s needs no order
    p.sorted = cells * size > double(1 << 20) && npts >= 4096;
    // bins of 16, 8 or 4 cells a side: few points share a counter
    long bins = 0;
    for (p.bin = 16; p.bin >= 4; p.bin /= 2) {
        bins = 1;
        for (int d = 0; d < 3; ++d) {
            p.bins[d] = (n[d] + p.bin - 1) / p.bin;
            bins *= p.bins[d];
        }
        if (p.bin == 4 || bins >= npts / 64) break;
    }
    p.nparts = static_cast<int>(std::min<long>((npts + 255) / 256, kMomentBlocks));
    size_t at = 0;
    auto take = [&](size_t bytes) {
        const size_t o = at;
        at += (bytes + 255) / 256 * 256;
        return o;
    };
    p.o_grid = take(size_t(cells) * size);
    p.o_record = take(size_t(5) * np_ * sizeof(double));
    p.o_work = take(p.grid.bytes);
    p.o_part = take(size_t(3) * (p.grid.nparts + p.grid.groups) * sizeof(double));
    p.o_count = take(size_t(bins) * sizeof(int));
    p.o_perm = take(p.sorted ? size_t(npts) * sizeof(int) : 0);
    p.bytes = at;
    return true;
}

// Fits to measured times. The harmonics fill 1 / oversampling of the grid's
// frequency columns, the others are skipped. The direct sum of a few points is
// bound by its chain over the harmonics (500 points x 3000: 0.31 ms in float,
// 0.11 this way; x 300 0.053 against 0.088).
double points_ms(const PointsPlan &p, bool f64)
{
    const double share = 0.35 + 0.65 / oversampling(f64);
    return 0.05 + share * transform_ms(p.grid, f64) + p.npts * (f64 ? 1.8e-6 : 3.5e-7);
}

double points_direct_ms(long npts, int np_, bool f64)
{
    return 0.025 + double(np_) * (f64 ? std::max(4.1e-4, npts / 7.5e8) : std::max(9.8e-5, npts / 4e9));
}

template <class Real>
bool points_field(const PointsPlan &p, const double *d_pts, const double *d_harm, void *ws, double scaling,
                  Real *d_field, double *d_part, hipStream_t stream, hipEvent_t tables_done, std::string &err)
{
    auto ok = [&](hipError_t e, const char *what) {
        if (e == hipSuccess) return true;
        err = std::string(what) + ": " + hipGetErrorString(e);
        return false;
    };
    char *base = static_cast<char *>(ws);
    GridArgs a{};
    const int n[3] = {p.g.nx, p.g.ny, p.g.nz};
    for (int d = 0; d < 3; ++d) {
        a.h[d] = p.h[d];
        a.ih[d] = 1.0 / p.h[d];
        a.x0[d] = p.x0[d];
        a.n[d] = n[d];
        a.bins[d] = p.bins[d];
    }
    a.beta = p.beta;
    a.flat = p.flat ? 1 : 0;
    a.bin = p.bin;
    Real *grid = reinterpret_cast<Real *>(base + p.o_grid);
    double *record = reinterpret_cast<double *>(base + p.o_record);
    int *count = reinterpret_cast<int *>(base + p.o_count);
    int *perm = p.sorted ? reinterpret_cast<int *>(base + p.o_perm) : nullptr;
    points_record<Real><<<(p.np_ + 255) / 256, 256, 0, stream>>>(d_harm, record, p.np_, a);
    if (!ok(hipGetLastError(), "points_record")) return false;
    if (!transform_field<Real>(p.grid, p.g, record, base + p.o_work, scaling, grid,
                               reinterpret_cast<double *>(base + p.o_part), stream, tables_done, err))
        return false;
    const int blocks = static_cast<int>(std::min<long>((p.npts + 255) / 256, 4096));
    if (perm) {
        const long bins = long(p.bins[0]) * p.bins[1] * p.bins[2];
        points_clear<<<int(std::min<long>((bins + 255) / 256, 1024)), 256, 0, stream>>>(count, bins);
        points_count<Real><<<blocks, 256, 0, stream>>>(a, d_pts, p.npts, count);
        points_scan<<<1, 1024, 0, stream>>>(count, bins);
        points_order<Real><<<blocks, 256, 0, stream>>>(a, d_pts, p.npts, count, perm);
        if (!ok(hipGetLastError(), "points_order")) return false;
    }
    for (const PointsLaunch &l : points_launches(p.npts, sizeof(Real) == sizeof(double))) {
        points_interpolate<Real><<<l.blocks, kPointsThreads, 0, stream>>>(a, grid, d_pts, l.first, p.npts, perm, d_field);
        if (!ok(hipGetLastError(), "points_interpolate")) return false;
    }
    points_moments<Real><<<p.nparts, 256, 0, stream>>>(d_field, p.npts, d_part);
    return ok(hipGetLastError(), "points_moments");
}

template bool points_field<float>(const PointsPlan &, const double *, const double *, void *, double, float *, double *,
                                  hipStream_t, hipEvent_t, std::string &);
template bool points_field<double>(const PointsPlan &, const double *, const double *, void *, double, double *, double *,
                                   hipStream_t, hipEvent_t, std::string &);

}  // namespace scarf
