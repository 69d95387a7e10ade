// Plane-wise fast transform of the structured-grid SRM (see srm_transform.hpp).
//
// With tx = wx ds / 2 pi and ty = wy ds / 2 pi (turns per grid step, reduced to
// [-1/2, 1/2]; a harmonic with tx < 0 is replaced by its conjugate, whose real
// part is the same), one plane's steps are
//   spread     b(kx, ky) = sum_n phi(kx - tx Nx) phi(ky - ty Ny) c_n(z), kx in
//              [-w/2, Nx/2 + w/2), ky modulo Ny
//   y pass     transform over ky, the ny kept outputs divided by phi^(y): T
//   x pass     columns outside 0 .. Nx/2 folded onto their conjugates, real
//              transform over kx, the nx kept outputs divided by phi^(x)
// with Nx, Ny at least 1.9 times nx, ny and w = 9 (float) or 16 (double) taps
// of the Kaiser-Bessel kernel: kernel errors of 2e-8 and 1e-14 of the field.
#include "srm_transform.hpp"

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <type_traits>

#include "fft_lds.hpp"
#include "kaiser_bessel.hpp"
#include "srm_stats.hpp"

namespace scarf {
namespace {

using fft::Cplx;

constexpr double kInvTwoPi = 0.15915494309189533577;
constexpr double kPiD = 3.14159265358979323846;
constexpr int kThreads = 512;
constexpr size_t kLineBytes = 64 << 10;  // lines of a block (unpadded): two blocks per CU
constexpr double kMinOversampling = 1.9;

typedef double f64x4 __attribute__((ext_vector_type(4)));

// Everything the kernels need besides the record and the output.
template <class Real>
struct Args {
    int w, nx, ny, nz, m, l, columns, np_;
    int ox, oy, oz;
    double ds, beta_x, beta_y, scaling;
    int px, rx[6], py, ry[6];
    int zb, yb, nzb, slab, z0, zn;  // zn: planes of this round
    unsigned *key;           // class of the first ky << 14 | first column; ~0: amplitude 0
    int *order, *start, *count;
    int *first;              // first column, from here on in sorted order
    double *tapx, *tapy;     // [np][w], [np][2 class widths] from the class' first ky on
    Cplx<Real> *twy, *twx, *twr;
    unsigned short *revy, *revx;
    Real *decy;
    double *decx;
    Cplx<Real> *wave, *t;
};

// Classes of the first ky: a class' harmonics reach two class widths of ky
// values, which is one 16-row matrix tile for 9 taps and two for 16.
template <class Real>
constexpr int kTiles = sizeof(Real) == 4 ? 1 : 2;
template <class Real>
constexpr int kClass = 8 * kTiles<Real>;

// first radix of the x pass: two of its butterflies live in registers, and two
// blocks per CU leave 128
template <class Real>
constexpr int kFirstX = sizeof(Real) == 4 ? 8 : 4;

// 1 / phi^ of output j of a transform of n frequencies
__device__ inline double deconvolution(int j, int n, int w, double beta)
{
    return kaiser_bessel_inverse(2.0 * kPiD * j / n, w, beta);
}

// One harmonic on the oversampled frequency grid: positions gx in [0, m], gy,
// and the first tap of each axis. flip: the conjugate is taken.
struct Placed {
    double gx, gy;
    int kx, ky;
    bool flip;
};
template <class Real>
__device__ inline Placed place(const Args<Real> &a, const double *__restrict__ harm, int n)
{
    double tx = harm[n] * a.ds * kInvTwoPi, ty = harm[a.np_ + n] * a.ds * kInvTwoPi;
    tx -= rint(tx);
    ty -= rint(ty);
    Placed p;
    p.flip = tx < 0.0;
    p.gx = (p.flip ? -tx : tx) * (2.0 * a.m);
    p.gy = (p.flip ? -ty : ty) * a.l;
    p.kx = int(ceil(p.gx - 0.5 * a.w));
    p.ky = int(ceil(p.gy - 0.5 * a.w));
    return p;
}

template <class Real>
__global__ __launch_bounds__(256) void transform_keys(Args<Real> a, const double *__restrict__ harm)
{
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n < a.columns) a.count[n] = 0;
    if (n >= a.np_) return;
    const Placed p = place(a, harm, n);
    const int col = min(max(p.kx + a.w / 2, 0), a.m), ky = p.ky < 0 ? p.ky + a.l : p.ky;
    a.key[n] = harm[4 * long(a.np_) + n] != 0.0 ? unsigned(ky / kClass<Real>) << 14 | unsigned(col) : ~0u;
}

// Harmonics ordered by (class, first column), ties in draw order: those of a
// class that touch column c are then one range, first columns c - w + 1 .. c.
// Block t orders class t by a stable counting sort (the draw order within a
// range keeps the sums the same on every run), each wave over its own
// contiguous share of the record; bound by the latency of its three scans of
// the keys, hence the many waves and the unrolled loads.
template <class Real>
__global__ __launch_bounds__(1024) void transform_order(Args<Real> a)
{
    extern __shared__ int hist[];  // [waves][m + 1]
    __shared__ int wave_sum[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, bins = a.m + 1;
    const int threads = blockDim.x, waves = threads >> 6;
    const unsigned cls = blockIdx.x;
    int *mine = hist + wave * bins;
    for (int q = tid; q < waves * bins; q += threads) hist[q] = 0;
    __syncthreads();
    const int share = ((a.np_ + waves - 1) / waves + 63) / 64 * 64;
    const int n0 = wave * share, n1 = min(a.np_, n0 + share);
    int below = 0;
    constexpr int U = 8;  // loads in flight per wave
    for (int b = n0 + lane; b < n1; b += 64 * U) {
        unsigned k[U];
#pragma unroll
        for (int u = 0; u < U; ++u) k[u] = b + 64 * u < n1 ? a.key[b + 64 * u] : ~0u;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            below += (k[u] >> 14) < cls;  // an absent harmonic is above every class
            if ((k[u] >> 14) == cls) atomicAdd(&mine[k[u] & 0x3fffu], 1);
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) below += __shfl_xor(below, off);
    if (lane == 0) wave_sum[wave] = below;
    __syncthreads();
    int running = 0;
    for (int q = 0; q < waves; ++q) running += wave_sum[q];
    int *start = a.start + long(cls) * (a.m + 2);
    for (int b0 = 0; b0 < bins; b0 += threads) {
        const int bin = b0 + tid;
        int tot = 0;
        if (bin < bins)
            for (int q = 0; q < waves; ++q) tot += hist[q * bins + bin];
        int inc = tot;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int o = __shfl_up(inc, off);
            if (lane >= off) inc += o;
        }
        __syncthreads();  // wave_sum has been read
        if (lane == 63) wave_sum[wave] = inc;
        __syncthreads();
        int at = running + inc - tot;
        for (int q = 0; q < waves; ++q) {
            if (q < wave) at += wave_sum[q];
            running += wave_sum[q];
        }
        if (bin < bins) {
            start[bin] = at;
            for (int q = 0; q < waves; ++q) {
                const int h = hist[q * bins + bin];
                hist[q * bins + bin] = at;
                at += h;
            }
            if (tot > 0)
                for (int c = bin; c < bin + a.w; ++c) a.count[c] = 1;  // every writer stores 1
        }
    }
    if (tid == 0) start[bins] = running;
    __syncthreads();
    volatile int *place = mine;  // this wave's own row
    for (int b = n0 + lane; b - lane < n1; b += 64 * U) {
        unsigned k[U];
#pragma unroll
        for (int u = 0; u < U; ++u) k[u] = b + 64 * u < n1 ? a.key[b + 64 * u] : ~0u;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            uint64_t left = __ballot((k[u] >> 14) == cls);
            while (left) {
                const unsigned key = __builtin_amdgcn_readlane(k[u], __ffsll(static_cast<unsigned long long>(left)) - 1);
                const uint64_t same = __ballot(k[u] == key);
                const int at = place[key & 0x3fffu];
                if (k[u] == key) a.order[at + __popcll(same & ((1ull << lane) - 1))] = b + 64 * u;
                __builtin_amdgcn_wave_barrier();
                if (lane == 0) place[key & 0x3fffu] = at + __popcll(same);
                __builtin_amdgcn_wave_barrier();
                left &= ~same;
            }
        }
    }
}

// c_n(z) of plane z of a round, harmonics in sorted order: wave[p][z]. Phases
// in FP64, about the centre of the block along x and y.
template <class Real>
__device__ inline void wave_item(const Args<Real> &a, const double *__restrict__ harm, long e)
{
    const int p = int(e / a.slab), z = int(e - long(p) * a.slab), n = a.order[p];
    const double wx = harm[n], wy = harm[a.np_ + n], wz = harm[2 * long(a.np_) + n];
    const double xc = double(a.ox + a.nx / 2) * a.ds, yc = double(a.oy + a.ny / 2) * a.ds;
    double t = (wz * (double(a.z0 + z + a.oz) * a.ds)) * kInvTwoPi +
               (wx * xc + wy * yc + harm[3 * long(a.np_) + n]) * kInvTwoPi;
    t -= rint(t);
    double tx = wx * a.ds * kInvTwoPi;
    tx -= rint(tx);
    double s, c;
    sincospi(tx < 0.0 ? -2.0 * t : 2.0 * t, &s, &c);
    const double amp = harm[4 * long(a.np_) + n];
    a.wave[e] = Cplx<Real>{static_cast<Real>(amp * c), static_cast<Real>(amp * s)};
}

template <class Real>
__global__ __launch_bounds__(256) void transform_waves(Args<Real> a, const double *__restrict__ harm)
{
    const long present = a.start[long(a.l / kClass<Real> - 1) * (a.m + 2) + a.m + 1];
    const long total = present * a.slab;
    for (long e = blockIdx.x * long(blockDim.x) + threadIdx.x; e < total; e += long(gridDim.x) * blockDim.x)
        wave_item(a, harm, e);
}

// Tables of one realization in sorted order, and the waves of the first
// round. Work items: waves; taps along y (the zeros around them included) and
// x, one each; first columns; twiddles, digit-reversed positions and
// deconvolution factors.
template <class Real>
__global__ __launch_bounds__(256) void transform_tables(Args<Real> a, const double *__restrict__ harm)
{
    constexpr int W = sizeof(Real) == 4 ? 9 : 16, K = sizeof(Real) == 4 ? 45 : 66, R = 2 * kClass<Real>;
    const long present = a.start[long(a.l / kClass<Real> - 1) * (a.m + 2) + a.m + 1];
    const long i0 = present * a.slab, i1 = i0 + present * R, i2 = i1 + present * W, i3 = i2 + present;
    const long total = i3 + a.l + 2 * long(a.m) + a.ny + a.nx;
    for (long e = blockIdx.x * long(blockDim.x) + threadIdx.x; e < total; e += long(gridDim.x) * blockDim.x) {
        if (e < i0) {
            wave_item(a, harm, e);
            continue;
        }
        if (e < i2) {
            const bool along_y = e < i1;
            const int p = int(along_y ? (e - i0) / R : (e - i1) / W);
            const Placed h = place(a, harm, a.order[p]);
            if (along_y) {
                const int ky = h.ky < 0 ? h.ky + a.l : h.ky;
                const int d = int((e - i0) % R) - ky % kClass<Real>;  // tap at the class' row
                a.tapy[e - i0] = d >= 0 && d < W ? kaiser_bessel<K>(h.ky + d - h.gy, W, a.beta_y, exp(-a.beta_y)) : 0.0;
            } else {
                a.tapx[e - i1] = kaiser_bessel<K>(h.kx + int((e - i1) % W) - h.gx, W, a.beta_x, exp(-a.beta_x));
            }
            continue;
        }
        if (e < i3) {
            a.first[e - i2] = int(a.key[a.order[e - i2]] & 0x3fffu);
            continue;
        }
        int r = int(e - i3);
        double s, c;
        if (r < a.l) {
            sincospi(2.0 * double(r) / a.l, &s, &c);
            a.twy[r] = Cplx<Real>{Real(c), Real(s)};
            a.revy[r] = static_cast<unsigned short>(fft::pad(fft::digit_reverse(r, a.l, a.py, a.ry)));
            continue;
        }
        r -= a.l;
        if (r < a.m) {
            sincospi(2.0 * double(r) / a.m, &s, &c);
            a.twx[r] = Cplx<Real>{Real(c), Real(s)};
            a.revx[r] = static_cast<unsigned short>(fft::pad(fft::digit_reverse(r, a.m, a.px, a.rx)));
            continue;
        }
        r -= a.m;
        if (r < a.m) {
            sincospi(double(r) / a.m, &s, &c);
            a.twr[r] = Cplx<Real>{Real(c), Real(s)};
            continue;
        }
        r -= a.m;
        if (r < a.ny) a.decy[r] = static_cast<Real>(deconvolution(r - a.ny / 2, a.l, W, a.beta_y));
        else if (r < a.ny + a.nx) a.decx[r - a.ny] = a.scaling * deconvolution(r - a.ny - a.nx / 2, 2 * a.m, W, a.beta_x);
    }
}

// LDS of the y pass behind the lines: partial sums of half the waves, the
// classes' ranges for the block's column and the digit-reversed positions.
constexpr int kYWaves = kThreads / 64;
template <class Real>
size_t lds_y_bytes(int zb, int l)
{
    const size_t classes = size_t(l) / kClass<Real>;
    return size_t(zb) * fft::pitch(l) * sizeof(Cplx<Real>) + 16 + size_t(kYWaves / 2) * 256 * sizeof(double) +
           classes * (sizeof(int2) + sizeof(unsigned short)) + size_t(l) * sizeof(unsigned short) + 16;
}

// Spread and y pass: one block per (kx column, zb planes). The spread is a
// product on the FP64 matrix cores: a class' 16-row tiles of ky, by (plane,
// re/im), summed over the class' harmonics that touch the column, four per
// instruction,
//   A[ky][p] = phi_y, B[p][z] = phi_x c_p(z),
// so the sums are FP64 in a fixed order for either field type. A class reaches
// the rows of the next one too: even classes, whose rows are disjoint, store
// their tiles over the cleared lines, then the odd ones add theirs. One wave takes a class, and all
// of them together one of kShared harmonics or more (most harmonics can sit in
// a few columns and classes: at a small correlation length per box nearly all
// do). Then the lines are transformed in LDS. Blocks of one z group follow
// each other nzb apart: with nzb = 8 each XCD's L2 holds one group's waves.
constexpr int kShared = 128;
template <class Real>
__global__ __launch_bounds__(kThreads, 4) void transform_y(Args<Real> a)
{
    constexpr int G = kTiles<Real>, CW = kClass<Real>, W = sizeof(Real) == 4 ? 9 : 16;
    extern __shared__ __align__(16) unsigned char smem[];
    const int zblk = blockIdx.x % a.nzb, col = blockIdx.x / a.nzb;
    if (!a.count[col]) return;  // the x pass takes this column as zero
    const int line = fft::pitch(a.l), classes = a.l / CW;
    Cplx<Real> *lds = reinterpret_cast<Cplx<Real> *>(smem);
    Real *flat = reinterpret_cast<Real *>(smem);
    double *slots = reinterpret_cast<double *>(smem + (size_t(a.zb) * line * sizeof(Cplx<Real>) + 15) / 16 * 16);
    int2 *range = reinterpret_cast<int2 *>(slots + (kYWaves / 2) * 256);
    unsigned short *shared_cls = reinterpret_cast<unsigned short *>(range + classes);
    unsigned short *rev = shared_cls + classes;
    __shared__ int nshared;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int jj = lane & 15, slot = lane >> 4;
    const int lo = max(0, col - W + 1), hi = min(col, a.m);
    const int zoff = zblk * a.zb;
    const bool mine = jj < 2 * a.zb;
    const Real *wv = reinterpret_cast<const Real *>(a.wave) + 2 * zoff + (mine ? jj : 0);
    if (tid == 0) nshared = 0;
    __syncthreads();
    for (int q = tid; q < classes; q += kThreads) {
        const int *st = a.start + long(q) * (a.m + 2);
        const int s0 = st[lo], n = st[hi + 1] - s0;
        range[q] = make_int2(s0, n);
        if (n >= kShared) shared_cls[atomicAdd(&nshared, 1)] = static_cast<unsigned short>(q);
    }
    for (int q = tid; q < a.l; q += kThreads) rev[q] = a.revy[q];
    const Cplx<Real> zero{Real(0), Real(0)};
    for (int q = tid; q < a.zb * line; q += kThreads) lds[q] = zero;
    __syncthreads();
    // A and B of this lane's harmonic i of a range (beyond it: a zero)
    auto load = [&](int s0, int n, int i, double &x, double &w, double (&y)[G]) __attribute__((always_inline)) {
        const long p = s0 + min(i, n - 1);
        x = a.tapx[p * W + (col - a.first[p])];
        w = static_cast<double>(wv[2 * p * a.slab]);
        x = i < n ? x : 0.0;
#pragma unroll
        for (int g = 0; g < G; ++g) y[g] = a.tapy[p * (16 * G) + 16 * g + jj];
    };
    // steps step, step + stride, ... of four harmonics each, added to acc; the
    // loads of U steps are issued together
    auto sum = [&](int s0, int n, int step, int stride, f64x4 (&acc)[G]) __attribute__((always_inline)) {
        auto steps = [&](int i0, auto count) __attribute__((always_inline)) {
            constexpr int U = decltype(count)::value;
            double x[U], w[U], y[U][G];
#pragma unroll
            for (int u = 0; u < U; ++u) load(s0, n, i0 + 4 * u * stride + slot, x[u], w[u], y[u]);
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int g = 0; g < G; ++g)
                    acc[g] = __builtin_amdgcn_mfma_f64_16x16x4f64(y[u][g], w[u] * x[u], acc[g], 0, 0, 0);
        };
        constexpr int U = 4;
        int i0 = 4 * step;
        for (; i0 + 4 * (U - 1) * stride < n; i0 += 4 * U * stride) steps(i0, std::integral_constant<int, U>{});
        for (; i0 < n; i0 += 4 * stride) steps(i0, std::integral_constant<int, 1>{});
    };
    auto put = [&](int q, bool add, const f64x4 (&acc)[G]) __attribute__((always_inline)) {
        if (!mine) return;
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                int ky = q * CW + 16 * g + 4 * r + slot;
                if (ky >= a.l) ky -= a.l;
                Real &v = flat[2 * ((jj >> 1) * line + rev[ky]) + (jj & 1)];
                v = static_cast<Real>(add ? static_cast<double>(v) + acc[g][r] : acc[g][r]);
            }
    };
    const int heavy = nshared;
    constexpr int B = 4 / G;
    for (int odd = 0; odd < 2; ++odd) {
        for (int q0 = 2 * wave + odd; q0 < classes; q0 += 2 * kYWaves * B) {
            // B classes at a time: most hold a few harmonics, and their loads overlap
            f64x4 acc[B][G];
            int s0[B], n[B];
            double x[B], w[B], y[B][G];
#pragma unroll
            for (int c = 0; c < B; ++c) {
                const int q = q0 + 2 * kYWaves * c;
                const int2 r = q < classes ? range[q] : make_int2(0, 0);
                s0[c] = __builtin_amdgcn_readfirstlane(r.x);
                n[c] = __builtin_amdgcn_readfirstlane(r.y);
                if (n[c] >= kShared) n[c] = -1;
                if (n[c] > 0) load(s0[c], n[c], slot, x[c], w[c], y[c]);
            }
#pragma unroll
            for (int c = 0; c < B; ++c) {
                const int q = q0 + 2 * kYWaves * c;
                if (n[c] <= 0) continue;
#pragma unroll
                for (int g = 0; g < G; ++g)
                    acc[c][g] = __builtin_amdgcn_mfma_f64_16x16x4f64(y[c][g], w[c] * x[c], f64x4{0.0, 0.0, 0.0, 0.0},
                                                                     0, 0, 0);
                sum(s0[c], n[c], 1, 1, acc[c]);
                put(q, odd, acc[c]);
            }
        }
        for (int h = 0; h < heavy; ++h) {
            const int q = __builtin_amdgcn_readfirstlane(shared_cls[h]);
            if ((q & 1) != odd) continue;
            const int s0 = __builtin_amdgcn_readfirstlane(range[q].x), n = __builtin_amdgcn_readfirstlane(range[q].y);
            f64x4 acc[G];
#pragma unroll
            for (int g = 0; g < G; ++g) acc[g] = f64x4{0.0, 0.0, 0.0, 0.0};
            sum(s0, n, wave, kYWaves, acc);
            for (int half = kYWaves / 2; half >= 1; half /= 2)
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    __syncthreads();
                    if (wave >= half && wave < 2 * half) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) slots[(wave - half) * 256 + 64 * r + lane] = acc[g][r];
                    }
                    __syncthreads();
                    if (wave < half) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[g][r] += slots[wave * 256 + 64 * r + lane];
                    }
                }
            if (wave == 0) put(q, odd, acc);
        }
        __syncthreads();
    }
    // the last pass' outputs leave the block: the ny kept ones, divided by phi^
    const int planes = min(a.zb, a.zn - zoff);
    Cplx<Real> *out = a.t + (size_t(zoff) * a.columns + col) * a.ny;
    const size_t plane = size_t(a.columns) * a.ny;
    fft::transform(lds, a.twy, a.l, 0, a.py, a.ry, line, a.zb, tid, kThreads,
                   [&](int z, int q, Cplx<Real> v) __attribute__((always_inline)) {
                       const int y = (2 * q < a.l ? q : q - a.l) + a.ny / 2;
                       if (z >= planes || y < 0 || y >= a.ny) return;
                       const Real d = a.decy[y];
                       out[z * plane + y] = Cplx<Real>{v.x * d, v.y * d};
                   });
}

// x pass: one block per (plane, yb lines). The real transform of 2m values is
// a complex one of m: Z_k = A + i e^(i pi k / m) D, Z_(m-k) = conj(A) + i
// conj(e^(i pi k / m) D) with A, D = H_k +- conj(H_(m-k)) and H the half
// spectrum (interior values halved: only the real part of the sum is kept).
// An item is the first butterflies, of radix R = kFirstX, of inputs b + r m/R
// and m/R - b + r m/R, which hold each other's partners (butterflies 0 and
// m/2R hold their own): T comes straight into registers, and the last pass
// stores the field from registers, scaled and rounded, with the statistics
// partials.
template <class Real>
__global__ __launch_bounds__(kThreads, 4) void transform_x(Args<Real> a, Real *__restrict__ field,
                                                                             double *__restrict__ part)
{
    extern __shared__ __align__(16) unsigned char smem[];
    using C = Cplx<Real>;
    C *lds = reinterpret_cast<C *>(smem);
    const int yblks = (a.ny + a.yb - 1) / a.yb;
    const int z = blockIdx.x / yblks, y0 = (blockIdx.x - z * yblks) * a.yb;
    const int tid = threadIdx.x, line = fft::pitch(a.m);
    const int lines = min(a.yb, a.ny - y0);
    const C *t = a.t + size_t(z) * a.columns * a.ny + y0;
    const int off = a.w / 2, above = a.w - 1 - a.w / 2;  // columns below 0 and above m
    constexpr int R = kFirstX<Real>;
    const int step = a.m / R;
    for (int e = tid; e < (step / 2) * a.yb; e += kThreads) {
        const int yy = e & (a.yb - 1), b = e / a.yb;
        if (yy >= lines) continue;
        auto at = [&](int kx) __attribute__((always_inline)) {
            return a.count[kx + off] ? t[size_t(kx + off) * a.ny + yy] : C{Real(0), Real(0)};
        };
        C p[R], q[R], pm{};
        const int bp = b, bq = b == 0 ? step / 2 : step - b;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            p[r] = at(bp + r * step);
            q[r] = at(bq + r * step);
        }
        if (b == 0) pm = at(a.m);
        // columns outside 0 .. m fold onto their conjugates
        auto fold = [&](C &v, int kx) __attribute__((always_inline)) {
            if (kx > 0 && kx <= off) {
                const C u = at(-kx);
                v = C{v.x + u.x, v.y - u.y};
            }
            if (a.m - kx <= above) {
                const C u = at(2 * a.m - kx);
                v = C{v.x + u.x, v.y - u.y};
            }
        };
#pragma unroll
        for (int r = 0; r < R; ++r) {
            fold(p[r], bp + r * step);
            fold(q[r], bq + r * step);
        }
        auto pair = [&](C &u, C &v, int k) __attribute__((always_inline)) {  // u = H_k, v = H_(m-k)
            const Real h = Real(0.5);
            const C s{h * (u.x + v.x), h * (u.y - v.y)};
            const C d = fft::mul(a.twr[k], C{h * (u.x - v.x), h * (u.y + v.y)});
            u = C{s.x - d.y, s.y + d.x};
            v = C{s.x + d.y, d.x - s.y};
        };
        if (b == 0) {
            p[0] = C{p[0].x + pm.x, p[0].x - pm.x};
#pragma unroll
            for (int r = 1; r < R / 2; ++r) pair(p[r], p[R - r], r * step);
            p[R / 2].y = -p[R / 2].y;  // k = m/2: its own partner, conj(H) with H not halved
#pragma unroll
            for (int r = 0; r < R / 2; ++r) pair(q[r], q[R - 1 - r], bq + r * step);
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r) pair(p[r], q[R - 1 - r], bp + r * step);
        }
        fft::dft<R>(p);
        fft::dft<R>(q);
        C *lp = lds + yy * line + a.revx[bp], *lq = lds + yy * line + a.revx[bq];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            lp[r] = p[r];
            lq[r] = q[r];
        }
    }
    // sums about the thread's first value: no cancellation whatever the mean
    double s1 = 0.0, s2 = 0.0, pivot = 0.0;
    int cnt = 0;
    Real *rows = field + (size_t(a.z0 + z) * a.ny + y0) * a.nx;
    fft::transform(lds, a.twx, a.m, 1, a.px, a.rx, line, a.yb, tid, kThreads,
                   [&](int yy, int q, C v) __attribute__((always_inline)) {
                       if (yy >= lines) return;
                       const int i = 2 * (2 * q < a.m ? q : q - a.m) + a.nx / 2;
                       const Real c[2] = {v.x, v.y};
#pragma unroll
                       for (int h = 0; h < 2; ++h) {
                           if (i + h < 0 || i + h >= a.nx) continue;
                           const Real o = static_cast<Real>(static_cast<double>(c[h]) * a.decx[i + h]);
                           rows[size_t(yy) * a.nx + i + h] = o;
                           if (cnt == 0) pivot = static_cast<double>(o);
                           const double d = static_cast<double>(o) - pivot;
                           s1 += d;
                           s2 = fma(d, d, s2);
                           ++cnt;
                       }
                   });
    Moments mo{double(cnt), 0.0, 0.0};
    if (cnt > 0) {
        mo.mean = pivot + s1 / cnt;
        mo.m2 = s2 - s1 * (s1 / cnt);
    }
    block_moments(mo, part + 3 * (size_t(a.z0 + z) * yblks + (blockIdx.x - z * yblks)));
}

// 256 partials to one, in a fixed order
__global__ __launch_bounds__(256) void transform_merge(const double *__restrict__ part, int nparts,
                                                       double *__restrict__ out)
{
    const long q = blockIdx.x * 256L + threadIdx.x;
    Moments m{0.0, 0.0, 0.0};
    if (q < nparts) m = Moments{part[3 * q], part[3 * q + 1], part[3 * q + 2]};
    block_moments(m, out + 3 * blockIdx.x);
}

// smallest length m * 2^a >= n with m in {1, 3, 5, 7, 9}, a multiple of 32
int good_length(double n)
{
    int best = 0;
    for (int m : {1, 3, 5, 7, 9}) {
        long v = 32L * m;
        while (double(v) < n) v *= 2;
        if (best == 0 || v < best) best = static_cast<int>(std::min<long>(v, 1 << 28));
    }
    return best;
}

FftPlan fft_plan(int n, int first)
{
    FftPlan p;
    p.n = n;
    p.passes = fft::plan(n, first, p.kind);
    return p;
}

}  // namespace

bool transform_plan(const Geometry &g, int np_, bool f64, TransformPlan &plan)
{
    plan = TransformPlan{};
    if (!g.structured || g.nx < 1 || g.ny < 1 || g.nz < 1 || g.nx > 8192 || g.ny > 8192) return false;
    TransformPlan &p = plan;
    const size_t csize = f64 ? 16 : 8;
    p.w = f64 ? 16 : 9;
    p.nx = g.nx;
    p.ny = g.ny;
    p.nz = g.nz;
    p.np_ = np_;
    const int fx = good_length(kMinOversampling * g.nx);
    p.m = fx / 2;
    p.l = good_length(kMinOversampling * g.ny);
    if (p.l * csize > kLineBytes || p.m * csize > kLineBytes) return false;
    p.columns = p.m + p.w;
    p.fx = fft_plan(p.m, f64 ? kFirstX<double> : kFirstX<float>);
    p.fy = fft_plan(p.l, 8);
    // Kaiser-Bessel shape for the axis' oversampling s (pi w (1 - 1/(2 s)), just inside)
    p.beta_x = 0.995 * kPiD * p.w * (1.0 - 0.5 * g.nx / fx);
    p.beta_y = 0.995 * kPiD * p.w * (1.0 - 0.5 * g.ny / p.l);
    p.zb = 8;
    while (p.zb > 1 && size_t(p.zb) * p.l * csize > kLineBytes) p.zb /= 2;
    while (p.zb > 1 && p.zb / 2 >= g.nz) p.zb /= 2;
    p.yb = 16;
    while (p.yb > 1 && size_t(p.yb) * p.m * csize > kLineBytes) p.yb /= 2;
    while (p.yb > 1 && p.yb / 2 >= g.ny) p.yb /= 2;
    // planes per round: eight blocks' worth, more while the intermediate stays small
    const size_t plane = size_t(p.columns) * p.ny * csize;
    const int zmax = (g.nz + p.zb - 1) / p.zb * p.zb;
    p.slab = 8 * p.zb;
    while (p.slab < zmax && plane * p.slab * 2 <= (size_t(192) << 20)) p.slab *= 2;
    p.slab = std::min(p.slab, zmax);
    // short lines: more of them per block, as long as the blocks still fill the device
    while (p.yb >= 16 && p.yb < 256 && 2 * p.yb * p.m <= 4096 && long(g.nz) * g.ny / (2 * p.yb) >= 1024) p.yb *= 2;
    const long yblks = (g.ny + p.yb - 1) / p.yb;
    if (yblks * g.nz > (1L << 28)) return false;
    p.nparts = static_cast<int>(yblks * g.nz);
    p.groups = (p.nparts + 255) / 256;

    size_t at = 0;
    auto take = [&](size_t bytes) {
        const size_t o = at;
        at += (bytes + 255) / 256 * 256;
        return o;
    };
    const size_t np = np_;
    const int cls = f64 ? kClass<double> : kClass<float>;
    p.o_key = take(np * sizeof(unsigned));
    p.o_first = take(np * sizeof(int));
    p.o_order = take(np * sizeof(int));
    p.o_start = take(size_t(p.l / cls) * (p.m + 2) * sizeof(int));
    p.o_count = take(size_t(p.columns) * sizeof(int));
    p.o_taps = take(np * (2 * cls + p.w) * sizeof(double));
    p.o_tw = take((size_t(p.l) + 2 * size_t(p.m)) * csize);
    p.o_rev = take((size_t(p.l) + p.m) * sizeof(unsigned short));
    p.o_dec = take((size_t(p.ny) + p.nx) * sizeof(double));
    p.o_wave = take(np * p.slab * csize);
    p.o_t = take(plane * p.slab);
    p.bytes = at;
    return true;
}

// Linear fits to measured times. Transform: the chain of small launches, the
// harmonics' tables and ordering, the cells of both passes (float 512^3: 2.7
// of 2.9 ms), their blocks, and the spread. The line between the two lies at
// a few hundred harmonics for FP32 grids (float, direct_f32: 64^3 x 256 0.065
// against 0.103 ms, x 64 0.058 against 0.045; bf16x3: 256^3 x 1024 0.36 against
// 0.36, x 4096 0.43 against 1.27) and below 64 for FP64 ones (64^3 x 64 0.069
// against 0.131 ms).
double transform_ms(const TransformPlan &p, bool f64)
{
    const double cells = double(p.columns) * p.l * p.nz;
    const double blocks = double(p.columns) * ((p.nz + p.zb - 1) / p.zb) + p.nparts;
    const double waves = double(p.np_) * p.nz;
    return f64 ? 0.05 + 1.2e-5 * p.np_ + 1.6e-8 * cells + 1.5e-5 * blocks + 8e-8 * waves
               : 0.05 + 8.5e-6 * p.np_ + 7.5e-9 * cells + 1.2e-5 * blocks + 3e-8 * waves;
}

// The direct kernels' points and harmonics per millisecond, and for those with
// one block per 4096 points the time of a harmonic in an underfilled device.
double direct_ms(const Geometry &g, int nharm, int kernel)
{
    const double pts = double(g.points());
    if (kernel == kKernelDirectF64) return 0.02 + nharm * std::max(1.6e-3, pts / 7.6e8);
    if (kernel == kKernelDirectF32) return 0.025 + nharm * std::max(3.05e-4, pts / 9.6e9);
    return 0.04 + nharm * (pts / 5.5e10);
}

template <class Real>
bool transform_field(const TransformPlan &p, const Geometry &g, const double *d_harm, void *ws, double scaling,
                     Real *d_field, double *d_part, hipStream_t stream, hipEvent_t tables_done, std::string &err)
{
    auto ok = [&](hipError_t e, const char *what) {
        if (e == hipSuccess) return true;
        err = std::string(what) + ": " + hipGetErrorString(e);
        return false;
    };
    char *base = static_cast<char *>(ws);
    Args<Real> a{};
    a.w = p.w;
    a.nx = p.nx;
    a.ny = p.ny;
    a.nz = p.nz;
    a.m = p.m;
    a.l = p.l;
    a.columns = p.columns;
    a.np_ = p.np_;
    a.ox = g.ox;
    a.oy = g.oy;
    a.oz = g.oz;
    a.ds = g.ds;
    a.beta_x = p.beta_x;
    a.beta_y = p.beta_y;
    a.scaling = scaling;
    a.px = p.fx.passes;
    a.py = p.fy.passes;
    for (int q = 0; q < 6; ++q) {
        a.rx[q] = p.fx.kind[q];
        a.ry[q] = p.fy.kind[q];
    }
    a.zb = p.zb;
    a.yb = p.yb;
    a.slab = p.slab;
    a.key = reinterpret_cast<unsigned *>(base + p.o_key);
    a.first = reinterpret_cast<int *>(base + p.o_first);
    a.order = reinterpret_cast<int *>(base + p.o_order);
    a.start = reinterpret_cast<int *>(base + p.o_start);
    a.count = reinterpret_cast<int *>(base + p.o_count);
    a.tapy = reinterpret_cast<double *>(base + p.o_taps);
    a.tapx = a.tapy + size_t(p.np_) * 2 * kClass<Real>;
    a.twy = reinterpret_cast<Cplx<Real> *>(base + p.o_tw);
    a.twx = a.twy + p.l;
    a.twr = a.twx + p.m;
    a.revy = reinterpret_cast<unsigned short *>(base + p.o_rev);
    a.revx = a.revy + p.l;
    a.decx = reinterpret_cast<double *>(base + p.o_dec);
    a.decy = reinterpret_cast<Real *>(a.decx + p.nx);
    a.wave = reinterpret_cast<Cplx<Real> *>(base + p.o_wave);
    a.t = reinterpret_cast<Cplx<Real> *>(base + p.o_t);

    transform_keys<Real><<<(std::max(p.np_, p.columns) + 255) / 256, 256, 0, stream>>>(a, d_harm);
    if (!ok(hipGetLastError(), "transform_keys")) return false;
    int sort_waves = 16;  // as many as their histograms fit in LDS
    while (size_t(sort_waves) * (p.m + 1) * sizeof(int) > (size_t(80) << 10)) sort_waves /= 2;
    transform_order<Real><<<p.l / kClass<Real>, 64 * sort_waves, size_t(sort_waves) * (p.m + 1) * sizeof(int), stream>>>(a);
    if (!ok(hipGetLastError(), "transform_order")) return false;
    a.zn = std::min(p.slab, p.nz);
    const long items = long(p.np_) * (p.slab + 2 * kClass<Real> + p.w + 1) + p.l + 2 * long(p.m) + p.ny + p.nx;
    transform_tables<Real><<<int(std::min<long>((items + 255) / 256, 65536)), 256, 0, stream>>>(a, d_harm);
    if (!ok(hipGetLastError(), "transform_tables")) return false;
    if (!ok(hipEventRecord(tables_done, stream), "hipEventRecord")) return false;
    const size_t lds_y = lds_y_bytes<Real>(p.zb, p.l);
    const size_t lds_x = size_t(p.yb) * fft::pitch(p.m) * sizeof(Cplx<Real>);
    const int yblks = (p.ny + p.yb - 1) / p.yb;
    for (int z0 = 0; z0 < p.nz; z0 += p.slab) {
        a.z0 = z0;
        a.zn = std::min(p.slab, p.nz - z0);
        a.nzb = (a.zn + p.zb - 1) / p.zb;
        const long waves = long(p.np_) * p.slab;
        if (z0 > 0) {
            transform_waves<Real><<<int(std::min<long>((waves + 255) / 256, 65536)), 256, 0, stream>>>(a, d_harm);
            if (!ok(hipGetLastError(), "transform_waves")) return false;
        }
        transform_y<Real><<<a.nzb * p.columns, kThreads, lds_y, stream>>>(a);
        if (!ok(hipGetLastError(), "transform_y")) return false;
        transform_x<Real><<<a.zn * yblks, kThreads, lds_x, stream>>>(a, d_field, d_part);
        if (!ok(hipGetLastError(), "transform_x")) return false;
    }
    transform_merge<<<p.groups, 256, 0, stream>>>(d_part, p.nparts, d_part + 3 * size_t(p.nparts));
    if (!ok(hipGetLastError(), "transform_merge")) return false;
    return true;
}

template bool transform_field<float>(const TransformPlan &, const Geometry &, const double *, void *, double, float *,
                                     double *, hipStream_t, hipEvent_t, std::string &);
template bool transform_field<double>(const TransformPlan &, const Geometry &, const double *, void *, double,
                                      double *, double *, hipStream_t, hipEvent_t, std::string &);

}  // namespace scarf
