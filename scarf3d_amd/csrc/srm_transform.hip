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
// of the Kaiser-Bessel kernel: kernel errors of 2e-8 and 1e-15 of the field.
// In FP64 the roundings count: the divisions by phi^ make those of a plane's
// corner 60 times as large, so positions and phases keep two doubles where one
// would round (turns()), and phi and phi^ are exact to a few ulps. Errors in the
// 2-norm, against the direct FP64 sum's: 20 x 33 x 27, 250 harmonics 1.4e-15
// (1.6e-15), 20000 1.9e-15 (5.2e-15); 128 x 100 x 60, 4000 harmonics 2.8e-15
// (3.8e-15); 2D 400 x 300, 500 harmonics 3.3e-15 (1.1e-14). With single doubles
// 4.4e-15, 4.5e-15, 6.7e-15 and 1.5e-14, in the same time.
#include "srm_transform.hpp"

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <type_traits>

#include "kaiser_bessel.hpp"
#include "srm_stats.hpp"

namespace scarf {
namespace {

using fft::Cplx;

constexpr double kInvTwoPi = 0.15915494309189533577;
constexpr double kPiD = 3.14159265358979323846;
constexpr int kThreads = 512;
constexpr size_t kLineBytes = 64 << 10;  // lines of a block (unpadded): two blocks per CU
constexpr size_t kMaxLds = 160 << 10;    // of a block alone
constexpr double kMinOversampling = 1.9;

typedef double f64x4 __attribute__((ext_vector_type(4)));

// Everything the kernels need besides the record and the output.
template <class Real>
struct Args {
    int w, nx, ny, nz, m, l, columns, np_;
    int ox, oy, oz;
    double ds, beta_x, beta_y, scaling;
    fft::Passes px, py;
    int zb, yb, nzb, slab, z0, zn;  // zn: planes of this round
    unsigned *key;           // class of the first ky << 14 | first column; ~0: amplitude 0
    int *order, *start;
    int *last;               // last column that a harmonic touches
    // in sorted order: [16][np], column c at c mod 16; [np][2 class widths] from the class' first ky on
    double *tapx, *tapy;
    Cplx<Real> *twy, *twx, *twr;
    unsigned short *revy, *revx;
    double *decx, *decy;
    bool pairs;              // the field takes aligned pairs
    Cplx<Real> *wave, *t;    // wave: [slab / zb][np][zb]
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
    double gx, gy, lx, ly;  // lx, ly: what gx, gy leave out (FP64 fields)
    int kx, ky;
    bool flip;
};
template <class Real>
__device__ inline Placed place(const Args<Real> &a, const double *__restrict__ harm, int n)
{
#pragma clang fp contract(off)
    const Turns tx = turns(harm[n], a.ds), ty = turns(harm[a.np_ + n], a.ds);
    Placed p;
    p.flip = tx.hi < 0.0;
    const double nx = p.flip ? -2.0 * a.m : 2.0 * a.m, ny = p.flip ? -a.l : a.l;
    p.gx = tx.hi * nx;
    p.gy = ty.hi * ny;
    p.lx = sizeof(Real) == 8 ? fma(tx.hi, nx, -p.gx) + tx.lo * nx : 0.0;
    p.ly = sizeof(Real) == 8 ? fma(ty.hi, ny, -p.gy) + ty.lo * ny : 0.0;
    p.kx = int(ceil(p.gx - 0.5 * a.w));
    p.ky = int(ceil(p.gy - 0.5 * a.w));
    return p;
}

template <class Real>
__global__ __launch_bounds__(256) void transform_keys(Args<Real> a, const double *__restrict__ harm)
{
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n == 0) *a.last = 0;
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
    int top = 0;
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
            if (tot > 0) top = bin + a.w - 1;
        }
    }
    if (top > 0) atomicMax(a.last, top);
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

// c_n(z) of the planes of a round, harmonics in sorted order: item e is plane
// e % zb of group e / (zb present). Phases in FP64, about the centre of the
// block along x and y.
template <class Real>
__device__ inline void wave_item(const Args<Real> &a, const double *__restrict__ harm, long e, int present)
{
    const long pairs = e / a.zb;
    const int group = int(pairs / present), p = int(pairs - long(group) * present), zz = int(e - pairs * a.zb);
    const int z = group * a.zb + zz, n = a.order[p];
    const double wx = harm[n], wy = harm[a.np_ + n], wz = harm[2 * long(a.np_) + n];
    const double xc = double(a.ox + a.nx / 2) * a.ds, yc = double(a.oy + a.ny / 2) * a.ds;
    const double zc = double(a.z0 + z + a.oz) * a.ds, phase = harm[3 * long(a.np_) + n];
    double t;
    if constexpr (sizeof(Real) == 8) {
        const Turns tx = turns(wx, xc), ty = turns(wy, yc), tz = turns(wz, zc), tp = turns(phase, 1.0);
        t = ((tx.hi + ty.hi) + (tz.hi + tp.hi)) + ((tx.lo + ty.lo) + (tz.lo + tp.lo));
    } else {
        t = (wz * zc) * kInvTwoPi + (wx * xc + wy * yc + phase) * kInvTwoPi;
    }
    t -= rint(t);
    double s, c;
    sincospi(turns(wx, a.ds).hi < 0.0 ? -2.0 * t : 2.0 * t, &s, &c);
    const double amp = harm[4 * long(a.np_) + n];
    a.wave[(long(group) * a.np_ + p) * a.zb + zz] = Cplx<Real>{static_cast<Real>(amp * c), static_cast<Real>(amp * s)};
}

template <class Real>
__global__ __launch_bounds__(256) void transform_waves(Args<Real> a, const double *__restrict__ harm)
{
    const long present = a.start[long(a.l / kClass<Real> - 1) * (a.m + 2) + a.m + 1];
    const long total = present * a.slab;
    for (long e = blockIdx.x * long(blockDim.x) + threadIdx.x; e < total; e += long(gridDim.x) * blockDim.x)
        wave_item(a, harm, e, int(present));
}

// Tables of one realization in sorted order, and the waves of the first
// round. Work items: waves; taps along y and x, one each, the zeros around them
// included; twiddles, digit-reversed positions and deconvolution factors.
template <class Real>
__global__ __launch_bounds__(256) void transform_tables(Args<Real> a, const double *__restrict__ harm)
{
    constexpr int W = sizeof(Real) == 4 ? 9 : 16, K = sizeof(Real) == 4 ? 45 : 66, R = 2 * kClass<Real>;
    constexpr bool F64 = sizeof(Real) == 8;
    const long present = a.start[long(a.l / kClass<Real> - 1) * (a.m + 2) + a.m + 1];
    const long i0 = present * a.slab, i1 = i0 + present * R, i2 = i1 + present * 16;
    const long total = i2 + a.l + 2 * long(a.m) + a.ny + a.nx;
    for (long e = blockIdx.x * long(blockDim.x) + threadIdx.x; e < total; e += long(gridDim.x) * blockDim.x) {
        if (e < i0) {
            wave_item(a, harm, e, int(present));
            continue;
        }
        if (e < i2) {
            const bool along_y = e < i1;
            const int p = int(along_y ? (e - i0) / R : (e - i1) % present);
            const Placed h = place(a, harm, a.order[p]);
            if (along_y) {
                const int ky = h.ky < 0 ? h.ky + a.l : h.ky;
                const int d = int((e - i0) % R) - ky % kClass<Real>;  // tap at the class' row
                a.tapy[e - i0] = d >= 0 && d < W ? kaiser_bessel<K, F64>(h.ky + d - h.gy - h.ly, W, a.beta_y, exp(-a.beta_y)) : 0.0;
            } else {
                const int slot = int((e - i1) / present), d = (slot - h.kx - a.w / 2) & 15;  // columns are kx + w/2
                a.tapx[long(slot) * a.np_ + p] = d < W ? kaiser_bessel<K, F64>(h.kx + d - h.gx - h.lx, W, a.beta_x, exp(-a.beta_x)) : 0.0;
            }
            continue;
        }
        int r = int(e - i2);
        double s, c;
        if (r < a.l) {
            sincospi(2.0 * fft::turns(r, a.py), &s, &c);
            a.twy[r] = Cplx<Real>{Real(c), Real(s)};
            a.revy[r] = static_cast<unsigned short>(fft::pad(fft::digit_reverse(r, a.py)));
            continue;
        }
        r -= a.l;
        if (r < a.m) {
            sincospi(2.0 * fft::turns(r, a.px), &s, &c);
            a.twx[r] = Cplx<Real>{Real(c), Real(s)};
            a.revx[r] = static_cast<unsigned short>(fft::pad(fft::digit_reverse(r, a.px)));
            continue;
        }
        r -= a.m;
        if (r < a.m) {
            sincospi(double(r) / a.m, &s, &c);
            a.twr[r] = Cplx<Real>{Real(c), Real(s)};
            continue;
        }
        r -= a.m;
        if (r < a.ny) a.decy[r] = deconvolution(r - a.ny / 2, a.l, W, a.beta_y);
        else if (r < a.ny + a.nx) a.decx[r - a.ny] = a.scaling * deconvolution(r - a.ny - a.nx / 2, 2 * a.m, W, a.beta_x);
    }
}

// LDS of the y pass behind the lines: partial sums of four waves, the
// classes' ranges for the block's column and the digit-reversed positions.
template <class Real>
size_t lds_y_bytes(int zb, int l)
{
    const size_t classes = size_t(l) / kClass<Real>;
    return size_t(zb) * fft::pitch(l) * sizeof(Cplx<Real>) + 16 + size_t(4) * 256 * sizeof(double) +
           classes * sizeof(int2) + size_t(l) * sizeof(unsigned short) + 16;
}

// inclusive sum over the lanes up to each one
__device__ inline int wave_scan(int v)
{
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr 1, 2, 4, 8
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // lane 15 of a row to the next one
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // lane 31 to the upper half
    return v;
}

// Spread and y pass: one block per (kx column, zb planes). The spread is a
// product on the FP64 matrix cores: a class' 16-row tiles of ky, by (plane,
// re/im), summed over the class' harmonics that touch the column, four per
// instruction,
//   A[ky][p] = phi_y, B[p][z] = phi_x c_p(z),
// so the sums are FP64 in a fixed order for either field type. A class reaches
// the rows of the next one too, and those are the upper half of its tiles:
// after a class' last step the lower half is stored and the upper one becomes
// the lower half of the next class' sums, with no exchange between lanes. A
// wave takes a run of classes with its share of the column's steps, kAhead of
// them in flight: most classes hold a few harmonics, and one class after the
// other is a chain of waits (512^3 float x 20k, 64 planes: 203 us; classes in
// flight but added to LDS by atomics, 298 us; so, 187 us, and 138 us with
// 32-bit offsets, a scan without LDS and the deconvolution left to the x
// pass). All waves together take a class of kShared steps and a sixteenth of
// the column's or more (at a small correlation length per box nearly all
// harmonics are in a few columns and classes); these columns are bound by the
// matrix cores. Then the lines are transformed in LDS. Blocks of
// one z group follow each other nzb apart: with nzb = 8 each XCD's L2 holds
// one group's waves.
constexpr int kShared = 32;
constexpr int kAhead = 4;
template <class Real, int Threads>
__global__ __launch_bounds__(Threads, 4) void transform_y(Args<Real> a)
{
    constexpr int G = kTiles<Real>, CW = kClass<Real>, W = sizeof(Real) == 4 ? 9 : 16, D = kAhead, kYWaves = Threads / 64;
    extern __shared__ __align__(16) unsigned char smem[];
    const int zblk = blockIdx.x % a.nzb, col = blockIdx.x / a.nzb;
    const int zoff = zblk * a.zb, planes = min(a.zb, a.zn - zoff);
    Cplx<Real> *out = a.t + (size_t(zoff) * a.columns + col) * a.ny;
    const unsigned plane = unsigned(a.columns) * a.ny;
    const Cplx<Real> zero{Real(0), Real(0)};
    const int line = fft::pitch(a.l), classes = a.l / CW;
    Cplx<Real> *lds = reinterpret_cast<Cplx<Real> *>(smem);
    Real *flat = reinterpret_cast<Real *>(smem);
    double *slots = reinterpret_cast<double *>(smem + (size_t(a.zb) * line * sizeof(Cplx<Real>) + 15) / 16 * 16);
    int2 *range = reinterpret_cast<int2 *>(slots + 4 * 256);
    unsigned short *rev = reinterpret_cast<unsigned short *>(range + classes);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int jj = lane & 15, slot = lane >> 4;
    const int lo = max(0, col - W + 1), hi = min(col, a.m);
    const bool mine = jj < 2 * a.zb;
    for (int q = tid; q < classes; q += Threads) {
        const int *st = a.start + long(q) * (a.m + 2);
        const int s0 = st[lo];
        range[q] = make_int2(s0, st[hi + 1] - s0);
    }
    for (int q = tid; q < a.l; q += Threads) rev[q] = a.revy[q];
    for (int q = tid; q < a.zb * line; q += Threads) lds[q] = zero;
    __syncthreads();
    // A and B of this lane's harmonic of step i of a range, or of its last one:
    // uniform bases and 32-bit offsets, which the loads take as they are
    const double *tapx = a.tapx + long(col & 15) * a.np_;
    const Cplx<Real> *waves = a.wave + long(zblk) * a.np_ * a.zb;
    const unsigned wave_step = unsigned(a.zb * sizeof(Cplx<Real>));
    const unsigned ylane = jj * sizeof(double), wlane = (mine ? jj : 0) * sizeof(Real);
    auto load = [&](int s0, int n, int i, double &x, Real &w, double (&y)[G]) __attribute__((always_inline)) {
        const unsigned k = static_cast<unsigned>(min(i + slot, n - 1));
        const char *yv = reinterpret_cast<const char *>(a.tapy + long(s0) * (16 * G));
        const char *wv = reinterpret_cast<const char *>(waves + long(s0) * a.zb);
        x = fft::element(tapx + s0, k);
        w = *reinterpret_cast<const Real *>(wv + (k * wave_step + wlane));
#pragma unroll
        for (int g = 0; g < G; ++g) y[g] = *reinterpret_cast<const double *>(yv + (k * (128u * G) + ylane) + 128 * g);
    };
    // rem: harmonics from the step on; those beyond count as zeros
    auto product = [&](int rem, double x, Real w, const double (&y)[G], f64x4 (&acc)[G]) __attribute__((always_inline)) {
        const double b = slot < rem ? static_cast<double>(w) * x : 0.0;
#pragma unroll
        for (int g = 0; g < G; ++g) acc[g] = __builtin_amdgcn_mfma_f64_16x16x4f64(y[g], b, acc[g], 0, 0, 0);
    };
    auto clear = [](f64x4 (&acc)[G]) __attribute__((always_inline)) {
#pragma unroll
        for (int g = 0; g < G; ++g) acc[g] = f64x4{0.0, 0.0, 0.0, 0.0};
    };
    // rows 4 r + slot of class q, from the lane's sums v[r], stored or added
    auto put = [&](int q, bool add, const double (&v)[CW / 4]) __attribute__((always_inline)) {
        int at[CW / 4];
#pragma unroll
        for (int r = 0; r < CW / 4; ++r) {
            const int ky = q * CW + 4 * r + slot;
            at[r] = 2 * ((jj >> 1) * line + rev[ky >= a.l ? ky - a.l : ky]) + (jj & 1);
        }
        if (!mine) return;
#pragma unroll
        for (int r = 0; r < CW / 4; ++r)
            flat[at[r]] = static_cast<Real>(add ? static_cast<double>(flat[at[r]]) + v[r] : v[r]);
    };
    // the halves of a class' tiles
    auto put_lower = [&](int q, bool add, const f64x4 (&acc)[G]) __attribute__((always_inline)) {
        if constexpr (G == 1) put(q, add, {acc[0][0], acc[0][1]});
        else put(q, add, {acc[0][0], acc[0][1], acc[0][2], acc[0][3]});
    };
    auto move_down = [&](f64x4 (&acc)[G]) __attribute__((always_inline)) {
        if constexpr (G == 1) acc[0] = f64x4{acc[0][2], acc[0][3], 0.0, 0.0};
        else {
            acc[0] = acc[G - 1];
            acc[G - 1] = f64x4{0.0, 0.0, 0.0, 0.0};
        }
    };
    // steps of classes base .. base + 63, one per lane
    auto steps = [&](int base, int2 &r) __attribute__((always_inline)) {
        r = base + lane < classes ? range[base + lane] : make_int2(0, 0);
        return (r.y + 3) >> 2;
    };
    int total = 0, light = 0, before = 0;
    for (int base = 0; base < classes; base += 64) {
        int2 r;
        total += __builtin_amdgcn_readlane(wave_scan(steps(base, r)), 63);
    }
    if (total == 0) {  // no harmonic touches the column: zeros, of which the x pass reads those of the next one too
        if (col <= *a.last + 1)
            for (int z = 0; z < planes; ++z)
                for (int y = tid; y < a.ny; y += Threads) fft::element(out, unsigned(z) * plane + y) = zero;
        return;
    }
    const int limit = max(kShared, total / 16);
    for (int base = 0; base < classes; base += 64) {
        int2 r;
        const int own = steps(base, r);
        light += __builtin_amdgcn_readlane(wave_scan(own <= limit ? own : 0), 63);
    }
    const int first = light * wave / kYWaves, last = light * (wave + 1) / kYWaves;
    f64x4 acc[G];
    clear(acc);
    int cur = -1;  // the class whose rows the lower half of acc belongs to
    for (int base = 0; base < classes; base += 64) {
        int2 r;
        int own = steps(base, r);
        own = own <= limit ? own : 0;
        const int upto = wave_scan(own), at = before + upto - own;
        uint64_t left = __ballot(own > 0 && at >= first && at < last);
        before += __builtin_amdgcn_readlane(upto, 63);
        if (left == 0) continue;
        int s0 = 0, n = 0, i = 0, q = 0;  // the next step: harmonics i .. i + 3 of class q
        double x[D], y[D][G];
        Real w[D];
        int rem[D], cls[D];
        auto issue = [&](int u) __attribute__((always_inline)) {
            if (i >= n && left) {
                const int k = __ffsll(static_cast<unsigned long long>(left)) - 1;
                left &= left - 1;
                s0 = __builtin_amdgcn_readlane(r.x, k);
                n = __builtin_amdgcn_readlane(r.y, k);
                q = base + k;
                i = 0;
            }
            rem[u] = n - i;  // none left: 0 or less
            cls[u] = q;
            load(s0, n, i, x[u], w[u], y[u]);
            i += 4;
        };
#pragma unroll
        for (int u = 0; u < D; ++u) issue(u);
        while (rem[0] > 0) {
#pragma unroll
            for (int u = 0; u < D; ++u) {
                const int rest = rem[u], c = cls[u];
                if (rest <= 0) break;
                if (c != cur) {  // not the class after the last one
                    if (cur >= 0) put_lower(cur, false, acc);
                    clear(acc);
                    cur = c;
                }
                product(rest, x[u], w[u], y[u], acc);
                issue(u);
                if (rest <= 4) {
                    put_lower(c, false, acc);
                    move_down(acc);
                    cur = c + 1;
                }
            }
        }
    }
    __syncthreads();
    if (cur >= 0) put_lower(cur, true, acc);  // another wave's class, or an empty one
    if (light < total) {
        int base = -64, s0 = 0, n = 0, q = 0;
        uint64_t left = 0;
        auto next = [&]() __attribute__((always_inline)) {
            while (left == 0) {
                base += 64;
                if (base >= classes) return false;
                int2 r;
                left = __ballot(steps(base, r) > limit);
            }
            q = base + __ffsll(static_cast<unsigned long long>(left)) - 1;
            left &= left - 1;
            s0 = __builtin_amdgcn_readfirstlane(range[q].x);
            n = __builtin_amdgcn_readfirstlane(range[q].y);
            return true;
        };
        constexpr int U = kAhead;
        double x[U], y[U][G];
        Real w[U];
        auto issue = [&](int i0) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < U; ++u) load(s0, n, i0 + 4 * u * kYWaves, x[u], w[u], y[u]);
        };
        bool more = next();
        issue(4 * wave);
        while (more) {
            clear(acc);
            for (int i0 = 4 * wave; i0 < n;) {
#pragma unroll
                for (int u = 0; u < U; ++u) product(n - i0 - 4 * u * kYWaves, x[u], w[u], y[u], acc);
                i0 += 4 * U * kYWaves;
                if (i0 < n) issue(i0);
            }
            const int c = q;
            more = next();
            if (more) issue(4 * wave);  // in flight over the reduction
#pragma unroll
            for (int g = 0; g < G; ++g) {
                double *mine_of = slots + (wave & 3) * 256 + lane;
                for (int four = 4; four < kYWaves; four += 4) {
                    fft::lds_barrier();
                    if (wave >= four && wave < four + 4)
#pragma unroll
                        for (int r = 0; r < 4; ++r) mine_of[64 * r] = acc[g][r];
                    fft::lds_barrier();
                    if (wave < 4)
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[g][r] += mine_of[64 * r];
                }
                fft::lds_barrier();
                if (wave >= 1 && wave < 4)
#pragma unroll
                    for (int r = 0; r < 4; ++r) mine_of[64 * r] = acc[g][r];
                fft::lds_barrier();
                if (wave == 0)
#pragma unroll
                    for (int v = 1; v < 4; ++v)
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[g][r] += slots[256 * v + 64 * r + lane];
            }
            if (wave == 0) {
                put_lower(c, true, acc);
                move_down(acc);
                put_lower(c + 1, true, acc);
            }
        }
    }
    // the ny kept outputs of the last pass leave the block
    fft::transform(lds, a.twy, 0, a.py, line, a.zb, tid, Threads,
                   [&](int z, int q, Cplx<Real> v) __attribute__((always_inline)) {
                       const unsigned y = (2 * q < a.l ? q : q - a.l) + a.ny / 2;
                       if (z < planes && y < unsigned(a.ny)) fft::element(out, unsigned(z) * plane + y) = v;
                   });
}

// x pass: one block per (plane, yb lines). The real transform of 2m values is
// a complex one of m: Z_k = A + i e^(i pi k / m) D, Z_(m-k) = conj(A) + i
// conj(e^(i pi k / m) D) with A, D = H_k +- conj(H_(m-k)) and H the half
// spectrum (interior values halved: only the real part of the sum is kept).
// An item is the first butterflies, of radix R = kFirstX, of inputs b + r m/R
// and m/R - b + r m/R, which hold each other's partners (butterflies 0 and
// m/2R hold their own): T comes straight into registers, and the last pass
// stores the field from registers, divided by phi^ of both axes, scaled and
// rounded, with the statistics partials. 512^3 float, 64 planes: 90 us (147
// with T through LDS; 110 with a check of every column, single stores and
// twiddles out of the lanes' order), of which the 200 MB moved take 43.
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
    const int zeros = *a.last + 1;  // the first column of zeros only
    constexpr int R = kFirstX<Real>;
    const int step = a.m / R;
    for (int e = tid; e < (step / 2) * a.yb; e += kThreads) {
        const int yy = e & (a.yb - 1), b = e / a.yb;
        if (yy >= lines) continue;
        auto at = [&](int kx) __attribute__((always_inline)) {
            return fft::element(t, unsigned(min(kx + off, zeros)) * unsigned(a.ny) + yy);
        };
        C p[R], q[R], pm{};
        const int bp = b, bq = b == 0 ? step / 2 : step - b;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            p[r] = at(bp + r * step);
            q[r] = at(bq + r * step);
        }
        if (b == 0) pm = at(a.m);
        // columns outside 0 .. m fold onto their conjugates: first and last few
        if (b <= a.w || step <= 2 * a.w) {
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
    const double *decy = a.decy + y0;
    auto add = [&](double o) __attribute__((always_inline)) {
        const double d = o - pivot;
        s1 += d;
        s2 = fma(d, d, s2);
    };
    fft::transform(lds, a.twx, 1, a.px, line, lines, tid, kThreads,
                   [&](int yy, int q, C v) __attribute__((always_inline)) {
                       const int i = 2 * (2 * q < a.m ? q : q - a.m) + a.nx / 2;
                       if (i < -1 || i >= a.nx) return;
                       const double dy = decy[yy];
                       Real *o = &fft::element(rows, unsigned(yy * a.nx + max(i, 0)));
                       const bool first = i >= 0, second = i + 1 < a.nx;
                       const C c{static_cast<Real>(static_cast<double>(v.x) * (dy * a.decx[max(i, 0)])),
                                 static_cast<Real>(static_cast<double>(v.y) * (dy * a.decx[min(i + 1, a.nx - 1)]))};
                       if (cnt == 0) pivot = static_cast<double>(first ? c.x : c.y);
                       if (a.pairs) {
                           *reinterpret_cast<C *>(o) = c;
                           add(c.x);
                           add(c.y);
                           cnt += 2;
                           return;
                       }
                       if (first) {
                           o[0] = c.x;
                           add(c.x);
                       }
                       if (second) {
                           o[int(first)] = c.y;
                           add(c.y);
                       }
                       cnt += int(first) + int(second);
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
    p.fx = fft::plan(p.m, f64 ? kFirstX<double> : kFirstX<float>, f64);
    p.fy = fft::plan(p.l, 8, f64);
    // Kaiser-Bessel shape for the axis' oversampling s (pi w (1 - 1/(2 s)), just inside)
    p.beta_x = 0.995 * kPiD * p.w * (1.0 - 0.5 * g.nx / fx);
    p.beta_y = 0.995 * kPiD * p.w * (1.0 - 0.5 * g.ny / p.l);
    p.zb = 8;
    while (p.zb > 1 && size_t(p.zb) * p.l * csize > kLineBytes) p.zb /= 2;
    // lines of which half a CU's LDS takes fewer planes than a matrix tile has:
    // a block of twice the threads with the CU to itself (1024^2 x 512 x 50k,
    // field: 12.1 -> 8.5 ms, and 6.6 -> 5.1 at longer correlation lengths)
    if (p.zb < 8 && g.nz > p.zb && (f64 ? lds_y_bytes<double>(2 * p.zb, p.l) : lds_y_bytes<float>(2 * p.zb, p.l)) <= kMaxLds) {
        p.zb *= 2;
        p.wide = true;
    }
    while (p.zb > 1 && p.zb / 2 >= g.nz) p.zb /= 2;
    p.yb = 16;
    while (p.yb > 1 && size_t(p.yb) * p.m * csize > kLineBytes) p.yb /= 2;
    while (p.yb > 1 && p.yb / 2 >= g.ny) p.yb /= 2;
    // planes per round: eight blocks' worth, more while the intermediate and
    // the harmonics' values (which outgrow it on thin blocks) stay small
    const size_t plane = size_t(p.columns) * p.ny * csize, values = size_t(np_) * csize;
    const int zmax = (g.nz + p.zb - 1) / p.zb * p.zb;
    p.slab = 8 * p.zb;
    while (p.slab < zmax && plane * p.slab * 2 <= (size_t(192) << 20) && values * p.slab * 2 <= (size_t(256) << 20))
        p.slab *= 2;
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
    p.o_order = take(np * sizeof(int));
    p.o_start = take(size_t(p.l / cls) * (p.m + 2) * sizeof(int));
    p.o_last = take(sizeof(int));
    p.o_taps = take(np * (2 * cls + 16) * sizeof(double));
    p.o_tw = take((size_t(p.l) + 2 * size_t(p.m)) * csize);
    p.o_rev = take((size_t(p.l) + p.m) * sizeof(unsigned short));
    p.o_dec = take((size_t(p.ny) + p.nx) * sizeof(double));
    p.o_wave = take(np * p.slab * csize);
    p.o_t = take(plane * p.slab);
    p.bytes = at;
    // the y pass counts bytes from a class' first harmonic on in 32 bits
    return np * size_t(2 * cls) * sizeof(double) < (size_t(1) << 32);
}

// Linear fits to measured times, from above. Transform: the chain of small
// launches, the harmonics' tables and ordering, the cells of both passes, their
// blocks, and the spread. The line between the two lies at a few hundred
// harmonics for FP32 grids (float, direct_f32: 64^3 x 256 0.060 against 0.103
// ms, x 64 0.058 against 0.045; bf16x3: 128^3 x 1024 0.10 against 0.12, 256^3 x
// 4096 0.33 against 1.27) and below 64 for FP64 ones (64^3 x 64 0.062 against
// 0.131 ms).
double transform_ms(const TransformPlan &p, bool f64)
{
    const double cells = double(p.columns) * p.l * p.nz;
    const double blocks = double(p.columns) * ((p.nz + p.zb - 1) / p.zb) + p.nparts;
    const double waves = double(p.np_) * p.nz;
    return f64 ? 0.055 + 1.05e-5 * p.np_ + 8e-9 * cells + 1e-5 * blocks + 4e-8 * waves
               : 0.053 + 7e-6 * p.np_ + 5e-9 * cells + 1.1e-5 * blocks + 2e-8 * waves;
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
    a.px = p.fx;
    a.py = p.fy;
    a.zb = p.zb;
    a.yb = p.yb;
    a.slab = p.slab;
    a.key = reinterpret_cast<unsigned *>(base + p.o_key);
    a.order = reinterpret_cast<int *>(base + p.o_order);
    a.start = reinterpret_cast<int *>(base + p.o_start);
    a.last = reinterpret_cast<int *>(base + p.o_last);
    a.tapy = reinterpret_cast<double *>(base + p.o_taps);
    a.tapx = a.tapy + size_t(p.np_) * 2 * kClass<Real>;
    a.twy = reinterpret_cast<Cplx<Real> *>(base + p.o_tw);
    a.twx = a.twy + p.l;
    a.twr = a.twx + p.m;
    a.revy = reinterpret_cast<unsigned short *>(base + p.o_rev);
    a.revx = a.revy + p.l;
    a.decx = reinterpret_cast<double *>(base + p.o_dec);
    a.decy = a.decx + p.nx;
    // a row's outputs 2 q + nx / 2 and the next one are then an aligned pair
    a.pairs = p.nx % 4 == 0 && reinterpret_cast<uintptr_t>(d_field) % (2 * sizeof(Real)) == 0;
    a.wave = reinterpret_cast<Cplx<Real> *>(base + p.o_wave);
    a.t = reinterpret_cast<Cplx<Real> *>(base + p.o_t);

    transform_keys<Real><<<(p.np_ + 255) / 256, 256, 0, stream>>>(a, d_harm);
    if (!ok(hipGetLastError(), "transform_keys")) return false;
    int sort_waves = 16;  // as many as their histograms fit in LDS
    while (size_t(sort_waves) * (p.m + 1) * sizeof(int) > (size_t(80) << 10)) sort_waves /= 2;
    transform_order<Real><<<p.l / kClass<Real>, 64 * sort_waves, size_t(sort_waves) * (p.m + 1) * sizeof(int), stream>>>(a);
    if (!ok(hipGetLastError(), "transform_order")) return false;
    a.zn = std::min(p.slab, p.nz);
    const long items = long(p.np_) * (p.slab + 2 * kClass<Real> + 16) + p.l + 2 * long(p.m) + p.ny + p.nx;
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
        if (p.wide) transform_y<Real, 1024><<<a.nzb * p.columns, 1024, lds_y, stream>>>(a);
        else transform_y<Real, 512><<<a.nzb * p.columns, 512, lds_y, stream>>>(a);
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
