// Dense transforms of the FIM grid (see fim_dft.hpp).
//
// Every axis has an even length N = 2 M. Along y and z the even and the odd
// inputs of a line have transforms Y0, Y1 of length M, and
//   out[k] = Y0[k] + w^k Y1[k], out[k + M] = Y0[k] - w^k Y1[k], w = e^{2 pi i / N}.
// With a[n] = x[n] + x[M - n] and d[n] = x[n] - x[M - n], n = 0 .. M/2,
//   Y[k], Y[M - k] = sum_n cos(2 pi k n / M) a[n] +- i sum_n sin(2 pi k n / M) d[n],
// so a line takes products with two real (M/2 + 1)-square matrices, an eighth
// of the full complex product. Along x the even and odd harmonics' cosine and
// sine sums over the real field's half spectrum give the outputs i, M - i,
// M + i and N - i by their signs.
//
// A block holds whole lines in LDS, in the order of the matrix operands (a
// wave reads 64 consecutive vectors), and each wave takes 16 rows of the
// matrices, whose elements it reads from L2 in lane order, once per block.
// At 502^3 in float a pass along y or z does 33 GFLOP on the FP32 matrix cores
// (0.21 ms at their peak) over 1 GB (0.2 ms), and takes 0.44 ms: two blocks
// share a CU, and the one's loads and stores cover only part of the other's
// products. With loads left in conditions it took 0.50 ms.
// The whole transform: 1.35 ms with its statistics (1.43 with the caller's
// block too), the FFT library's 2.77 ms and 0.13 ms for them.
#include "fim_dft.hpp"

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "srm_stats.hpp"

namespace scarf {
namespace fim_dft {
namespace {

template <class Real, int N>
using Vec = Real __attribute__((ext_vector_type(N)));

constexpr size_t kLds = 160 << 10;
constexpr int kXcds = 8;
template <class Real>
constexpr int kColumnWaves = sizeof(Real) == 4 ? 16 : 8;  // of a block at most: FP64 sums alone fill 128 registers
constexpr int kAhead = 4;  // items of a thread whose loads are in flight together

// inputs of a line's products, padded to the four of a matrix instruction
__host__ __device__ constexpr int depth(int n) { return (n / 4 + 1 + 3) / 4 * 4; }
// 16-row tiles of the outputs
__host__ __device__ constexpr int tiles(int n) { return (n / 4 + 1 + 15) / 16; }

// lines of a block of the x pass
template <class Real>
constexpr int kRows = sizeof(Real) == 4 ? 32 : 16;

template <class Real>
size_t columns_lds(int n)
{
    return size_t(depth(n)) * 16 * 8 * sizeof(Real);
}
template <class Real>
size_t rows_lds(int n)
{
    return std::max(size_t(depth(n)) * (kRows<Real> + 1) * 4, size_t(kRows<Real>) * (n + 1)) * sizeof(Real);
}

__device__ inline Vec<float, 4> product(float a, float b, Vec<float, 4> c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ inline Vec<double, 4> product(double a, double b, Vec<double, 4> c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
// row of a product's element r
template <class Real>
__device__ inline int row_of(int lane, int r)
{
    return sizeof(Real) == 4 ? 4 * (lane >> 4) + r : 4 * r + (lane >> 4);
}

// Keeps loads whose use is conditional where they are: their values are
// needed here, and a load is not moved into the condition.
template <class... T>
__device__ __forceinline__ void together(T &...v)
{
    auto need = [](auto &x) __attribute__((always_inline)) { asm volatile("" : "+v"(x)); };
    (need(v), ...);
}

// step(s, table value) for s = 0 .. steps - 1, with the table values of the
// next group of steps in flight from L2 while one is multiplied. The sums of F
// steps, of a group at most, start from zero and are added to the totals by
// flush(): a chain of 16 terms and one of steps / 4 sums round less than one
// over all terms (502^3 in float 3.0e-7 off FP64, with one chain 5.3e-7, the FFT
// library 4.1e-7; 214 x 186 x 138 in double 4.7e-16 off extended precision, the
// library 9.9e-16).
//
// The library's FP32 transform rounds less where its lengths are short (of a
// field's 3.1e-7 some 2.9e-7 are the spectrum's) or few have a large prime factor.
// So float lines up to 64 take chains of 4 terms, and lines up to 128, or 288
// where at most one axis has a large prime factor, of 8 terms, with totals and
// last combinations in FP64. Float fields against extended precision, so / with
// chains of 16 / the library, and their calls: 62 x 58 x 46 3.11e-7 / 3.45e-7 /
// 3.23e-7; 96 x 120 x 64 2.73e-7 / 3.07e-7 / 2.87e-7, 89 / 87 / 106 us; 128^3
// 3.10e-7 / 3.39e-7 / 3.06e-7, 115 / 111 / 112 us; 256 x 252 x 62 3.31e-7 / 3.64e-7
// / 3.29e-7, 150 / 135 / 172 us; 256 x 256 x 102 3.17e-7 / 3.50e-7 / 3.13e-7, 214 /
// 183 / 187 us. Other lines stay as they are: with two large prime factors the
// library is further off (214 x 186 x 138 3.20e-7 / 3.38e-7), and 258^3 would pay
// 338 -> 438 us.
template <int F, class V, class Step, class Flush>
__device__ __forceinline__ void for_steps(const V *__restrict__ t, int steps, const Step &step, const Flush &flush)
{
    constexpr int U = sizeof(V) > 16 ? 2 : 4;
    V w[U];
#pragma unroll
    for (int u = 0; u < U; ++u) w[u] = t[min(u, steps - 1) * 64];
    int s = 0;
    for (; s + U <= steps; s += U) {
        V next[U];
#pragma unroll
        for (int u = 0; u < U; ++u) next[u] = t[min(s + U + u, steps - 1) * 64];
        __builtin_amdgcn_sched_barrier(0);  // not moved down to their use
#pragma unroll
        for (int u = 0; u < U; ++u) {
            step(s + u, w[u], u % F == 0);
            if (u % F == F - 1 || u == U - 1) flush();
        }
#pragma unroll
        for (int u = 0; u < U; ++u) w[u] = next[u];
    }
    if (s == steps) return;
#pragma unroll
    for (int u = 0; u < U - 1; ++u)
        if (s + u < steps) {
            step(s + u, w[u], u % F == 0);
            if (u % F == F - 1 || s + u == steps - 1) flush();
        }
}


// sine and cosine of r/n turns, 0 <= r < n, from the distance to the nearest
// quarter: a quotient near 1 would lose up to 7e-16 to its own rounding
__device__ inline void sincos_turns(int64_t r, int n, double *s, double *c)
{
    const int quarter = int((8 * r + n) / (2 * n));  // 0 .. 4
    double x, y;
    sincospi(double(4 * r - int64_t(quarter) * n) / (2.0 * n), &y, &x);
    *c = quarter & 1 ? -y : x;
    *s = quarter & 1 ? x : y;
    if (quarter & 2) {
        *c = -*c;
        *s = -*s;
    }
}

// Tables of one axis of length n. Columns (y, z): [tile][step][lane] {cos,
// sin}(2 pi k q / M) of row k and input q, then w^k, k = 0 .. M/2. Rows (x):
// [tile][step][lane] {cos, sin} of harmonic 2q, then of 2q + 1, at output i,
// times 2 for a harmonic whose conjugate is not stored.
template <class Real>
__global__ __launch_bounds__(256) void dft_columns_table(Vec<Real, 2> *__restrict__ t, int n)
{
    const int m = n / 2, half = n / 4, steps = depth(n) / 4, total = tiles(n) * steps * 64;
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    double s = 0.0, c = 0.0;
    if (e < total) {
        const int lane = e & 63, k = e / 64 / steps * 16 + (lane & 15), q = e / 64 % steps * 4 + (lane >> 4);
        if (k <= half && q <= half) sincos_turns(k * q % m, m, &s, &c);
    } else if (e <= total + half) {
        sincos_turns(e - total, n, &s, &c);
    } else {
        return;
    }
    t[e] = Vec<Real, 2>{Real(c), Real(s)};
}
template <class Real>
__global__ __launch_bounds__(256) void dft_rows_table(Vec<Real, 4> *__restrict__ t, int n)
{
    const int m = n / 2, half = n / 4, steps = depth(n) / 4, total = tiles(n) * steps * 64;
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= total) return;
    const int lane = e & 63, i = e / 64 / steps * 16 + (lane & 15), q = e / 64 % steps * 4 + (lane >> 4);
    Vec<Real, 4> v{Real(0), Real(0), Real(0), Real(0)};
#pragma unroll
    for (int odd = 0; odd < 2; ++odd) {
        const int k = 2 * q + odd;
        if (i > half || k > m) continue;
        const bool alone = k == 0 || k == m;
        double s, c;
        sincos_turns(k * i % n, n, &s, &c);
        v[2 * odd] = Real(alone ? c : 2.0 * c);
        v[2 * odd + 1] = Real(alone ? 0.0 : 2.0 * s);
    }
    t[e] = v;
}

// Blocks are dealt to the XCDs in turn: the block's place in an order where
// each XCD has a contiguous range, so that neighbours, which share cache
// lines, meet in one L2.
__device__ inline long place_of(long block, long total)
{
    const long chunk = (total + kXcds - 1) / kXcds;
    return block % kXcds * chunk + block / kXcds;
}

// Lines of n elements `stride` apart, 16 neighbouring ones per block, in place:
// a block reads its lines before it writes any. Sum: the type of the totals; FP64
// ones of FP32 fields take more registers, and their blocks have 8 waves at most.
template <class Real, class Sum, int Chain>
__global__ __launch_bounds__(sizeof(Sum) > sizeof(Real) ? 512 : 64 * kColumnWaves<Real>) void dft_columns(Vec<Real, 2> *__restrict__ S, const Vec<Real, 2> *__restrict__ table,
                                                    int n, long stride, int columns, long plane, int per_plane,
                                                    long blocks)
{
    using V2 = Vec<Real, 2>;
    using V4 = Vec<Real, 4>;
    using S2 = Vec<Sum, 2>;
    using S4 = Vec<Sum, 4>;
    extern __shared__ __align__(16) char shared[];
    const long place = place_of(blockIdx.x, blocks);
    if (place >= blocks) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, waves = blockDim.x >> 6;
    const int m = n / 2, half = n / 4, deep = depth(n), steps = deep / 4;
    const int first = int(place % per_plane) * 16;
    V2 *base = S + place / per_plane * plane + first;
    V4 *sum = reinterpret_cast<V4 *>(shared), *diff = sum + deep * 16;
    // item: input q of column e & 15, the same for every item of a thread; all
    // loads of kAhead items before the first is used, at clamped places, since
    // a condition would wait for one load after the other
    const bool in = first + (tid & 15) < columns;
    const V2 *line = base + (in ? tid & 15 : 0);
    for (int e0 = tid; e0 < deep * 16; e0 += kAhead * int(blockDim.x)) {
        V2 x0[kAhead], x1[kAhead], y0[kAhead], y1[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int q = min((e0 + u * int(blockDim.x)) >> 4, half), mirror = q == 0 ? 0 : m - q;
            x0[u] = line[2 * q * stride];
            x1[u] = line[(2 * q + 1) * stride];
            y0[u] = line[2 * mirror * stride];
            y1[u] = line[(2 * mirror + 1) * stride];
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) together(x0[u], x1[u], y0[u], y1[u]);
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int e = e0 + u * int(blockDim.x), q = e >> 4;
            if (e >= deep * 16) break;
            V4 a = V4{x0[u].x, x0[u].y, x1[u].x, x1[u].y}, d = a;
            if (q > 0 && 2 * q < m) {
                const V4 y{y0[u].x, y0[u].y, y1[u].x, y1[u].y};
                a += y;
                d -= y;
            }
            if (q > half || !in) a = d = V4{Real(0), Real(0), Real(0), Real(0)};
            sum[e] = a;
            diff[e] = d;
        }
    }
    __syncthreads();
    const V2 *turn = table + tiles(n) * steps * 64;
    for (int tile = wave; tile < tiles(n); tile += waves) {
        V4 part[8];
        S4 ca[4], sd[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) ca[r] = sd[r] = S4{Sum(0), Sum(0), Sum(0), Sum(0)};
        V2 wk[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) wk[r] = turn[min(tile * 16 + row_of<Real>(lane, r), half)];
        for_steps<Chain>(table + tile * steps * 64 + lane, steps, [&](int s, V2 w, bool fresh) __attribute__((always_inline)) {
            const V4 a = sum[s * 64 + lane], d = diff[s * 64 + lane], zero{Real(0), Real(0), Real(0), Real(0)};
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                part[r] = product(w.x, a[r], fresh ? zero : part[r]);
                part[4 + r] = product(w.y, d[r], fresh ? zero : part[4 + r]);
            }
        }, [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                ca[r] += __builtin_convertvector(part[r], S4);
                sd[r] += __builtin_convertvector(part[4 + r], S4);
            }
        });
        if (first + (lane & 15) >= columns) continue;
        V2 *out = base + (lane & 15);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int k = tile * 16 + row_of<Real>(lane, r);
            if (k > half) continue;
            const S2 w = __builtin_convertvector(wk[r], S2);
            auto put = [&](int at, S2 v) __attribute__((always_inline)) { out[at * stride] = __builtin_convertvector(v, V2); };
            const S2 y0{ca[0][r] - sd[1][r], ca[1][r] + sd[0][r]}, y1{ca[2][r] - sd[3][r], ca[3][r] + sd[2][r]};
            const S2 wy{w.x * y1.x - w.y * y1.y, w.x * y1.y + w.y * y1.x};
            put(k, y0 + wy);
            put(k + m, y0 - wy);
            if (k == 0 || 2 * k == m) continue;
            // Y[M - k] and w^(M - k) = -conj(w^k)
            const S2 z0{ca[0][r] + sd[1][r], ca[1][r] - sd[0][r]}, z1{ca[2][r] + sd[3][r], ca[3][r] - sd[2][r]};
            const S2 wz{w.x * z1.x + w.y * z1.y, w.x * z1.y - w.y * z1.x};
            put(m - k, z0 - wz);
            put(n - k, z0 + wz);
        }
    }
}

// Real lines along x from their half spectra, kRows lines per block, and the
// block's moments of the outputs times scaling: each value is the `real`
// product the reference stores, summed in FP64 as a sum and a sum of squares
// per thread (the field's mean is zero up to rounding). The outputs go by way
// of LDS, since a wave's product holds 16 positions of 16 lines; from there
// they go to the caller's grid where nothing else follows (500^3: 1 GB and
// 0.27 ms less than by way of R and a pass that gathers).
template <class Real, class Sum, int Chain>
__global__ __launch_bounds__(sizeof(Sum) > sizeof(Real) ? 512 : 1024) void dft_rows(const Vec<Real, 2> *__restrict__ S, Real *__restrict__ R,
                                                 Nearest<Real> to, const Vec<Real, 4> *__restrict__ table, int n,
                                                 int n2, int lines, Real scaling, double *__restrict__ part)
{
    using V2 = Vec<Real, 2>;
    using V4 = Vec<Real, 4>;
    constexpr int L = kRows<Real>, T = L / 16;
    extern __shared__ __align__(16) char shared[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, waves = blockDim.x >> 6;
    const int m = n / 2, half = n / 4, deep = depth(n), steps = deep / 4;
    const int line0 = blockIdx.x * L, count = min(L, lines - line0);
    V4 *x = reinterpret_cast<V4 *>(shared);  // [deep][L + 1]
    int j0 = 0, j1 = 0, k0 = 0, k1 = 0;      // outputs of the line of this lane's number
    if (to.field && lane < count) {
        const int j = (line0 + lane) % n2, k = (line0 + lane) / n2;
        j0 = to.first_y[j + 1];
        j1 = to.first_y[j + 2];
        k0 = to.first_z[k + 1];
        k1 = to.first_z[k + 2];
    }
    // a wave takes lines wave, wave + waves, ..., kAhead of them in flight
    for (int q = lane; q < deep; q += 64) {
        const int even = min(2 * q, m), odd = min(2 * q + 1, m);
        for (int l0 = wave; l0 < L; l0 += kAhead * waves) {
            V2 e[kAhead], o[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const V2 *s = S + size_t(line0 + min(l0 + u * waves, count - 1)) * (m + 1);
                e[u] = s[even];
                o[u] = s[odd];
            }
#pragma unroll
            for (int u = 0; u < kAhead; ++u) together(e[u], o[u]);
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const int line = l0 + u * waves;
                if (line >= L) break;
                const bool has = line < count && 2 * q <= m, both = has && 2 * q < m;
                x[q * (L + 1) + line] = V4{has ? e[u].x : Real(0), has ? e[u].y : Real(0), both ? o[u].x : Real(0),
                                           both ? o[u].y : Real(0)};
            }
        }
    }
    __syncthreads();
    using S4 = Vec<Sum, 4>;
    V4 sums[T][4];
    S4 ce[T], se[T], co[T], so[T];
#pragma unroll
    for (int t = 0; t < T; ++t) ce[t] = se[t] = co[t] = so[t] = S4{Sum(0), Sum(0), Sum(0), Sum(0)};
    const bool busy = wave < tiles(n);
    if (busy) {
        const V4 *b = x + (lane >> 4) * (L + 1) + (lane & 15);
        for_steps<Chain>(table + wave * steps * 64 + lane, steps, [&](int s, V4 c, bool fresh) __attribute__((always_inline)) {
            const V4 zero{Real(0), Real(0), Real(0), Real(0)};
#pragma unroll
            for (int t = 0; t < T; ++t) {
                const V4 v = b[s * 4 * (L + 1) + 16 * t];
#pragma unroll
                for (int j = 0; j < 4; ++j) sums[t][j] = product(c[j], v[j], fresh ? zero : sums[t][j]);
            }
        }, [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int t = 0; t < T; ++t) {
                ce[t] += __builtin_convertvector(sums[t][0], S4);
                se[t] += __builtin_convertvector(sums[t][1], S4);
                co[t] += __builtin_convertvector(sums[t][2], S4);
                so[t] += __builtin_convertvector(sums[t][3], S4);
            }
        });
    }
    __syncthreads();
    Real *y = reinterpret_cast<Real *>(shared);  // [L][n + 1]
    if (busy) {
#pragma unroll
        for (int t = 0; t < T; ++t) {
            Real *line = y + (16 * t + (lane & 15)) * (n + 1);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = wave * 16 + row_of<Real>(lane, r);
                if (i > half) continue;
                const Sum c = ce[t][r] + co[t][r], d = ce[t][r] - co[t][r];
                const Sum s = se[t][r] + so[t][r], u = se[t][r] - so[t][r];
                line[i] = Real(c - s);
                line[m + i] = Real(d - u);
                if (i == 0) continue;
                line[n - i] = Real(c + s);
                if (2 * i < m) line[m - i] = Real(d + u);
            }
        }
    }
    __syncthreads();
    double s1 = 0.0, s2 = 0.0;
    int mine = 0;
    for (int line = wave; line < count; line += waves) {
        const Real *v = y + line * (n + 1);
        Real *out = to.field ? nullptr : R + size_t(line0 + line) * n;
        for (int i = lane; i < n; i += 64) {
            if (out) out[i] = v[i];
            const double f = static_cast<double>(v[i] * scaling);
            s1 += f;
            s2 += f * f;
            ++mine;
        }
    }
    for (int l0 = wave; to.field && l0 < count; l0 += kAhead * waves) {
        // kAhead lines together where each has one output line or none
        const Real *from[kAhead];
        Real *row[kAhead];
        bool simple = true;
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int line = l0 + u * waves, at = min(line, L - 1);
            const int jj = __shfl(j0, at), nj = __shfl(j1, at) - jj, kk = __shfl(k0, at), nk = __shfl(k1, at) - kk;
            from[u] = y + at * (n + 1);
            row[u] = line < count && nj * nk > 0 ? to.field + (size_t(kk) * to.ny + jj) * to.nx : nullptr;
            simple = simple && nj * nk <= 1 && (line0 + line) / n2 + 1 < lines / n2;
        }
        if (simple) {
            for (int i = lane; i < to.nx; i += 64) {
                const int node = to.x[i] - 1;
#pragma unroll
                for (int u = 0; u < kAhead; ++u)
                    if (row[u]) row[u][i] = from[u][node] * scaling;
            }
            continue;
        }
        for (int line = l0; line < min(count, l0 + kAhead * waves); line += waves) {
            const Real *v = y + line * (n + 1);
            const int ja = __shfl(j0, line), jb = __shfl(j1, line), ka = __shfl(k0, line), kb = __shfl(k1, line);
            auto put = [&](int kfirst, int kend) {
                for (int kk = kfirst; kk < kend; ++kk)
                    for (int jj = ja; jj < jb; ++jj) {
                        Real *out = to.field + (size_t(kk) * to.ny + jj) * to.nx;
                        for (int i = lane; i < to.nx; i += 64) out[i] = v[to.x[i] - 1] * scaling;
                    }
            };
            put(ka, kb);
            if ((line0 + line) / n2 + 1 == lines / n2) put(to.first_z[0], to.first_z[1]);
        }
    }
    Moments mo{double(mine), 0.0, 0.0};
    if (mine > 0) {
        mo.mean = s1 / mine;
        mo.m2 = s2 - s1 * mo.mean;
    }
    block_moments(mo, part + 3 * size_t(blockIdx.x));
}

template <class Real>
size_t columns_table(int n)
{
    return n > 1 ? (size_t(tiles(n)) * (depth(n) / 4) * 64 + n / 4 + 1 + 1) / 2 * 2 : 0;  // elements; rows stay aligned
}
template <class Real>
size_t rows_table(int n)
{
    return size_t(tiles(n)) * (depth(n) / 4) * 64;
}

// waves of a block: its tiles in as few equal turns as its registers and LDS allow
template <class Real>
int column_threads(int n, size_t lds)
{
    const int most = lds > kLds / 2 ? kColumnWaves<Real> : 8, turns = (tiles(n) + most - 1) / most;
    return 64 * std::max(4, (tiles(n) + turns - 1) / turns);
}

bool even(int n) { return n >= 2 && n % 2 == 0; }

bool large_prime(int n)
{
    for (int p : {2, 3, 5, 7, 11, 13})
        while (n % p == 0) n /= p;
    return n > 1;
}

template <class Real>
hipError_t columns_pass(Vec<Real, 2> *S, const Vec<Real, 2> *table, int n, long stride, int columns, long plane,
                        int planes, int careful, hipStream_t stream)
{
    const size_t lds = columns_lds<Real>(n);
    const int per_plane = (columns + 15) / 16;
    const long blocks = long(per_plane) * planes;
    auto kernel = &dft_columns<Real, Real, 4>;
    if constexpr (sizeof(Real) == 4) {
        if (n <= careful) kernel = &dft_columns<Real, double, 2>;
        if (n <= 64) kernel = &dft_columns<Real, double, 1>;
    }
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
    if (e != hipSuccess) return e;
    kernel<<<unsigned((blocks + kXcds - 1) / kXcds * kXcds), column_threads<Real>(n, lds), lds, stream>>>(
        S, table, n, stride, columns, plane, per_plane, blocks);
    return hipGetLastError();
}

}  // namespace

// The dense transform's work grows with the length, the FFT library's hardly
// does but triples at a prime factor above 13, where it runs Bluestein's
// algorithm, and its plan takes 0.5 to 2 s at the first call of a size
// (the tables here: 0.1 ms). Calls measured, dense against library, in ms:
//   a large prime factor   502^3 1.90 : 3.41, 258^3 0.35 : 0.75, 802 x 802 x 257 3.41 : 5.61,
//                          double 214 x 186 x 138 0.23 : 0.42, 2D 302 x 258 0.090 : 0.101,
//                          502 x 502 0.102 : 0.107, 614 x 402 0.113 : 0.113, 802 x 802 0.149 : 0.135
//   none                   32 x 48 x 40 0.078 : 0.093, 64^3 0.081 : 0.079, 96 x 120 x 64 0.089 : 0.106,
//                          128^3 0.115 : 0.112, 256^3 0.33 : 0.31,
//                          800 x 800 x 256 3.13 : 2.74, 2D 64 x 64 0.080 : 0.071, double 64^3 0.085 : 0.091,
//                          128^3 0.158 : 0.152, 256^3 0.65 : 0.52
// So: with a large prime factor every 3D grid whose lines fit the LDS, and 2D
// ones up to 640 (longer lines leave most of the chip without a block); without
// one only 3D grids of short lines.
template <class Real>
bool chosen(int n1, int n2, int n3)
{
    if (!even(n1) || !even(n2) || (n3 != 1 && !even(n3))) return false;
    const size_t lds = std::max({rows_lds<Real>(n1), columns_lds<Real>(n2), n3 > 1 ? columns_lds<Real>(n3) : 0});
    if (lds + 1024 > kLds || tiles(n1) > 16 || long(n1 / 2 + 1) * n2 >= (1L << 31)) return false;
    const int most = std::max({n1, n2, n3});
    if (large_prime(n1) || large_prime(n2) || large_prime(n3)) return n3 > 1 || most <= 640;
    if (n3 == 1) return false;
    return most <= (sizeof(Real) == 4 ? 128 : 64);
}

template <class Real>
size_t table_bytes(int n1, int n2, int n3)
{
    return sizeof(Vec<Real, 4>) * rows_table<Real>(n1) +
           sizeof(Vec<Real, 2>) * (columns_table<Real>(n2) + columns_table<Real>(n3));
}

template <class Real>
long parts(int, int n2, int n3)
{
    return (long(n2) * n3 + kRows<Real> - 1) / kRows<Real>;
}

template <class Real>
hipError_t make_tables(void *tables, int n1, int n2, int n3, hipStream_t stream)
{
    auto *x = static_cast<Vec<Real, 4> *>(tables);
    auto *y = reinterpret_cast<Vec<Real, 2> *>(x + rows_table<Real>(n1));
    dft_rows_table<Real><<<unsigned((rows_table<Real>(n1) + 255) / 256), 256, 0, stream>>>(x, n1);
    dft_columns_table<Real><<<unsigned((columns_table<Real>(n2) + 255) / 256), 256, 0, stream>>>(y, n2);
    if (n3 > 1)
        dft_columns_table<Real><<<unsigned((columns_table<Real>(n3) + 255) / 256), 256, 0, stream>>>(
            y + columns_table<Real>(n2), n3);
    return hipGetLastError();
}

template <class Real>
hipError_t run(void *S, Real *R, const Nearest<Real> &to, const void *tables, int n1, int n2, int n3, Real scaling,
               double *part, hipStream_t stream)
{
    auto *s = static_cast<Vec<Real, 2> *>(S);
    const auto *x = static_cast<const Vec<Real, 4> *>(tables);
    const auto *y = reinterpret_cast<const Vec<Real, 2> *>(x + rows_table<Real>(n1));
    const int h = n1 / 2 + 1;
    // float lines up to this length have FP64 totals (for_steps)
    const int careful = int(large_prime(n1)) + int(large_prime(n2)) + int(large_prime(n3)) <= 1 ? 288 : 128;
    hipError_t e = hipSuccess;
    if (n3 > 1)
        e = columns_pass<Real>(s, y + columns_table<Real>(n2), n3, long(h) * n2, h * n2, 0, 1, careful, stream);
    if (e == hipSuccess) e = columns_pass<Real>(s, y, n2, h, h, long(h) * n2, n3, careful, stream);
    if (e != hipSuccess) return e;
    const size_t lds = rows_lds<Real>(n1);
    auto kernel = &dft_rows<Real, Real, 4>;
    if constexpr (sizeof(Real) == 4) {
        if (n1 <= careful) kernel = &dft_rows<Real, double, 2>;
        if (n1 <= 64) kernel = &dft_rows<Real, double, 1>;
    }
    e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                            hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
    if (e != hipSuccess) return e;
    kernel<<<unsigned(parts<Real>(n1, n2, n3)), 64 * std::max(4, tiles(n1)), lds, stream>>>(
        s, R, to, x, n1, n2, n2 * n3, scaling, part);
    return hipGetLastError();
}

#define SCARF_FIM_DFT(Real)                                                                                        \
    template bool chosen<Real>(int, int, int);                                                                     \
    template size_t table_bytes<Real>(int, int, int);                                                              \
    template long parts<Real>(int, int, int);                                                                      \
    template hipError_t make_tables<Real>(void *, int, int, int, hipStream_t);                                     \
    template hipError_t run<Real>(void *, Real *, const Nearest<Real> &, const void *, int, int, int, Real, double *,   \
                                  hipStream_t);
SCARF_FIM_DFT(float)
SCARF_FIM_DFT(double)
#undef SCARF_FIM_DFT

}  // namespace fim_dft
}  // namespace scarf
