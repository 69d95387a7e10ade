// In-place complex Fourier transforms of lines held in LDS, sign +1,
// unnormalised, for lengths m * 2^a (m = 1, 3, 5, 7 or 9, a >= 4).
//
// Decimation in time: the input sits at digit-reversed positions, each pass
// reads and writes the same positions, so a pass needs one barrier and no
// second buffer, and the output is in natural order. The power-of-two radices
// come first, so every span but the full length is a power of two.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

namespace scarf {
namespace fft {

template <class Real>
struct Cplx {
    Real x, y;
};
template <class Real>
__device__ __forceinline__ Cplx<Real> operator+(Cplx<Real> a, Cplx<Real> b)
{
    return {a.x + b.x, a.y + b.y};
}
template <class Real>
__device__ __forceinline__ Cplx<Real> operator-(Cplx<Real> a, Cplx<Real> b)
{
    return {a.x - b.x, a.y - b.y};
}
template <class Real>
__device__ __forceinline__ Cplx<Real> mul(Cplx<Real> a, Cplx<Real> b)
{
    return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
template <class Real>
__device__ __forceinline__ Cplx<Real> mul_i(Cplx<Real> a)  // i a
{
    return {-a.y, a.x};
}

// element `offset` of an array at a uniform address, counted in 32 bits: the
// form that loads and stores take without address arithmetic
template <class T>
__device__ __forceinline__ const T &element(const T *p, unsigned offset)
{
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + offset * unsigned(sizeof(T)));
}
template <class T>
__device__ __forceinline__ T &element(T *p, unsigned offset)
{
    return *reinterpret_cast<T *>(reinterpret_cast<char *>(p) + offset * unsigned(sizeof(T)));
}

// a pass: radix | log2 of the span << 8
__host__ __device__ constexpr int kind_of(int radix, int shift) { return radix | shift << 8; }

// one empty element after every 16: lanes a power of two apart then fall on
// different LDS banks in the passes of small span
__host__ __device__ inline int pad(int i) { return i + (i >> 4); }
// line pitch, odd, so that lanes writing one position of consecutive lines do too
__host__ __device__ inline int pitch(int n) { return (n + (n >> 4)) | 1; }

template <class Real>
__device__ __forceinline__ void dft4(Cplx<Real> &a, Cplx<Real> &b, Cplx<Real> &c, Cplx<Real> &d)
{
    const Cplx<Real> s = a + c, t = a - c, u = b + d, v = mul_i(b - d);
    a = s + u;
    b = t + v;
    c = s - u;
    d = t - v;
}

// y[k] = sum_n x[n] e^{2 pi i n k / R}
template <int R, class Real>
__device__ __forceinline__ void dft(Cplx<Real> (&x)[R])
{
    using C = Cplx<Real>;
    if constexpr (R == 2) {
        const C t = x[1];
        x[1] = x[0] - t;
        x[0] = x[0] + t;
    } else if constexpr (R == 4) {
        dft4(x[0], x[1], x[2], x[3]);
    } else if constexpr (R == 8) {
        constexpr Real h = static_cast<Real>(0.70710678118654752440);
        C e[4] = {x[0], x[2], x[4], x[6]}, o[4] = {x[1], x[3], x[5], x[7]};
        dft4(e[0], e[1], e[2], e[3]);
        dft4(o[0], o[1], o[2], o[3]);
        o[1] = C{h * (o[1].x - o[1].y), h * (o[1].x + o[1].y)};
        o[2] = mul_i(o[2]);
        o[3] = C{h * (-o[3].x - o[3].y), h * (o[3].x - o[3].y)};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            x[k] = e[k] + o[k];
            x[k + 4] = e[k] - o[k];
        }
    } else if constexpr (R == 16) {
        constexpr Real h = static_cast<Real>(0.70710678118654752440);
        constexpr Real c = static_cast<Real>(0.92387953251128675613), s = static_cast<Real>(0.38268343236508977173);
        // n = 4 a + b, k = p + 4 q: columns over a, twiddles w16^(b p), rows over b
        C t[4][4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            dft4(x[b], x[4 + b], x[8 + b], x[12 + b]);
#pragma unroll
            for (int p = 0; p < 4; ++p) t[p][b] = x[4 * p + b];
        }
        t[1][1] = mul(t[1][1], C{c, s});
        t[1][2] = C{h * (t[1][2].x - t[1][2].y), h * (t[1][2].x + t[1][2].y)};
        t[1][3] = mul(t[1][3], C{s, c});
        t[2][1] = C{h * (t[2][1].x - t[2][1].y), h * (t[2][1].x + t[2][1].y)};
        t[2][2] = mul_i(t[2][2]);
        t[2][3] = C{h * (-t[2][3].x - t[2][3].y), h * (t[2][3].x - t[2][3].y)};
        t[3][1] = mul(t[3][1], C{s, c});
        t[3][2] = C{h * (-t[3][2].x - t[3][2].y), h * (t[3][2].x - t[3][2].y)};
        t[3][3] = mul(t[3][3], C{-c, -s});
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            dft4(t[p][0], t[p][1], t[p][2], t[p][3]);
#pragma unroll
            for (int q = 0; q < 4; ++q) x[p + 4 * q] = t[p][q];
        }
    } else if constexpr (R == 9) {
        // n = 3 a + b, k = p + 3 q
        constexpr Real w[3][2] = {{static_cast<Real>(0.76604444311897803520), static_cast<Real>(0.64278760968653932632)},
                                  {static_cast<Real>(0.17364817766693034885), static_cast<Real>(0.98480775301220805937)},
                                  {static_cast<Real>(-0.93969262078590838405), static_cast<Real>(0.34202014332566873304)}};
        C t[3][3];
#pragma unroll
        for (int b = 0; b < 3; ++b) {
            C col[3] = {x[b], x[3 + b], x[6 + b]};
            dft<3>(col);
#pragma unroll
            for (int p = 0; p < 3; ++p) t[p][b] = col[p];
        }
        t[1][1] = mul(t[1][1], C{w[0][0], w[0][1]});
        t[1][2] = mul(t[1][2], C{w[1][0], w[1][1]});
        t[2][1] = mul(t[2][1], C{w[1][0], w[1][1]});
        t[2][2] = mul(t[2][2], C{w[2][0], w[2][1]});
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            dft<3>(t[p]);
#pragma unroll
            for (int q = 0; q < 3; ++q) x[p + 3 * q] = t[p][q];
        }
    } else {
        // odd prime R: pairs (n, R - n) give the cosine and sine sums
        constexpr int H = R / 2;
        constexpr double cs[8][3] = {{}, {}, {}, {-0.5},
                                     {}, {0.30901699437494742410, -0.80901699437494742410},
                                     {}, {0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624}};
        constexpr double sn[8][3] = {{}, {}, {}, {0.86602540378443864676},
                                     {}, {0.95105651629515357212, 0.58778525229247312917},
                                     {}, {0.78183148246802980871, 0.97492791218182360702, 0.43388373911755812048}};
        C s[H], d[H];
        C sum = x[0];
#pragma unroll
        for (int q = 0; q < H; ++q) {
            s[q] = x[q + 1] + x[R - 1 - q];
            d[q] = x[q + 1] - x[R - 1 - q];
            sum = sum + s[q];
        }
        C out[R];
        out[0] = sum;
#pragma unroll
        for (int k = 1; k <= H; ++k) {
            C u = x[0], v = C{Real(0), Real(0)};
#pragma unroll
            for (int q = 1; q <= H; ++q) {
                const int r = (q * k) % R;
                const Real cc = static_cast<Real>(cs[R][(r <= H ? r : R - r) - 1]);
                const Real ss = static_cast<Real>(r <= H ? sn[R][r - 1] : -sn[R][R - r - 1]);
                u.x += cc * s[q - 1].x;
                u.y += cc * s[q - 1].y;
                v.x += ss * d[q - 1].x;
                v.y += ss * d[q - 1].y;
            }
            out[k] = u + mul_i(v);
            out[R - k] = u - mul_i(v);
        }
#pragma unroll
        for (int k = 0; k < R; ++k) x[k] = out[k];
    }
}

// A length's passes, for the device.
struct Passes {
    int n = 0, count = 0;
    int kind[6] = {};
    uint32_t magic[6] = {};  // 2^32 / (n / radix), rounded up: exact quotients for the counts of a block
};

// A barrier for LDS alone: loads from global memory stay in flight across it.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// One pass of radix R and span 2^S (S < 0: 2^shift, at least 16) over `lines`
// lines of n elements, behind a barrier. With the span known the positions of
// a butterfly are one address and constant offsets, and a span up to 64
// divides the block: every butterfly of a thread has the same twiddles, loaded
// before the barrier. They come from a table (one rounding each), not from
// products, in the order of the lanes: read at multiples of the butterfly's
// number they cost a cache line per lane, which bound the pass (512^3 float,
// y pass of 64 planes, 201 us; in order, 179 us). store(line, index, value)
// receives the outputs of a last pass; otherwise they go back to their places.
struct InPlace {};
template <int R, int S, class Real, class Store>
__device__ __forceinline__ void pass(Cplx<Real> *lds, const Cplx<Real> *__restrict__ tw, int n, uint32_t magic,
                                     int line_pitch, int lines, int shift, int tid, int threads, const Store &store)
{
    using C = Cplx<Real>;
    if constexpr (S >= 0) shift = S;
    const int per = n / R;
    const int span = 1 << shift;
    const int total = lines * per;
    auto off = [&](int r) {  // of element base + r * span
        if constexpr (S >= 0 && S < 4) return (r << S) + ((r << S) >> 4);
        else return r * (span + (span >> 4));
    };
    C t[R];
    auto twiddles = [&](int j) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 1; r < R; ++r) t[r] = element(tw + (r << shift), unsigned(j));
    };
    if constexpr (S > 0) twiddles(tid & (span - 1));
    lds_barrier();
    for (int q = tid; q < total; q += threads) {
        const int line = per == 1 ? q : static_cast<int>(__umulhi(static_cast<uint32_t>(q), magic));
        const int b = q - line * per;
        const int base = ((b >> shift) * R << shift) + (b & (span - 1));
        C *p = lds + line * line_pitch + pad(base);
        C x[R];
#pragma unroll
        for (int r = 0; r < R; ++r) x[r] = p[off(r)];
        if constexpr (S < 0) twiddles(base & (span - 1));
        if constexpr (S != 0) {
#pragma unroll
            for (int r = 1; r < R; ++r) x[r] = mul(x[r], t[r]);
        }
        dft<R>(x);
        if constexpr (std::is_same_v<Store, InPlace>) {
#pragma unroll
            for (int r = 0; r < R; ++r) p[off(r)] = x[r];
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if (r > 0 && r % 4 == 0) __builtin_amdgcn_sched_barrier(0);  // store's operands of 4 outputs at a time
                store(line, base + (r << shift), x[r]);
            }
        }
    }
}

// The passes from `first` on; the last one's outputs go to store. A barrier
// precedes every pass.
template <class Real, class Store>
__device__ __forceinline__ void transform(Cplx<Real> *lds, const Cplx<Real> *__restrict__ tw, int first,
                                          const Passes &plan, int line_pitch, int lines, int tid, int threads,
                                          const Store &store)
{
    for (int p = first; p < plan.count; ++p) {
        const int radix = plan.kind[p] & 255, shift = plan.kind[p] >> 8, n = plan.n;
        const uint32_t magic = plan.magic[p];
        asm volatile("" : "+v"(tid));  // keeps the addresses of all kinds of pass from being held over the loop
        auto go = [&](const auto &out) __attribute__((always_inline)) {
            if constexpr (sizeof(Real) == 4) {
                switch (plan.kind[p]) {
                case kind_of(16, 2): pass<16, 2>(lds, tw, n, magic, line_pitch, lines, shift, tid, threads, out); return;
                case kind_of(16, 3): pass<16, 3>(lds, tw, n, magic, line_pitch, lines, shift, tid, threads, out); return;
                case kind_of(16, 6): pass<16, 6>(lds, tw, n, magic, line_pitch, lines, shift, tid, threads, out); return;
                default: break;
                }
                if (radix == 16) {
                    pass<16, -1>(lds, tw, n, magic, line_pitch, lines, shift, tid, threads, out);
                    return;
                }
            }
            switch (plan.kind[p]) {
            case kind_of(4, 0): pass<4, 0>(lds, tw, n, magic, line_pitch, lines, shift, tid, threads, out); break;
            case kind_of(4, 2): pass<4, 2>(lds, tw, n, magic, line_pitch, lines, shift, tid, threads, out); break;
            case kind_of(8, 2): pass<8, 2>(lds, tw, n, magic, line_pitch, lines, shift, tid, threads, out); break;
            case kind_of(8, 0): pass<8, 0>(lds, tw, n, magic, line_pitch, lines, shift, tid, threads, out); break;
            case kind_of(2, 3): pass<2, 3>(lds, tw, n, magic, line_pitch, lines, shift, tid, threads, out); break;
            case kind_of(4, 3): pass<4, 3>(lds, tw, n, magic, line_pitch, lines, shift, tid, threads, out); break;
            case kind_of(8, 3): pass<8, 3>(lds, tw, n, magic, line_pitch, lines, shift, tid, threads, out); break;
            case kind_of(8, 6): pass<8, 6>(lds, tw, n, magic, line_pitch, lines, shift, tid, threads, out); break;
            default:
                switch (radix) {
                case 3: pass<3, -1>(lds, tw, n, magic, line_pitch, lines, shift, tid, threads, out); break;
                case 4: pass<4, -1>(lds, tw, n, magic, line_pitch, lines, shift, tid, threads, out); break;
                case 5: pass<5, -1>(lds, tw, n, magic, line_pitch, lines, shift, tid, threads, out); break;
                case 7: pass<7, -1>(lds, tw, n, magic, line_pitch, lines, shift, tid, threads, out); break;
                case 8: pass<8, -1>(lds, tw, n, magic, line_pitch, lines, shift, tid, threads, out); break;
                default: pass<9, -1>(lds, tw, n, magic, line_pitch, lines, shift, tid, threads, out); break;
                }
            }
        };
        if (p + 1 < plan.count) go(InPlace{});
        else go(store);
    }
}

// Radices of a length m * 2^a, `first` (4 or 8) first. wide: none above 8 and
// 9, since 16 FP64 values do not fit the registers.
__host__ inline Passes plan(int length, int first, bool wide)
{
    Passes p;
    p.n = length;
    int a = 0, shift = 0, n = length;
    while (n % 2 == 0) {
        n /= 2;
        ++a;
    }
    auto add = [&](int radix, int log2_radix) {
        const uint64_t per = length / radix;
        p.magic[p.count] = static_cast<uint32_t>((0x100000000ull + per - 1) / per);
        p.kind[p.count++] = kind_of(radix, shift);
        shift += log2_radix;
    };
    add(first, first == 4 ? 2 : 3);
    // the rest in 8s and 16s, and one 2 or 4 where it has to be
    static const int narrow_logs[12][4] = {{}, {1}, {2}, {3}, {4}, {3, 2}, {3, 3}, {3, 4}, {4, 4}, {3, 3, 3}, {3, 3, 4},
                                           {3, 4, 4}};
    static const int wide_logs[12][4] = {{}, {1}, {2}, {3}, {2, 2}, {3, 2}, {3, 3}, {3, 2, 2}, {3, 3, 2}, {3, 3, 3},
                                         {3, 3, 2, 2}, {3, 3, 3, 2}};
    const int *rest = (wide ? wide_logs : narrow_logs)[a - shift];
    for (int q = 0; q < 4 && rest[q] > 0; ++q) add(1 << rest[q], rest[q]);
    if (n > 1) add(n, 0);
    return p;
}

// Entry e of a plan's table of n twiddles: r j / (radix span) turns for
// e = r span + j, j < span, 0 < r < radix: the passes' ranges follow each other.
__device__ inline double turns(int e, const Passes &plan)
{
    int p = 0;
    while (p + 1 < plan.count && (1 << (plan.kind[p + 1] >> 8)) <= e) ++p;
    const int shift = plan.kind[p] >> 8, r = e >> shift, j = e & ((1 << shift) - 1);
    return double(r * j) / double((plan.kind[p] & 255) << shift);
}

// position of natural index k before the first pass
__host__ __device__ inline int digit_reverse(int k, const Passes &plan)
{
    int pos = 0, n = plan.n;
    for (int p = plan.count - 1; p >= 0; --p) {
        const int radix = plan.kind[p] & 255, q = k % radix;
        k /= radix;
        n /= radix;
        pos += q * n;
    }
    return pos;
}

}  // namespace fft
}  // namespace scarf
