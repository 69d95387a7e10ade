// Trial screening on the GPU (see srm_draw.hpp).
//
// A pair of stream values passes as a trial when its second uniform is below
// the acceptance at its first. The host's table bounds the acceptance over
// equal bins of the first value, so `second < limit[first's bin]`, on the
// integers themselves, keeps every pair that passes (0.35% of 6.4 million at
// 512^3 x 20k). Those get the test itself in FP64, with a margin that is wide
// against the roundings of the host's: what the margin leaves open (1e-5 of
// them in float) is the host's to decide, so the decisions are the host's.
// Integer arithmetic otherwise: two steps of the generator and two powers of
// its primitive root per pair. A second kernel puts the records in stream
// order and stores them in the host's memory: the host walked and tested them
// by chunk, one cache line after the other, in 320 us of the 600 that a draw
// took at 512^3 x 20k; now 300 in all, of which screening 110 and the
// harmonics 145 (500 harmonics: 180 -> 75 us; with the stream generated and
// screened on the host's 16 threads 10-12 ms at 20k).
#include "srm_draw.hpp"

#include <algorithm>
#include <cmath>
#include <cstdlib>

#include "device_budget.hpp"
#include "fim_stream.hpp"

namespace scarf {
namespace {

using fim_stream::kPowWords;
using GenTables = fim_stream::Tables;

constexpr int kRounds = 32;       // of 64 pairs, that a wave takes at most
constexpr int kThreads = 512;
constexpr int kWaves = kThreads / 64;
constexpr int kBinsMax = 4096;
constexpr int kRaw = TrialBlock::kRaw, kWords = kRaw + 1;
constexpr double kMostRecords = 1 << 20;  // expected ones, of a block
constexpr int kGroup = 64;  // chunks that a block puts in order

struct ScreenArgs {
    uint32_t state[2];  // of stream position 0
    uint32_t pair64[4]; // A^128: 64 pairs on
    long first, count;
    int chunks, rounds, bins, shift;  // a chunk is 64 * rounds pairs
    uint32_t records;   // capacity
    TrialTest test;
};

// The pair's verdict. `u` and whether it is above kc are the host's to the
// last bit (one rounding per operation), the acceptance to the margin.
template <class Real>
__device__ uint32_t verdict(const TrialTest &t, uint32_t v0, uint32_t v1)
{
    const Real r0 = static_cast<Real>(double(v0) / double(Yarn2::kModulus));
    const double r1 = static_cast<Real>(double(v1) / double(Yarn2::kModulus));
    Real u;
    if constexpr (sizeof(Real) == 4) u = __fadd_rn(__fmul_rn(r0, float(t.range)), float(t.kmin));
    else u = __dadd_rn(__dmul_rn(r0, t.range), t.kmin);
    const double x = u;
    double a = t.acf == 0 ? exp(-t.nu * log(1.0 + x * x)) : exp(-0.25 * (x * x));
    a *= (t.ndim == 3 ? x * x : x) * t.cnst;
    const double margin = sizeof(Real) == 4 ? 2e-5 : 1e-10;
    if (r1 < a * (1.0 - margin) && a > 1e-30) return u > static_cast<Real>(t.kc) ? TrialBlock::kDrop : TrialBlock::kKeep;
    if (r1 > a * (1.0 + margin) + 1e-30) return TrialBlock::kReject;
    return TrialBlock::kUnsure;
}

// One wave per chunk of consecutive pairs, 64 at a time. The kept pairs are
// listed in LDS; the wave then claims room for them with one atomic and writes
// their records in stream order, a lane each: the verdict and the values of
// the pair and of the three after it (a harmonic's direction and amplitudes),
// recomputed from the chunk's first state. Bound by its integer
// multiplications; a short draw by the length of a wave's chain, so that its
// chunks are short too.
__global__ __launch_bounds__(kThreads) void draw_screen(ScreenArgs a, const GenTables *__restrict__ gt,
                                                        const uint32_t *__restrict__ limit, uint2 *__restrict__ span,
                                                        uint32_t *__restrict__ total, uint32_t *__restrict__ rec)
{
    __shared__ uint32_t pw[kPowWords];
    __shared__ uint32_t lim[kBinsMax];
    __shared__ uint16_t list[kWaves][kRounds * 64];
    for (int q = threadIdx.x; q < kPowWords; q += kThreads) pw[q] = gt->pw[q];
    for (int q = threadIdx.x; q < a.bins; q += kThreads) lim[q] = limit[q];
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    constexpr uint32_t step1[4] = {uint32_t(Yarn2::kA0), uint32_t(Yarn2::kA1), 1u, 0u};
    for (int chunk = blockIdx.x * kWaves + wave; chunk < a.chunks; chunk += gridDim.x * kWaves) {
        const int pairs = 64 * a.rounds;
        const long p0 = a.first + long(chunk) * pairs;
        const int n = int(min(long(pairs), a.first + a.count - p0));
        uint32_t b0 = a.state[0], b1 = a.state[1];
        fim_stream::jump(gt->jump, 2 * uint64_t(p0), b0, b1);
        uint32_t r0 = b0, r1 = b1;
        fim_stream::matvec(gt->lane[lane], r0, r1);
        fim_stream::matvec(gt->lane[lane], r0, r1);
        int tot = 0;
        for (int it = 0; it < a.rounds; ++it) {
            uint32_t s0 = r0, s1 = r1;
            fim_stream::matvec(step1, s0, s1);
            const uint32_t v0 = fim_stream::value(pw, r0), v1 = fim_stream::value(pw, s0);
            const bool keep = it * 64 + lane < n && v1 < lim[v0 >> a.shift];
            const uint64_t m = __ballot(keep);
            if (keep) list[wave][tot + __popcll(m & ((1ull << lane) - 1))] = static_cast<uint16_t>(it * 64 + lane);
            tot += __popcll(m);
            fim_stream::matvec(a.pair64, r0, r1);
        }
        __builtin_amdgcn_wave_barrier();
        uint32_t base = 0;
        if (lane == 0) {
            base = atomicAdd(total, uint32_t(tot));
            span[chunk] = make_uint2(base, uint32_t(tot));
        }
        base = __shfl(base, 0);
        for (int i = lane; i < tot; i += 64) {
            const uint32_t at = base + uint32_t(i);
            if (at >= a.records) break;  // the host sees the total and redoes the block
            const int pair = static_cast<volatile uint16_t *>(list[wave])[i];
            uint32_t q0 = b0, q1 = b1;
            fim_stream::jump(gt->jump, 2 * uint64_t(pair), q0, q1);
            uint32_t *out = rec + size_t(kWords) * at;
            uint32_t v[kRaw];
#pragma unroll
            for (int k = 0; k < kRaw; ++k) {
                v[k] = fim_stream::value(pw, q0);
                fim_stream::matvec(step1, q0, q1);
            }
            const uint32_t how = a.test.f64 ? verdict<double>(a.test, v[0], v[1]) : verdict<float>(a.test, v[0], v[1]);
            out[0] = (uint32_t(p0 - a.first) + uint32_t(pair)) | how << 30;
#pragma unroll
            for (int k = 0; k < kRaw; ++k) out[1 + k] = v[k];
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// The records in stream order, into the host's memory: a block finds the
// position of its kGroup chunks' first record from the spans before them.
__global__ __launch_bounds__(kThreads) void draw_order(int chunks, uint32_t records, const uint2 *__restrict__ span,
                                                       const uint32_t *__restrict__ total,
                                                       const uint32_t *__restrict__ rec, uint32_t *__restrict__ out)
{
    __shared__ uint32_t part[kWaves], end[kGroup], base[kGroup];
    if (blockIdx.x == 0 && threadIdx.x == 0) out[0] = *total;
    if (*total > records) return;  // the host gives the block up
    const int c0 = blockIdx.x * kGroup, c1 = min(c0 + kGroup, chunks);
    uint32_t sum = 0;
    for (int c = threadIdx.x; c < c0; c += kThreads) sum += span[c].y;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) sum += __shfl_xor(sum, off);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = sum;
    __syncthreads();
    uint32_t at = 0;
    for (int w = 0; w < kWaves; ++w) at += part[w];
    if (threadIdx.x < 64) {
        const uint2 s = c0 + int(threadIdx.x) < c1 ? span[c0 + threadIdx.x] : make_uint2(0, 0);
        uint32_t upto = s.y;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t o = __shfl_up(upto, off);
            if (int(threadIdx.x) >= off) upto += o;
        }
        end[threadIdx.x] = upto;
        base[threadIdx.x] = s.x - (upto - s.y);  // of record 0 of the group, were it this chunk's
    }
    __syncthreads();
    uint32_t *pairs = out + 4 + at, *raw = out + 4 + (records + 3) / 4 * 4 + size_t(kRaw) * at;
    for (uint32_t e = threadIdx.x; e < end[kGroup - 1] * kWords; e += kThreads) {
        const uint32_t i = e / kWords, k = e - i * kWords;
        int c = 0;  // the chunk of record i
#pragma unroll
        for (int half = kGroup / 2; half >= 1; half /= 2)
            if (end[c + half - 1] <= i) c += half;
        const uint32_t v = rec[size_t(kWords) * (base[c] + i) + k];
        if (k == 0) pairs[i] = v;
        else raw[size_t(kRaw) * i + k - 1] = v;
    }
}

}  // namespace

TrialDevice::TrialDevice()
{
    device_budget().add_spare(this, [this] { drop(); });
}

TrialDevice::~TrialDevice()
{
    device_budget().remove_spare(this);
    drop();
    if (h_out_) (void)hipHostFree(h_out_);
    if (h_limit_) (void)hipHostFree(h_limit_);
    if (stream_) (void)hipStreamDestroy(stream_);
}

// words of the device's block: a span per chunk, the records; of the host's:
// the total, the pairs, the outputs
static size_t device_words(size_t chunks, size_t records) { return (2 * chunks + 3) / 4 * 4 + kWords * records; }
static size_t host_words(size_t records) { return 4 + (records + 3) / 4 * 4 + kRaw * records; }

constexpr size_t kLimitBytes = (kBinsMax + 1) * sizeof(uint32_t);

void TrialDevice::drop()
{
    if (stream_) (void)hipStreamSynchronize(stream_);
    auto free = [](void *p, size_t bytes) {
        if (!p) return;
        (void)hipFree(p);
        device_budget().give(bytes);
    };
    free(d_gen_, sizeof(GenTables));
    free(d_limit_, kLimitBytes);
    free(d_out_, device_words(chunks_, records_) * sizeof(uint32_t));
    d_gen_ = nullptr;
    d_limit_ = d_out_ = nullptr;
    chunks_ = records_ = 0;
}

bool TrialDevice::reserve(size_t chunks, size_t records)
{
    DeviceBudget &budget = device_budget();
    auto ok = [](hipError_t e) {
        if (e == hipSuccess) return true;
        (void)hipGetLastError();  // leaves no error for the launch checks of other calls
        return false;
    };
    if (!stream_ && !ok(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking))) return false;
    if (!d_gen_) {
        if (!budget.fits(sizeof(GenTables))) return false;
        GenTables t;
        fim_stream::make_tables(t);
        void *g = nullptr;
        if (!ok(hipMalloc(&g, sizeof t))) return false;
        if (!ok(hipMemcpy(g, &t, sizeof t, hipMemcpyHostToDevice))) {
            (void)hipFree(g);
            return false;
        }
        d_gen_ = g;
        budget.take(sizeof t);
    }
    if (!d_limit_) {
        void *p = nullptr;
        if (!budget.fits(kLimitBytes) || !ok(hipMalloc(&p, kLimitBytes))) return false;
        d_limit_ = static_cast<uint32_t *>(p);
        budget.take(kLimitBytes);
    }
    if (!h_limit_) {
        void *p = nullptr;
        if (!ok(hipHostMalloc(&p, kLimitBytes, hipHostMallocDefault))) return false;
        h_limit_ = static_cast<uint32_t *>(p);
    }
    if (chunks <= chunks_ && records <= records_ && d_out_ && h_out_) return true;
    const size_t old = device_words(chunks_, records_) * sizeof(uint32_t);
    const size_t c = std::max(chunks, chunks_), r = std::max(records, records_);
    const size_t bytes = device_words(c, r) * sizeof(uint32_t);
    if (d_out_) {
        (void)hipStreamSynchronize(stream_);
        (void)hipFree(d_out_);
        d_out_ = nullptr;
        budget.give(old);
    }
    if (h_out_) {
        (void)hipHostFree(h_out_);
        h_out_ = nullptr;
    }
    chunks_ = records_ = 0;
    void *d = nullptr, *h = nullptr;
    if (!budget.fits(bytes) || !ok(hipMalloc(&d, bytes))) return false;
    if (!ok(hipHostMalloc(&h, host_words(r) * sizeof(uint32_t), hipHostMallocDefault))) {
        (void)hipFree(d);
        return false;
    }
    d_out_ = static_cast<uint32_t *>(d);
    h_out_ = static_cast<uint32_t *>(h);
    chunks_ = c;
    records_ = r;
    budget.take(bytes);
    return true;
}

bool TrialDevice::screen(int seed, long first, long count, const TrialTest &test, const uint32_t *limit, int bins,
                         TrialBlock &out)
{
    int log2 = 0;
    while ((1 << log2) < bins) ++log2;
    // positions stay below the jump tables' 2^40 and a block's pair index below 2^30
    if (bins > kBinsMax || (1 << log2) != bins || first < 0 || count < 1 || count >= (1L << 30) ||
        2 * (first + count + 4) >= (1L << fim_stream::kJumpBits))
        return false;
    double share = 0.0;
    for (int b = 0; b < bins; ++b) share += std::min(1.0, double(limit[b]) / Yarn2::kModulus) / bins;
    // the records of a block take 36 bytes each here and in pinned memory: a
    // long draw takes several blocks
    if (share * double(count) > kMostRecords) count = std::max(4L, static_cast<long>(kMostRecords / share));
    const double mean = share * double(count);
    const int rounds = static_cast<int>(std::clamp(count / (64L * 1024), 1L, long(kRounds)));
    const size_t chunks = size_t((count + 64L * rounds - 1) / (64L * rounds));
    const size_t records = size_t(mean + 10.0 * std::sqrt(mean + 1.0) + 256.0);
    if (!reserve(chunks, records)) return false;
    auto ok = [](hipError_t e) {
        if (e == hipSuccess) return true;
        (void)hipGetLastError();
        return false;
    };
    ScreenArgs a{};
    fim_stream::position0(seed, a.state);
    fim_stream::power(128, a.pair64);
    a.first = first;
    a.count = count;
    a.chunks = static_cast<int>(chunks);
    a.rounds = rounds;
    a.bins = bins;
    a.shift = 31 - log2;
    a.records = static_cast<uint32_t>(records);
    a.test = test;
    std::copy(limit, limit + bins, h_limit_);
    h_limit_[bins] = 0;  // the count of records
    uint2 *span = reinterpret_cast<uint2 *>(d_out_);
    uint32_t *total = d_limit_ + bins, *rec = d_out_ + (2 * chunks + 3) / 4 * 4;
    if (!ok(hipMemcpyAsync(d_limit_, h_limit_, size_t(bins + 1) * sizeof(uint32_t), hipMemcpyHostToDevice, stream_)))
        return false;
    const int blocks = static_cast<int>(std::min<size_t>((chunks + kWaves - 1) / kWaves, 1024));
    draw_screen<<<blocks, kThreads, 0, stream_>>>(a, static_cast<const GenTables *>(d_gen_), d_limit_, span, total, rec);
    if (!ok(hipGetLastError())) return false;
    draw_order<<<static_cast<int>((chunks + kGroup - 1) / kGroup), kThreads, 0, stream_>>>(
        static_cast<int>(chunks), a.records, span, total, rec, h_out_);
    if (!ok(hipGetLastError()) || !ok(hipStreamSynchronize(stream_))) return false;
    if (h_out_[0] > records) return false;
    out.start = first;
    out.end = first + count;
    out.pairs = h_out_ + 4;
    out.raw = out.pairs + (records + 3) / 4 * 4;
    out.total = h_out_[0];
    return true;
}

}  // namespace scarf
