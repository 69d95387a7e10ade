// Trial screening on the GPU (see srm_draw.hpp).
//
// A pair of stream values passes as a trial when its second uniform is below
// the acceptance at its first. The host's table bounds the acceptance over
// equal bins of the first value, so `second < limit[first's bin]`, on the
// integers themselves, keeps every pair that passes; the exact test, whose
// roundings decide, runs on the host for the few pairs kept (0.3% of 6.6
// million at 512^3 x 20k). Integer arithmetic throughout: two steps of the
// generator and two powers of its primitive root per pair. The whole draw at
// 512^3 x 20k takes 0.67 ms of the host's clock, 10-12 ms with the stream
// generated and screened on its 16 threads (1024^2 x 512 x 50k: 1.26 against
// 18-20 ms).
#include "srm_draw.hpp"

#include <algorithm>
#include <cmath>
#include <cstdlib>

#include "fim_stream.hpp"

namespace scarf {
namespace {

using fim_stream::kPowWords;
using GenTables = fim_stream::Tables;

constexpr int kChunk = 2048;      // pairs of a wave, a multiple of 64 and at most 64 * 64
constexpr int kThreads = 512;
constexpr int kWaves = kThreads / 64;
constexpr int kBinsMax = 4096;
constexpr int kWords = TrialBlock::kWords;

struct ScreenArgs {
    uint32_t state[2];  // of stream position 0
    uint32_t pair64[4]; // A^128: 64 pairs on
    long first, count;
    int chunks, bins, shift;
    uint32_t records;   // capacity
};

// One wave per chunk of consecutive pairs, 64 at a time. The kept pairs'
// masks are held in LDS; the wave then claims room for them with one atomic
// and writes their records in stream order, the values of the pair and of the
// three after it (a harmonic's direction and amplitudes) recomputed from the
// chunk's first state. Bound by its integer multiplications.
__global__ __launch_bounds__(kThreads) void draw_screen(ScreenArgs a, const GenTables *__restrict__ gt,
                                                        const uint32_t *__restrict__ limit, uint2 *__restrict__ span,
                                                        uint32_t *__restrict__ total, uint32_t *__restrict__ rec)
{
    __shared__ uint32_t pw[kPowWords];
    __shared__ uint32_t lim[kBinsMax];
    __shared__ uint64_t masks[kWaves][kChunk / 64];
    for (int q = threadIdx.x; q < kPowWords; q += kThreads) pw[q] = gt->pw[q];
    for (int q = threadIdx.x; q < a.bins; q += kThreads) lim[q] = limit[q];
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    constexpr uint32_t step1[4] = {uint32_t(Yarn2::kA0), uint32_t(Yarn2::kA1), 1u, 0u};
    for (int chunk = blockIdx.x * kWaves + wave; chunk < a.chunks; chunk += gridDim.x * kWaves) {
        const long p0 = a.first + long(chunk) * kChunk;
        const int n = int(min(long(kChunk), a.first + a.count - p0));
        uint32_t b0 = a.state[0], b1 = a.state[1];
        fim_stream::jump(gt->jump, 2 * uint64_t(p0), b0, b1);
        uint32_t r0 = b0, r1 = b1;
        fim_stream::matvec(gt->lane[lane], r0, r1);
        fim_stream::matvec(gt->lane[lane], r0, r1);
        for (int it = 0; it < kChunk / 64; ++it) {
            uint32_t s0 = r0, s1 = r1;
            fim_stream::matvec(step1, s0, s1);
            const uint32_t v0 = fim_stream::value(pw, r0), v1 = fim_stream::value(pw, s0);
            const bool keep = it * 64 + lane < n && v1 < lim[v0 >> a.shift];
            const uint64_t m = __ballot(keep);
            if (lane == 0) masks[wave][it] = m;
            fim_stream::matvec(a.pair64, r0, r1);
        }
        __builtin_amdgcn_wave_barrier();
        uint64_t mine = lane < kChunk / 64 ? static_cast<volatile uint64_t *>(masks[wave])[lane] : 0;
        int inc = __popcll(mine);
        const int own = inc;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int o = __shfl_up(inc, off);
            if (lane >= off) inc += o;
        }
        const int tot = __shfl(inc, 63);
        uint32_t base = 0;
        if (lane == 0) {
            base = atomicAdd(total, uint32_t(tot));
            span[chunk] = make_uint2(base, uint32_t(tot));
        }
        uint32_t at = __shfl(base, 0) + uint32_t(inc - own);
        for (; mine; mine &= mine - 1, ++at) {
            if (at >= a.records) break;  // the host sees the total and redoes the block
            const int pair = lane * 64 + __ffsll(static_cast<unsigned long long>(mine)) - 1;
            uint32_t q0 = b0, q1 = b1;
            fim_stream::jump(gt->jump, 2 * uint64_t(pair), q0, q1);
            uint32_t *out = rec + size_t(kWords) * at;
            out[0] = uint32_t(p0 - a.first) + uint32_t(pair);
            for (int k = 1; k < kWords; ++k) {
                out[k] = fim_stream::value(pw, q0);
                fim_stream::matvec(step1, q0, q1);
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

__global__ void clear_total(uint32_t *total) { *total = 0; }

}  // namespace

TrialDevice::~TrialDevice()
{
    if (stream_) (void)hipStreamSynchronize(stream_);
    void *dev[] = {d_gen_, d_limit_, d_out_};
    for (void *p : dev)
        if (p) (void)hipFree(p);
    if (h_out_) (void)hipHostFree(h_out_);
    if (h_limit_) (void)hipHostFree(h_limit_);
    if (stream_) (void)hipStreamDestroy(stream_);
}

bool TrialDevice::room(size_t bytes) const
{
    const char *e = std::getenv("SCARF_DEVICE_MEMORY_LIMIT");
    const double limit = e ? std::atof(e) : 0.0;
    return !(limit > 0 && double(elsewhere_ + reserved_ + bytes) > limit);
}

// words of the header: a span per chunk, the total, padding to 16 bytes
static size_t header_words(size_t chunks) { return (2 * chunks + 1 + 3) / 4 * 4; }

bool TrialDevice::reserve(size_t chunks, size_t records)
{
    auto ok = [](hipError_t e) {
        if (e == hipSuccess) return true;
        (void)hipGetLastError();  // leaves no error for the launch checks of other calls
        return false;
    };
    if (!stream_ && !ok(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking))) return false;
    if (!d_gen_) {
        if (!room(sizeof(GenTables))) return false;
        GenTables t;
        fim_stream::make_tables(t);
        void *g = nullptr;
        if (!ok(hipMalloc(&g, sizeof t))) return false;
        if (!ok(hipMemcpy(g, &t, sizeof t, hipMemcpyHostToDevice))) {
            (void)hipFree(g);
            return false;
        }
        d_gen_ = g;
        reserved_ += sizeof t;
    }
    if (!d_limit_) {
        if (!room(kBinsMax * sizeof(uint32_t)) || !ok(hipMalloc(reinterpret_cast<void **>(&d_limit_), kBinsMax * sizeof(uint32_t))))
            return false;
        reserved_ += kBinsMax * sizeof(uint32_t);
    }
    if (!h_limit_ && !ok(hipHostMalloc(reinterpret_cast<void **>(&h_limit_), kBinsMax * sizeof(uint32_t), hipHostMallocDefault)))
        return false;
    if (chunks <= chunks_ && records <= records_ && d_out_ && h_out_) return true;
    const size_t old = (header_words(chunks_) + kWords * records_) * sizeof(uint32_t);
    const size_t c = std::max(chunks, chunks_), r = std::max(records, records_);
    const size_t bytes = (header_words(c) + kWords * r) * sizeof(uint32_t);
    if (d_out_) {
        (void)hipStreamSynchronize(stream_);
        (void)hipFree(d_out_);
        d_out_ = nullptr;
        reserved_ -= old;
    }
    if (h_out_) {
        (void)hipHostFree(h_out_);
        h_out_ = nullptr;
    }
    chunks_ = records_ = 0;
    if (!room(bytes) || !ok(hipMalloc(reinterpret_cast<void **>(&d_out_), bytes))) return false;
    if (!ok(hipHostMalloc(reinterpret_cast<void **>(&h_out_), bytes, hipHostMallocDefault))) {
        (void)hipFree(d_out_);
        d_out_ = nullptr;
        return false;
    }
    chunks_ = c;
    records_ = r;
    reserved_ += bytes;
    return true;
}

bool TrialDevice::screen(int seed, long first, long count, const uint32_t *limit, int bins, TrialBlock &out)
{
    int log2 = 0;
    while ((1 << log2) < bins) ++log2;
    // positions stay below the jump tables' 2^40 and a block's pair index below 2^32
    if (bins > kBinsMax || (1 << log2) != bins || first < 0 || count < 1 || count >= (1L << 31) ||
        2 * (first + count + 4) >= (1L << fim_stream::kJumpBits))
        return false;
    double share = 0.0;
    for (int b = 0; b < bins; ++b) share += std::min(1.0, double(limit[b]) / Yarn2::kModulus) / bins;
    const double mean = share * double(count);
    const size_t chunks = size_t((count + kChunk - 1) / kChunk);
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
    a.bins = bins;
    a.shift = 31 - log2;
    a.records = static_cast<uint32_t>(records);
    std::copy(limit, limit + bins, h_limit_);
    const size_t head = header_words(chunks);
    uint2 *span = reinterpret_cast<uint2 *>(d_out_);
    uint32_t *total = d_out_ + 2 * chunks, *rec = d_out_ + head;
    if (!ok(hipMemcpyAsync(d_limit_, h_limit_, size_t(bins) * sizeof(uint32_t), hipMemcpyHostToDevice, stream_))) return false;
    clear_total<<<1, 1, 0, stream_>>>(total);
    const int blocks = static_cast<int>(std::min<size_t>((chunks + kWaves - 1) / kWaves, 1024));
    draw_screen<<<blocks, kThreads, 0, stream_>>>(a, static_cast<const GenTables *>(d_gen_), d_limit_, span, total, rec);
    if (!ok(hipGetLastError())) return false;
    // header and records in one copy
    if (!ok(hipMemcpyAsync(h_out_, d_out_, (head + kWords * records) * sizeof(uint32_t), hipMemcpyDeviceToHost, stream_)) ||
        !ok(hipStreamSynchronize(stream_)))
        return false;
    if (h_out_[2 * chunks] > records) return false;
    out.start = first;
    out.end = first + count;
    out.spans = h_out_;
    out.chunks = chunks;
    out.records = h_out_ + head;
    out.total = h_out_[2 * chunks];
    return true;
}

}  // namespace scarf
