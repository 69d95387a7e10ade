// Screening of the draw's trials on the GPU (see srm_host.hpp, TrialScreen):
// the seed's stream is generated and tested there and only the pairs that may
// pass come back.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "srm_host.hpp"

namespace scarf {

class TrialDevice : public TrialScreen {
public:
    TrialDevice();
    ~TrialDevice() override;
    TrialDevice(const TrialDevice &) = delete;
    TrialDevice &operator=(const TrialDevice &) = delete;

    bool screen(int seed, long first, long count, const TrialTest &test, const uint32_t *limit, int bins,
                TrialBlock &out) override;

private:
    bool reserve(size_t pairs_chunks, size_t records);
    void drop();  // the device's buffers; the last block of records stays in the host's memory
    hipStream_t stream_ = nullptr;
    void *d_gen_ = nullptr;      // generator tables
    uint32_t *d_limit_ = nullptr;  // and the count of records after it
    uint32_t *d_out_ = nullptr;    // spans of the chunks, records
    uint32_t *h_out_ = nullptr;    // pinned, written by the device: total, pairs, raw outputs
    uint32_t *h_limit_ = nullptr;
    size_t chunks_ = 0, records_ = 0;
};

}  // namespace scarf
