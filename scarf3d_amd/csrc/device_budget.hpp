// Device memory that the library's buffers hold, all objects together, and
// what a call may add to it. Buffers that carry nothing from one use to the
// next (workspaces, tables that are made again) belong to their owners as
// spares: they are given back when another buffer finds no room, so that a
// call needs no more room than what it computes from.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <functional>
#include <string>
#include <utility>
#include <vector>

namespace scarf {

class DeviceBudget {
public:
    size_t held() const { return held_; }
    void take(size_t bytes) { held_ += bytes; }
    void give(size_t bytes) { held_ -= bytes; }
    // Whether `more` bytes stay within SCARF_DEVICE_MEMORY_LIMIT=<bytes> (unset
    // or 0: no limit); the refusal in err.
    bool fits(size_t more, std::string *err = nullptr) const;

    // drop() frees the owner's spares, which no work in flight may use by then.
    // It allocates nothing.
    void add_spare(const void *owner, std::function<void()> drop) { spares_.emplace_back(owner, std::move(drop)); }
    void remove_spare(const void *owner);
    void drop_spares();

private:
    size_t held_ = 0;
    std::vector<std::pair<const void *, std::function<void()>>> spares_;
};

DeviceBudget &device_budget();

// hipMalloc of a buffer outside the account, the spares making room where the
// device has none left; leaves no error for the launch checks of other calls
hipError_t malloc_with_spares(void **ptr, size_t bytes);

}  // namespace scarf
