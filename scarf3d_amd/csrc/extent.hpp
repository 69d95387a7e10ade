// Smallest and largest value of an array, as one scan with std::min/std::max
// from the first value on finds them (values that are not numbers are passed
// over, unless the first is one).
#pragma once
#include <algorithm>
#include <cstddef>

namespace scarf {

// src[0, n) added to lo, hi: sixteen running extremes, which the compiler keeps
// in vector registers
template <class Real>
void add_extent(const Real *src, size_t n, Real &lo, Real &hi)
{
    Real l[16], h[16];
    std::fill(l, l + 16, lo);
    std::fill(h, h + 16, hi);
    size_t i = 0;
    for (; i + 16 <= n; i += 16)
        for (int q = 0; q < 16; ++q) {
            l[q] = src[i + q] < l[q] ? src[i + q] : l[q];
            h[q] = h[q] < src[i + q] ? src[i + q] : h[q];
        }
    for (; i < n; ++i) {
        l[0] = src[i] < l[0] ? src[i] : l[0];
        h[0] = h[0] < src[i] ? src[i] : h[0];
    }
    for (int q = 0; q < 16; ++q) {
        lo = std::min(lo, l[q]);
        hi = std::max(hi, h[q]);
    }
}

}  // namespace scarf
