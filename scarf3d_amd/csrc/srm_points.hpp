// The point-list SRM by way of a grid.
//
// The field is band-limited: |w_n| <= W per axis. On a grid of step pi / (2.5
// W), or pi / (2 W) in double, around the points it is known at every point by
// interpolation with the transform's compact kernel, if each harmonic is divided by the kernel's
// transform at its wavenumber first (the third nonuniform transform of Lee
// and Greengard, J. Comput. Phys. 206, 2005). The grid's values come from the
// plane-wise transform (srm_transform.hpp), so a point costs w^3 products
// (8^3 float, 16^3 double) whatever the number of harmonics.
#pragma once
#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "srm_transform.hpp"

namespace scarf {

struct PointsPlan {
    int w = 0;                // taps per axis of the interpolation
    double h[3] = {1, 1, 1}, x0[3] = {0, 0, 0}, beta = 0;
    bool flat = false;        // 2D: one plane, no taps along z
    Geometry g;               // the grid, in units of its steps
    TransformPlan grid;
    long npts = 0;
    int np_ = 0;
    bool sorted = false;      // points visited by blocks of bin^3 cells
    int bin = 16, bins[3] = {0, 0, 0};
    int nparts = 0;           // statistics partials
    size_t bytes = 0;
    size_t o_grid = 0, o_record = 0, o_work = 0, o_part = 0, o_count = 0, o_perm = 0;
};

// The interpolation's launches: a thread per point and tap would pass the 2^32
// threads that one launch can have (from 2^29 points in float, 2^28 in double),
// so each takes the points of 2^18 blocks, 8M in float and 4M in double.
struct PointsLaunch {
    long first = 0;  // point
    unsigned blocks = 0;
};
constexpr int kPointsThreads = 256;
constexpr long kPointsBlocks = 1L << 18;
std::vector<PointsLaunch> points_launches(long npts, bool f64);

// lo, hi: the points' extent; wmax: the largest |w| per axis of the record.
// False where the grid would be too large or the extent is not finite.
bool points_plan(const double lo[3], const double hi[3], const double wmax[3], bool flat, long npts, int np_, bool f64,
                 PointsPlan &plan);
// estimated device milliseconds, this way and by the direct sum
double points_ms(const PointsPlan &plan, bool f64);
double points_direct_ms(long npts, int np_, bool f64);

// d_pts: FP64 x, y, z blocks of npts values
template <class Real>
bool points_field(const PointsPlan &plan, const double *d_pts, const double *d_harm, void *ws, double scaling,
                  Real *d_field, double *d_part, hipStream_t stream, hipEvent_t tables_done, std::string &err);

}  // namespace scarf
