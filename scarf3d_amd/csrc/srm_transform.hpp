// The structured-grid SRM as a fast transform.
//
// On one z plane the field is a nonuniform Fourier sum over the two grid axes,
//   F(i, j) = Re sum_n c_n(z) e^{i (wx_n ds i + wy_n ds j)},
//   c_n(z) = amp_n e^{i (wz_n z + phase_n)},
// evaluated by spreading every harmonic onto an oversampled grid of
// frequencies with a compact kernel, a Fourier transform of that grid, and a
// division by the kernel's transform (Dutt and Rokhlin, SIAM J. Sci. Comput.
// 14, 1993; Kaiser-Bessel kernel as in Jackson et al., IEEE Trans. Med.
// Imaging 10, 1991). The cost per value is that of two 1D transforms and
// hardly depends on the number of harmonics, where the direct sums and the
// GEMM take one operation or more per point and harmonic. z stays a direct
// sum: planes are independent, and a plane's values depend on its own z only.
//
// Measured, tables + field + statistics: float 512^3 x 20k 2.0 ms (mfma_bf16x3
// 47.6, direct_f32 270), 128^3 x 5k 0.13 ms (0.44, 1.7); double 128^3 x 5k
// 0.20 ms (direct_f64 13.9). 2-norm error against the FP64 sum 1.4e-7 (4e-7,
// 2.5e-7) in float; against extended precision 2.8e-15 (3.8e-15) in double, 128
// x 100 x 60 x 4000.
#pragma once
#include <hip/hip_runtime.h>

#include <string>

#include "fft_lds.hpp"
#include "srm_device.hpp"

namespace scarf {

struct TransformPlan {
    int w = 0;             // kernel taps per axis
    int nx = 0, ny = 0, nz = 0;
    int m = 0;             // x: half the oversampled length
    int l = 0;             // y: oversampled length, a multiple of 16
    int columns = 0;       // kept kx columns, -w/2 .. m + w - 1 - w/2
    fft::Passes fx, fy;    // lengths m (complex, for 2m reals) and l
    double beta_x = 0, beta_y = 0;
    int zb = 0, yb = 0;    // z planes per block of the y pass, y lines per block of the x pass
    bool wide = false;     // y pass: one block of 1024 threads per CU
    int slab = 0;          // z planes per round of both passes
    int np_ = 0;           // padded harmonic count
    int nparts = 0;        // statistics partials, one per block of the x pass
    int groups = 0;        // their merged groups
    size_t bytes = 0;      // workspace
    // workspace offsets
    size_t o_key = 0, o_order = 0, o_start = 0, o_last = 0, o_taps = 0, o_tw = 0, o_rev = 0, o_dec = 0,
           o_wave = 0, o_t = 0;
};

// False where the grid's lines are too long for the transform's LDS lines.
bool transform_plan(const Geometry &g, int np_, bool f64, TransformPlan &plan);
// Estimated device milliseconds of the transform and of the direct-sum kernel
// `kernel` on the same grid, from measured rates, to choose between them.
double transform_ms(const TransformPlan &plan, bool f64);
double direct_ms(const Geometry &g, int nharm, int kernel);

// Tables, field and statistics partials of the resident record (np_ values per
// field) in the workspace of plan.bytes. d_part: plan.nparts triples, then the
// plan.groups that they are merged into.
template <class Real>
bool transform_field(const TransformPlan &plan, const Geometry &g, const double *d_harm, void *ws, double scaling,
                     Real *d_field, double *d_part, hipStream_t stream, hipEvent_t tables_done, std::string &err);

}  // namespace scarf
