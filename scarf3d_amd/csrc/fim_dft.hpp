// Backward transform of the FIM half spectrum as products with dense cosine
// and sine matrices on the matrix cores: for lengths whose large prime factors
// leave a fast transform nothing but Bluestein's detour over twice the length.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace scarf {
namespace fim_dft {

// Whether a grid's transform runs here (the comment at the definition has the
// rule and both sides' times); otherwise it is left to the FFT library.
template <class Real>
bool chosen(int n1, int n2, int n3);

// bytes of the tables of a grid's three axes
template <class Real>
size_t table_bytes(int n1, int n2, int n3);

// blocks of the last pass: it writes that many moment triples
template <class Real>
long parts(int n1, int n2, int n3);

template <class Real>
hipError_t make_tables(void *tables, int n1, int n2, int n3, hipStream_t stream);

// Where the field goes when nothing changes it after the transform: output
// point (i, j, k) of an nx x ny x nz grid takes the node x[i] (1-based) of the
// line whose outputs along y include j and along z include k. A node v
// (1-based) has the outputs first[v] .. first[v + 1] - 1; node 0 along z is the
// last plane's copy beyond the first.
template <class Real>
struct Nearest {
    Real *field = nullptr;  // null: the transform is stored as it is
    int nx = 0, ny = 0;
    const int *x = nullptr, *first_y = nullptr, *first_z = nullptr;
};

// R = the real transform of the half spectrum S (complex, n1/2 + 1 x n2 x n3,
// overwritten), or its multiple by `scaling` at the nearest nodes of an output
// grid, and the moments of R * scaling as one triple per block.
template <class Real>
hipError_t run(void *S, Real *R, const Nearest<Real> &to, const void *tables, int n1, int n2, int n3, Real scaling,
               double *part, hipStream_t stream);

}  // namespace fim_dft
}  // namespace scarf
