// Argument blocks of the Stokes coupling / mass kernels.
#pragma once

#include "tn_eps_march.hpp"
#include "tn_internal.hpp"

namespace tn {

// Coupling tables of a velocity mesh (kernels_stokes.hip): per fine node column
// COUPLING_SLOTS pairs of vectors, then the unit normal, padded to whole cache lines;
// per fine level six radial weights
constexpr int COUPLING_SLOTS = 7;
constexpr int COUPLING_NORMAL = 6 * COUPLING_SLOTS;
constexpr int COUPLING_ENTRIES = 48;
inline int64_t coupling_lat_elems(int nf) { return 10LL * nf * nf * COUPLING_ENTRIES; }
template <typename T>
void launch_coupling_tables(const double* coords, const double* radii, int n, int nr, T* lat, T* rad, hipStream_t s);

template <typename T>
struct DivArgs {
    const T* tab;  // coupling tables
    const T* rad;
    int nf, nrf, nc, nrc;
    int bc_cmb, bc_surf;
    const T* u;   // fine velocity [3][Nf]
    T* p;        // coarse pressure [Nc] (every copy written)
    int run = 0;  // columns per wave (set by the launcher)
};

template <typename T>
struct GradArgs {
    const T* tab;
    const T* rad;
    int nf, nrf, nc, nrc;
    int bc_cmb, bc_surf;
    const T* p;  // coarse pressure
    T* u;        // fine velocity
    int add;     // 1: u += B^T p, 0: u = B^T p
    int run = 0;  // set by the launcher: columns per wave,
    int tail = 0, tail_blocks = 0;  // levels past whole chunks that take a thread each, their blocks
};

// the same products by fine cells, for the solves (kernels_coupling_cells.hip)
template <typename T>
struct DivCellArgs {
    const double* coords;  // fine lateral coords
    const double* radii;   // fine radii
    int nf, nrf, nc, nrc;
    int bc_cmb, bc_surf;
    const T* u;  // fine velocity [3][Nf]
    T* p;        // coarse pressure [Nc] (every copy written)
    T* csum;     // scratch, div_scratch_elems(nc, nrc): per-cell corner sums, then the chunk tops
};
// scratch elements of B: 4 corners x (coarse cells + one top level per 64-cell chunk)
inline int64_t div_scratch_elems(int nc, int nrc)
{
    const int64_t ncol = 10LL * (nc - 1) * (nc - 1);
    return 4 * ncol * ((int64_t)(nrc - 1) + (nrc - 1 + 63) / 64);
}

template <typename T>
struct GradCellArgs {
    const double* coords;
    const double* radii;
    int nf, nrf, nc, nrc;
    int bc_cmb, bc_surf;
    const T* p;  // coarse pressure
    T* u;        // fine velocity
    int seg;     // node columns per block of the march
    int add;     // 1: u += B^T p, 0: u = B^T p
    MarchGuard guard;
};

// waves per block of the B^T march (node rows per block + 1): FP64 12 (one
// block per CU at 3 waves per SIMD, <= 168 VGPRs), FP32 8 (two blocks per CU)
template <typename T>
constexpr int grad_march_waves()
{
    return sizeof(T) == 8 ? 12 : 8;
}

template <typename T>
struct MassArgs {
    const double* radii;
    int n, nr, ncomp;
    const T* x;         // input field
    T* y;               // output, every node copy written (before the interface sum)
    const double* geo;  // the mesh's wedge table [10][n-1][n-1][2][GEO_STRIDE]
    double* dot = nullptr;  // optional: mass_blocks(n) partial sums of x . y over all node copies
};
int mass_blocks(int n);

template <typename T>
void launch_div(const DivArgs<T>& a, hipStream_t s);
template <typename T>
void launch_grad(const GradArgs<T>& a, hipStream_t s);
template <typename T>
void launch_div_cells(const DivCellArgs<T>& a, hipStream_t s);
template <typename T>
void launch_grad_cells(const GradCellArgs<T>& a, hipStream_t s);
template <typename T>
void launch_mass(const MassArgs<T>& a, hipStream_t s);
// lumped k-weighted mass of the nodal field k, every node copy written (before the interface sum)
template <typename T>
void launch_kmass_lumped(const double* coords, const double* radii, int n, int nr, const T* k, T* out, hipStream_t s);

}  // namespace tn
