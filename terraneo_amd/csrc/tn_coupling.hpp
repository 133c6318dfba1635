// Moments of the coarse pressure shapes on the fine wedges, shared by the two forms of
// B and B^T (kernels_stokes.hip, kernels_coupling_cells.hip).  Device-only header.
#pragma once

#include <hip/hip_runtime.h>

namespace tn {
namespace {

__device__ constexpr double GAUSS2 = 0.57735026918962576451;  // 1/sqrt(3)

// coarse lateral shape il on fine lateral wedge flw: alpha + beta xi + gamma eta
// (integrands.hpp:103-190; flw from kernel_helpers.hpp:600-608)
__host__ __device__ constexpr double coarse_lat_coef(int flw, int il, int k)
{
    constexpr double C[4][3][3] = {{{1.0, -0.5, -0.5}, {0.0, 0.5, 0.0}, {0.0, 0.0, 0.5}},
                                   {{0.5, -0.5, -0.5}, {0.5, 0.5, 0.0}, {0.0, 0.0, 0.5}},
                                   {{0.5, -0.5, -0.5}, {0.0, 0.5, 0.0}, {0.5, 0.0, 0.5}},
                                   {{0.0, 0.5, 0.5}, {0.5, -0.5, 0.0}, {0.5, 0.0, -0.5}}};
    return C[flw][il][k];
}

// int over the reference triangle of (alpha + beta xi + gamma eta) * {1, xi, eta}
struct LatMoments {
    double m[4][3][3];  // [flw][il][M0, Mx, Me]
};
__host__ __device__ constexpr LatMoments make_lat_moments()
{
    LatMoments r{};
    for (int f = 0; f < 4; ++f)
        for (int i = 0; i < 3; ++i) {
            const double al = coarse_lat_coef(f, i, 0), be = coarse_lat_coef(f, i, 1), ga = coarse_lat_coef(f, i, 2);
            r.m[f][i][0] = al / 2 + (be + ga) / 6;
            r.m[f][i][1] = al / 6 + be / 12 + ga / 24;
            r.m[f][i][2] = al / 6 + be / 24 + ga / 12;
        }
    return r;
}
__device__ constexpr LatMoments LATM = make_lat_moments();

__device__ inline int fine_lateral_wedge_idx(int xp, int yp, int w)
{
    // kernel_helpers.hpp:600-608 (xp, yp: parities of the fine quad indices)
    constexpr int ind[2][2][2] = {{{0, 1}, {2, 3}}, {{3, 2}, {1, 0}}};
    return ind[w][yp][xp];
}

}  // namespace
}  // namespace tn
