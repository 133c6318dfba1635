// Hex finite-volume energy step: flux-corrected transport (FCT) of a scalar
// by the Stokes velocity, with two-point diffusion (FP64).
//
// Reference: fv/hex/operators/fct_advection_diffusion.hpp (stages),
// fv/hex/operators/geometry_helper.hpp:178-360 (cell geometry),
// fv/hex/helpers.hpp:64-190 (Dirichlet values, cell centres),
// fv/hex/conversion.hpp:131-211 (FV -> FE projection right-hand side),
// communication/shell/fv_communication.hpp (ghost layers).
//
// FV fields carry one ghost layer: [10][n+1][n+1][nr+1], r fastest; real
// cells (xc, yc, rc) in [1, n-1]^2 x [1, nr-1] are the FE hex cells
// (xc-1, yc-1, rc-1).  A kernel runs one thread per real cell (or per
// FE node for the projection), radially consecutive threads on radially
// consecutive cells, so every field access of a wave is one contiguous
// radial run; the stable step and the predictor walk along columns where the mesh
// fills their lanes (walk_columns).  Nothing is accumulated with atomics: every output element is
// written by one thread, so results repeat bit for bit.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "tn_eps_march.hpp"
#include "tn_fv.hpp"
#include "tn_march.hpp"

namespace tn {

namespace {

constexpr int FV_BLOCK = 256;

__device__ __forceinline__ int64_t fvi(int n, int nr, int d, int x, int y, int r)
{
    return (((int64_t)d * (n + 1) + x) * (n + 1) + y) * (nr + 1) + r;
}

// wedge local node offsets (kernel_helpers.hpp:302-327)
__constant__ int FV_WOFF[2][6][3] = {{{0, 0, 0}, {1, 0, 0}, {0, 1, 0}, {0, 0, 1}, {1, 0, 1}, {0, 1, 1}},
                                     {{1, 1, 0}, {0, 1, 0}, {1, 0, 0}, {1, 1, 1}, {0, 1, 1}, {1, 0, 1}}};

// Felippa 3x2 wedge rule (fe/wedge/quadrature/quadrature.hpp:67-110): triangle
// points (2/3,1/6), (1/6,2/3), (1/6,1/6) at zeta = -+1/sqrt(3), weight 1/6
constexpr double QT_A = 0.6666666666666666, QT_B = 0.1666666666666667, QZ = 0.5773502691896257,
                 QW = 0.1666666666666667;

__device__ __forceinline__ void cell_real(int64_t t, int n, int nr, int& d, int& xc, int& yc, int& rc)
{
    rc = 1 + (int)(t % (nr - 1));
    t /= (nr - 1);
    yc = 1 + (int)(t % (n - 1));
    t /= (n - 1);
    xc = 1 + (int)(t % (n - 1));
    d = (int)(t / (n - 1));
}

// lateral corner positions of the two wedges of FE hex cell (x, y)
__device__ __forceinline__ void wedge_corners(const double* __restrict__ coords, int n, int d, int x, int y,
                                              double P[2][3][3])
{
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const double* c = coords + 3 * (((int64_t)d * n + x + FV_WOFF[w][i][0]) * n + y + FV_WOFF[w][i][1]);
            P[w][i][0] = c[0];
            P[w][i][1] = c[1];
            P[w][i][2] = c[2];
        }
}

// |det J| of the wedge map x = r(zeta) L(xi, eta) at (xi, eta, zeta)
// (integrands.hpp:623-670): det [r (p1-p0), r (p2-p0), (dr/2) L]
__device__ __forceinline__ double abs_det(const double P[3][3], double r1, double r2, double xi, double eta,
                                          double zeta)
{
    const double r = r1 + 0.5 * (r2 - r1) * (1 + zeta);
    const double gr = 0.5 * (r2 - r1);
    double J[3][3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        J[a][0] = (P[1][a] - P[0][a]) * r;
        J[a][1] = (P[2][a] - P[0][a]) * r;
        J[a][2] = ((1 - xi - eta) * P[0][a] + xi * P[1][a] + eta * P[2][a]) * gr;
    }
    const double det = J[0][0] * (J[1][1] * J[2][2] - J[1][2] * J[2][1]) -
                       J[0][1] * (J[1][0] * J[2][2] - J[1][2] * J[2][0]) +
                       J[0][2] * (J[1][0] * J[2][1] - J[1][1] * J[2][0]);
    return fabs(det);
}

__device__ __forceinline__ void qpoint(int q, double& xi, double& eta, double& zeta)
{
    const int k = q % 3;
    xi = k == 0 ? QT_A : QT_B;
    eta = k == 1 ? QT_A : QT_B;
    zeta = q < 3 ? -QZ : QZ;
}

// Geometry of real FV cell (d, xc, yc, rc): beta[f] = int_face u.n dS and
// S[f] = int_face n dS (faces 0: x-1, 1: x+1, 2: y-1, 3: y+1, 4: r-1, 5: r+1),
// each oriented towards the neighbour's centre, and the cell volume M.
//
// The reference integrates the faces with 2 x 2 Gauss points (lateral faces)
// and the 3-point triangle rule on both wedges (radial faces), and the volume
// with the Felippa 3x2 rule.  With the wedge map X = rho(zeta) L(xi, eta)
// (rho linear from r1 to r2, L on the flat triangle V0 V1 V2, h = (r2-r1)/2)
// these rules are exact, and the integrals have closed forms:
//   lateral face xi = 0 of a wedge:  n = rho h (V2 x V0), nodes V0, V2
//   lateral face eta = 0:            n = rho h (V1 x V0), nodes V0, V1
//     S = h (r1 + r2) (Vb x Va),
//     beta = h (Vb x Va) . [ab (u_a,bot + u_b,bot) + at (u_a,top + u_b,top)] / 2,
//     ab = (2 r1 + r2) / 3, at = (r1 + 2 r2) / 3     (int rho (1 -+ zeta)/2 dzeta)
//   radial face at radius rr (r1 bottom, r2 top), summed over both wedges:
//     n = rr^2 (V1 - V0) x (V2 - V0),  S = n / 2,  beta = n . (u_0 + u_1 + u_2) / 6
//   volume: sum over the wedges of |det(V0, V1, V2)| (r2^3 - r1^3) / 6
// so the results equal the reference's quadrature up to rounding.
__device__ __forceinline__ void cross3(const double a[3], const double b[3], double o[3])
{
    o[0] = a[1] * b[2] - a[2] * b[1];
    o[1] = a[2] * b[0] - a[0] * b[2];
    o[2] = a[0] * b[1] - a[1] * b[0];
}

// Lateral part of the geometry of hex column (d, x, y), the same at every
// radius.  Corners c00 = (x, y), c10 = (x+1, y), c01 = (x, y+1), c11 = (x+1, y+1);
// wedge 0: V0 = c00, V1 = c10, V2 = c01; wedge 1: W0 = c11, W1 = c01, W2 = c10.
// Lateral faces (face, Va, Vb), normal Vb x Va: 0 (c00, c01) xi = 0 of wedge 0:
// n ~ V2 x V0 = c01 x c00; 2 (c00, c10) eta = 0 of wedge 0: V1 x V0 = c10 x c00;
// 1 (c11, c10): W2 x W0 = c10 x c11; 3 (c11, c01): W1 x W0 = c01 x c11.
__device__ __forceinline__ void column_corners(const double* __restrict__ coords, int n, int d, int x, int y,
                                               double c[4][3])
{
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const double* p = coords + 3 * (((int64_t)d * n + x + (k & 1)) * n + y + (k >> 1));
        c[k][0] = p[0];
        c[k][1] = p[1];
        c[k][2] = p[2];
    }
}
// |det(V0, V1, V2)| of the two wedges (= V0 . (V1 x V2))
__device__ __forceinline__ void column_dets(const double c[4][3], double det[2])
{
    double v12[3], w12[3];
    cross3(c[1], c[2], v12);
    cross3(c[2], c[1], w12);
    det[0] = fabs(c[0][0] * v12[0] + c[0][1] * v12[1] + c[0][2] * v12[2]);
    det[1] = fabs(c[3][0] * w12[0] + c[3][1] * w12[1] + c[3][2] * w12[2]);
}

__device__ __forceinline__ double dot3d(const double a[3], const double b[3])
{
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
}

// The layer's part of a cell's geometry, held in a lane's registers: the flux
// factors and, times kappa, the diffusion factors of the faces.
struct Layer {
    double r1, r2, hh;     // radii, (r2 - r1) / 4 (half of h, the mean of the two node levels' weights)
    double ab, at;         // weights of the bottom / top velocities in a lateral face
    double q1, q2;         // r^2 / 6 of the radial faces, signed with the layers' order
    double kl, k4, k5;     // diffusion factors: lateral, radial bottom, radial top
    double vol;            // (r2^3 - r1^3) / 6
    __device__ void set(const FvArgs& a, int rc, double kappa)
    {
        r1 = a.radii[rc - 1];
        r2 = a.radii[rc];
        const double s0 = a.layers[rc - 1], s1 = a.layers[rc], s2 = a.layers[rc + 1];
        const double h = 0.5 * (r2 - r1);
        hh = 0.5 * h;
        ab = (2.0 * r1 + r2) / 3.0;
        at = (r1 + 2.0 * r2) / 3.0;
        q1 = (s0 < s1 ? -1.0 : 1.0) * (r1 * r1 / 6.0);
        q2 = (s2 < s1 ? -1.0 : 1.0) * (r2 * r2 / 6.0);
        kl = kappa * (h * (r1 + r2) / s1);
        k4 = kappa * (0.5 * r1 * r1 / fabs(s0 - s1));
        k5 = kappa * (0.5 * r2 * r2 / fabs(s2 - s1));
        vol = (r2 - r1) * (r1 * r1 + r1 * r2 + r2 * r2) / 6.0;  // without cancellation
    }
};

// A corner column's velocity on one layer: bottom and top node, and their
// combination in the lateral faces
struct CornerVel {
    double b[3], t[3], l[3];
    __device__ __forceinline__ void load(const double* __restrict__ vel, int64_t N, int64_t node)
    {
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            b[j] = vel[j * N + node];
            t[j] = vel[j * N + node + 1];
        }
    }
    __device__ __forceinline__ void combine(const Layer& L)
    {
#pragma unroll
        for (int j = 0; j < 3; ++j) l[j] = L.ab * b[j] + L.at * t[j];
    }
};

// Face fluxes beta (towards the neighbours), diffusion coefficients and volume of
// a cell from its column's table g, its layer and the corners c00, c10, c01, c11.
__device__ __forceinline__ void cell_faces(const double* __restrict__ g, const Layer& L, const CornerVel& c00,
                                           const CornerVel& c10, const CornerVel& c01, const CornerVel& c11,
                                           double beta[6], double dc[6], double& M)
{
    double f0 = 0, f1 = 0, f2 = 0, f3 = 0, bb = 0, bt = 0;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        f0 += g[j] * (c00.l[j] + c01.l[j]);
        f1 += g[3 + j] * (c11.l[j] + c10.l[j]);
        f2 += g[6 + j] * (c00.l[j] + c10.l[j]);
        f3 += g[9 + j] * (c11.l[j] + c01.l[j]);
        bb += g[12 + j] * (c00.b[j] + c10.b[j] + c01.b[j]) + g[15 + j] * (c11.b[j] + c01.b[j] + c10.b[j]);
        bt += g[12 + j] * (c00.t[j] + c10.t[j] + c01.t[j]) + g[15 + j] * (c11.t[j] + c01.t[j] + c10.t[j]);
    }
    beta[0] = L.hh * f0;
    beta[1] = L.hh * f1;
    beta[2] = L.hh * f2;
    beta[3] = L.hh * f3;
    beta[4] = g[19] * (L.q1 * bb);
    beta[5] = g[19] * (L.q2 * bt);
#pragma unroll
    for (int f = 0; f < 4; ++f) dc[f] = L.kl * g[20 + f];
    dc[4] = L.k4 * g[24];
    dc[5] = L.k5 * g[24];
    M = g[18] * L.vol;
}

// The hex columns of a block: FV_STRIPS waves on neighbouring strips x of one
// diamond and one chunk of 64 layers, marching together along y, so that a column
// of nodes or cells that two strips share is read into the caches at one time
// (with strips far apart the stable step took 258 us and the predictor 710 us at
// level 7 x 129, with the loads of a column issued in its own step 231 and 756 us,
// a step ahead of the stores 233 and 650 us; call times, the predictor as a stage of
// its own).  The columns of all strip groups
// are split evenly over the blocks.  The corner velocities shared by consecutive
// columns stay in registers.  f.load(pre, d, x, y, rc) a step ahead,
// then f(valid, rc, pre, beta, dc, M).
constexpr int FV_STRIPS = 8;
__host__ __device__ inline int walk_groups(int n, int nr)
{
    return 10 * ((n - 1 + FV_STRIPS - 1) / FV_STRIPS) * ((nr - 1 + 63) / 64);
}
template <class F>
__device__ __forceinline__ void walk_columns(const FvArgs& a, const double* __restrict__ columns,
                                             const double* __restrict__ vel, double kappa, F& f)
{
    const int n = a.n, nr = a.nr, nq = n - 1, ncr = nr - 1;
    const int64_t N = 10LL * n * n * nr;
    const int nxg = (nq + FV_STRIPS - 1) / FV_STRIPS, total = walk_groups(n, nr) * nq;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    int pos = march::run_begin(total, tile, gridDim.x);
    const int end = march::run_begin(total, tile + 1, gridDim.x);
    while (pos < end) {
        const int group = pos / nq, y0 = pos - group * nq, y1 = min(nq, y0 + end - pos);
        pos += y1 - y0;
        const int x = (group % nxg) * FV_STRIPS + w, d = (group / nxg) % 10, chunk = group / (nxg * 10);
        if (x >= nq) continue;  // (no barrier in the walk)
        const int rc = 1 + 64 * chunk + (threadIdx.x & 63);
        const bool valid = rc <= ncr;
        const int rcc = valid ? rc : ncr;
        Layer L;
        L.set(a, rcc, kappa);
        // corners (x, .), (x + 1, .) at y, y + 1 and, loaded a step ahead, y + 2 (roles
        // rotate by copies): a step's loads are in flight before the last one's stores
        CornerVel A0, A1, B0, B1, C0, C1;
        typename F::Pre cur, nxt;
        const int64_t row = (int64_t)n * nr;
        int64_t node = (((int64_t)d * n + x) * n + y0) * nr + rcc - 1;
        A0.load(vel, N, node);
        A1.load(vel, N, node + row);
        node += nr;
        B0.load(vel, N, node);
        B1.load(vel, N, node + row);
        f.load(cur, d, x, y0, rcc);
        A0.combine(L);
        A1.combine(L);
        const double* __restrict__ g = columns + (int64_t)FV_COLUMN * __builtin_amdgcn_readfirstlane((d * nq + x) * nq + y0);
        for (int y = y0; y < y1; ++y, g += FV_COLUMN) {
            if (y + 1 < y1) {
                node += nr;
                C0.load(vel, N, node);
                C1.load(vel, N, node + row);
                f.load(nxt, d, x, y + 1, rcc);
            }
            B0.combine(L);
            B1.combine(L);
            double beta[6], dc[6], M;
            cell_faces(g, L, A0, A1, B0, B1, beta, dc, M);
            f(valid, rcc, cur, beta, dc, M);
            A0 = B0;
            A1 = B1;
            B0 = C0;
            B1 = C1;
            cur = nxt;
        }
    }
}

// The same a thread per cell: the column's table and both levels of four corners for
// each.  For the meshes that leave the walk's lanes or its CUs empty (walk_pays); the
// arithmetic, and so the result, is the walk's.
template <class F>
__device__ __forceinline__ void visit_cells(const FvArgs& a, const double* __restrict__ columns,
                                            const double* __restrict__ vel, double kappa, F& f)
{
    const int n = a.n, nr = a.nr, nq = n - 1, ncr = nr - 1;
    const int64_t N = 10LL * n * n * nr, cells = 10LL * nq * nq * ncr;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < cells; t += (int64_t)gridDim.x * blockDim.x) {
        const int q = (int)(t / ncr), rc = 1 + (int)(t - (int64_t)q * ncr);
        const int y = q % nq, x = (q / nq) % nq, d = q / (nq * nq);
        double g[FV_COLUMN];
        const double2* row = reinterpret_cast<const double2*>(columns + (int64_t)FV_COLUMN * q);
#pragma unroll
        for (int k = 0; k < FV_COLUMN / 2; ++k) {
            const double2 v = row[k];
            g[2 * k] = v.x;
            g[2 * k + 1] = v.y;
        }
        CornerVel c00, c10, c01, c11;
        const int64_t node = (((int64_t)d * n + x) * n + y) * nr + rc - 1, step = (int64_t)n * nr;
        c00.load(vel, N, node);
        c10.load(vel, N, node + step);
        c01.load(vel, N, node + nr);
        c11.load(vel, N, node + step + nr);
        typename F::Pre pre;
        f.load(pre, d, x, y, rc);
        Layer L;
        L.set(a, rc, kappa);
        c00.combine(L);
        c10.combine(L);
        c01.combine(L);
        c11.combine(L);
        double beta[6], dc[6], M;
        cell_faces(g, L, c00, c10, c01, c11, beta, dc, M);
        f(true, rc, pre, beta, dc, M);
    }
}

__device__ __forceinline__ int64_t neighbour(int n, int nr, int d, int xc, int yc, int rc, int f)
{
    const int ox = f == 0 ? -1 : (f == 1 ? 1 : 0), oy = f == 2 ? -1 : (f == 3 ? 1 : 0),
              orr = f == 4 ? -1 : (f == 5 ? 1 : 0);
    return fvi(n, nr, d, xc + ox, yc + oy, rc + orr);
}

// ---------------------------------------------------------------- kernels

// Column part c of the cell centres: int_K x / |K| = s c with
// c = sum_w |det_w| (V0 + V1 + V2)_w / 3 / sum_w |det_w| and the layer part
// s = int rho^3 / int rho^2 (the Felippa rule integrates both exactly)
__global__ __launch_bounds__(FV_BLOCK) void k_fv_centroids(FvArgs a, double* __restrict__ centroids)
{
    const int n = a.n;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 10LL * (n - 1) * (n - 1)) return;
    const int y = (int)(t % (n - 1)), x = (int)((t / (n - 1)) % (n - 1)), d = (int)(t / ((int64_t)(n - 1) * (n - 1)));
    double c[4][3], det[2];
    column_corners(a.coords, n, d, x, y, c);
    column_dets(c, det);
    double* o = centroids + 3 * (((int64_t)d * (n + 1) + x + 1) * (n + 1) + y + 1);
#pragma unroll
    for (int j = 0; j < 3; ++j)
        o[j] = (det[0] * (c[0][j] + c[1][j] + c[2][j]) + det[1] * (c[3][j] + c[2][j] + c[1][j])) /
               (3.0 * (det[0] + det[1]));
}

// lateral ghost columns of the centroids
__global__ __launch_bounds__(FV_BLOCK) void k_fv_ghost_columns(const int32_t* __restrict__ pairs, int cnt,
                                                               double* __restrict__ centroids)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= cnt) return;
    for (int j = 0; j < 3; ++j) centroids[3LL * pairs[2 * t] + j] = centroids[3LL * pairs[2 * t + 1] + j];
}

// the table of every hex column (FV_COLUMN), one thread per column
__global__ __launch_bounds__(FV_BLOCK) void k_fv_columns(FvArgs a, const double* __restrict__ centroids,
                                                         double* __restrict__ columns)
{
    const int n = a.n;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 10LL * (n - 1) * (n - 1)) return;
    const int y = (int)(t % (n - 1)), x = (int)((t / (n - 1)) % (n - 1)), d = (int)(t / ((int64_t)(n - 1) * (n - 1)));
    double c[4][3], det[2], g[FV_COLUMN];
    column_corners(a.coords, n, d, x, y, c);
    column_dets(c, det);
    const int64_t fl = ((int64_t)d * (n + 1) + x + 1) * (n + 1) + y + 1;
    const double* ci = centroids + 3 * fl;
    const int FA[4] = {0, 3, 0, 3}, FB[4] = {2, 1, 1, 2};  // corner indices of faces 0, 1, 2, 3
    const int64_t nb[4] = {fl - (n + 1), fl + (n + 1), fl - 1, fl + 1};
#pragma unroll
    for (int f = 0; f < 4; ++f) {
        double N[3], dx[3];
        cross3(c[FB[f]], c[FA[f]], N);
        for (int j = 0; j < 3; ++j) dx[j] = centroids[3 * nb[f] + j] - ci[j];
        const double s = dot3d(N, dx);
        for (int j = 0; j < 3; ++j) g[3 * f + j] = s < 0 ? -N[j] : N[j];
        g[20 + f] = dot3d(N, N) / fabs(s);
    }
    double e1[3], e2[3], nn[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        e1[j] = c[1][j] - c[0][j];
        e2[j] = c[2][j] - c[0][j];
    }
    cross3(e1, e2, g + 12);
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        e1[j] = c[2][j] - c[3][j];
        e2[j] = c[1][j] - c[3][j];
    }
    cross3(e1, e2, g + 15);
    for (int j = 0; j < 3; ++j) nn[j] = g[12 + j] + g[15 + j];
    const double ar = dot3d(nn, ci);
    g[18] = det[0] + det[1];
    g[19] = ar < 0 ? -1.0 : 1.0;
    g[24] = dot3d(nn, nn) / fabs(ar);
    g[25] = 0.0;
    double2* o = reinterpret_cast<double2*>(columns + FV_COLUMN * t);
#pragma unroll
    for (int k = 0; k < FV_COLUMN / 2; ++k) o[k] = make_double2(g[2 * k], g[2 * k + 1]);
}

// cell centre = (int_K x) / |K| with the Felippa rule on both wedges (helpers.hpp:123-175)
__global__ __launch_bounds__(FV_BLOCK) void k_fv_centers(FvArgs a, double* __restrict__ c)
{
    const int n = a.n, nr = a.nr;
    const int64_t cells = 10LL * (n - 1) * (n - 1) * (nr - 1);
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= cells) return;
    int d, xc, yc, rc;
    cell_real(t, n, nr, d, xc, yc, rc);
    double P[2][3][3];
    wedge_corners(a.coords, n, d, xc - 1, yc - 1, P);
    const double r1 = a.radii[rc - 1], r2 = a.radii[rc];
    double vol = 0, I[3] = {0, 0, 0};
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            double xi, eta, zeta;
            qpoint(q, xi, eta, zeta);
            const double Jw = abs_det(P[w], r1, r2, xi, eta, zeta) * QW;
            vol += Jw;
            const double rr = r1 + 0.5 * (r2 - r1) * (1 + zeta);
#pragma unroll
            for (int k = 0; k < 3; ++k)
                I[k] += rr * ((1 - xi - eta) * P[w][0][k] + xi * P[w][1][k] + eta * P[w][2][k]) * Jw;
        }
    double* o = c + 3 * fvi(n, nr, d, xc, yc, rc);
    o[0] = I[0] / vol;
    o[1] = I[1] / vol;
    o[2] = I[2] / vol;
}

// lateral ghost cells <- the neighbouring diamonds' real cells (real radial range)
__global__ __launch_bounds__(FV_BLOCK) void k_fv_ghost(const int32_t* __restrict__ pairs, int cnt, int nr,
                                                       int ncomp, double* __restrict__ f)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)cnt * (nr - 1)) return;
    const int rc = 1 + (int)(t % (nr - 1));
    const int k = (int)(t / (nr - 1));
    const int64_t dst = ((int64_t)pairs[2 * k] * (nr + 1) + rc) * ncomp;
    const int64_t src = ((int64_t)pairs[2 * k + 1] * (nr + 1) + rc) * ncomp;
    for (int c = 0; c < ncomp; ++c) f[dst + c] = f[src + c];
}

// the same for two scalars at once
__global__ __launch_bounds__(FV_BLOCK) void k_fv_ghost2(const int32_t* __restrict__ pairs, int cnt, int nr,
                                                        double* __restrict__ f, double* __restrict__ g)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)cnt * (nr - 1)) return;
    const int rc = 1 + (int)(t % (nr - 1));
    const int k = (int)(t / (nr - 1));
    const int64_t dst = (int64_t)pairs[2 * k] * (nr + 1) + rc, src = (int64_t)pairs[2 * k + 1] * (nr + 1) + rc;
    const double a = f[src], b = g[src];
    f[dst] = a;
    g[dst] = b;
}

// local stable time step M / lambda per cell, minimum per block
// (fct_advection_diffusion.hpp:110-164)
// (geometry as the predictor's: 750 us at lateral level 7 x 129 when every cell
// read its seven centres, 174 us so; both repeated alone, in an energy step 831 and 206)
struct StableStep {
    double dt = 1e300;
    bool diffusion;
    struct Pre {};
    __device__ __forceinline__ void load(Pre&, int, int, int, int) {}
    __device__ __forceinline__ void operator()(bool valid, int, const Pre&, const double beta[6], const double dc[6],
                                               double M)
    {
        double lambda = 0;
#pragma unroll
        for (int f = 0; f < 6; ++f) {
            if (beta[f] < 0) lambda -= beta[f];
            if (diffusion) lambda += dc[f];
        }
        if (valid) dt = fmin(dt, lambda > 0 ? M / lambda : 1e30);
    }
};

// block minimum (order-independent) into part[blockIdx.x]
__device__ __forceinline__ void block_min(double v, double* __restrict__ part)
{
    __shared__ double red[16];
    for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = red[0];
        for (int k = 1; k < (int)(blockDim.x >> 6); ++k) m = fmin(m, red[k]);
        part[blockIdx.x] = m;
    }
}

__global__ __launch_bounds__(64 * FV_STRIPS) __attribute__((amdgpu_waves_per_eu(4, 4)))
void k_fv_dt(FvArgs a, const double* __restrict__ columns, const double* __restrict__ vel, double kappa,
             double* __restrict__ part)
{
    StableStep st;
    st.diffusion = kappa > 0;
    walk_columns(a, columns, vel, kappa, st);
    block_min(st.dt, part);
}

__global__ __launch_bounds__(FV_BLOCK) void k_fv_dt_cells(FvArgs a, const double* __restrict__ columns,
                                                          const double* __restrict__ vel, double kappa,
                                                          double* __restrict__ part)
{
    StableStep st;
    st.diffusion = kappa > 0;
    visit_cells(a, columns, vel, kappa, st);
    block_min(st.dt, part);
}

__global__ __launch_bounds__(256) void k_min_finalize(const double* __restrict__ part, int nblk,
                                                      double* __restrict__ out)
{
    double m = 1e300;
    for (int b = threadIdx.x; b < nblk; b += blockDim.x) m = fmin(m, part[b]);
    for (int o = 32; o > 0; o >>= 1) m = fmin(m, __shfl_xor(m, o));
    __shared__ double red[4];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) out[0] = fmin(fmin(red[0], red[1]), fmin(red[2], red[3]));
}

// predictor (fct_advection_diffusion.hpp:261-402): low-order upwind +
// two-point diffusion T_L, and the pre-scaled antidiffusive fluxes
// (dt / M) (|beta| / 2) (T_i - T_j), stored face-major [6][fv cells].
// What binds is memory: velocity and T in, T_L and six fluxes out (88 B a cell,
// 104 with the flux sums).  A thread per cell that read the centres of its cell
// and six neighbours and both levels of four corners took 962 us at lateral level
// 7 x 129; the column / layer split of the geometry needs no centres, and a run of
// columns loads two corners a step: 646 us as a stage of its own, 715 us in the step,
// where the flux sums are written too (731 in the energy case, behind other work).
struct Predict {
    const double* __restrict__ T;
    const double* __restrict__ source;
    double* __restrict__ TL;
    double* __restrict__ ad;
    double dt;
    int subtract_div, n, nr;
    int64_t fvsize;
    FctFused fu;
    struct Pre {
        int64_t i;
        double Ti, Tj[6], src;
    };
    __device__ __forceinline__ void load(Pre& q, int d, int x, int y, int rcc)
    {
        q.i = fvi(n, nr, d, x + 1, y + 1, rcc);
        q.Ti = T[q.i];
#pragma unroll
        for (int f = 0; f < 6; ++f) q.Tj[f] = T[neighbour(n, nr, d, x + 1, y + 1, rcc, f)];
        q.src = source ? source[q.i] : 0.0;
    }
    __device__ __forceinline__ void operator()(bool valid, int rcc, const Pre& q, const double beta[6],
                                               const double dc[6], double M)
    {
        const int64_t i = q.i;
        const double Ti = q.Ti;
        const double(&Tj)[6] = q.Tj;
        const double sc = dt / M;
        double lo_diag = 0, lo_update = 0, bsum = 0, pp = 0, pm = 0;
        double fl[6];
#pragma unroll
        for (int f = 0; f < 6; ++f) {
            if (beta[f] >= 0)
                lo_diag += beta[f];
            else
                lo_update += beta[f] * Tj[f];
            bsum += beta[f];
            lo_diag += dc[f];
            lo_update -= dc[f] * Tj[f];
            fl[f] = sc * (fabs(beta[f]) / 2.0) * (Ti - Tj[f]);
            if (fl[f] > 0)
                pp += fl[f];
            else
                pm += fl[f];
        }
        if (subtract_div) lo_diag -= bsum;
        double v = Ti - sc * (lo_diag * Ti + lo_update);
        if (source) v += dt * q.src;
        if (!valid) return;
#pragma unroll
        for (int f = 0; f < 6; ++f) ad[f * fvsize + i] = fl[f];
        if (fu.pp) {
            fu.pp[i] = pp;
            fu.pm[i] = pm;
        }
        if (rcc == 1 && fu.apply_cmb) {
            v = fu.t_cmb;
            TL[i - 1] = v;
        }
        if (rcc == nr - 1 && fu.apply_surf) {
            v = fu.t_surf;
            TL[i + 1] = v;
        }
        TL[i] = v;
    }
};

__global__ __launch_bounds__(64 * FV_STRIPS) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_fct_predictor(FvArgs a, const double* __restrict__ columns, const double* __restrict__ vel, const double* __restrict__ T,
        double dt, double kappa, const double* __restrict__ source, int subtract_div, double* __restrict__ TL,
        double* __restrict__ ad, int64_t fvsize, FctFused fu)
{
    Predict p{T, source, TL, ad, dt, subtract_div, a.n, a.nr, fvsize, fu};
    walk_columns(a, columns, vel, kappa, p);
}

__global__ __launch_bounds__(FV_BLOCK)
void k_fct_predictor_cells(FvArgs a, const double* __restrict__ columns, const double* __restrict__ vel, const double* __restrict__ T,
        double dt, double kappa, const double* __restrict__ source, int subtract_div, double* __restrict__ TL,
        double* __restrict__ ad, int64_t fvsize, FctFused fu)
{
    Predict p{T, source, TL, ad, dt, subtract_div, a.n, a.nr, fvsize, fu};
    visit_cells(a, columns, vel, kappa, p);
}

// Dirichlet values on the shells: the real boundary cell and the ghost beyond (helpers.hpp:64-96)
__global__ __launch_bounds__(FV_BLOCK) void k_fv_dirichlet(int n, int nr, double* __restrict__ f, int apply_cmb,
                                                           double t_cmb, int apply_surf, double t_surf)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 10LL * (n - 1) * (n - 1)) return;
    const int yc = 1 + (int)(t % (n - 1));
    const int xc = 1 + (int)((t / (n - 1)) % (n - 1));
    const int d = (int)(t / ((int64_t)(n - 1) * (n - 1)));
    if (apply_cmb) {
        f[fvi(n, nr, d, xc, yc, 1)] = t_cmb;
        f[fvi(n, nr, d, xc, yc, 0)] = t_cmb;
    }
    if (apply_surf) {
        f[fvi(n, nr, d, xc, yc, nr - 1)] = t_surf;
        f[fvi(n, nr, d, xc, yc, nr)] = t_surf;
    }
}

// limiter (fct_advection_diffusion.hpp:485-537): Zalesak R+ / R-
__global__ __launch_bounds__(FV_BLOCK) void k_fct_limiter(int n, int nr, const double* __restrict__ TL,
                                                          const double* __restrict__ ad, int64_t fvsize,
                                                          double* __restrict__ Rp, double* __restrict__ Rm)
{
    const int64_t cells = 10LL * (n - 1) * (n - 1) * (nr - 1);
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= cells) return;
    int d, xc, yc, rc;
    cell_real(t, n, nr, d, xc, yc, rc);
    const int64_t i = fvi(n, nr, d, xc, yc, rc);
    const double ti = TL[i];
    double pp = 0, pm = 0, tmax = ti, tmin = ti;
#pragma unroll
    for (int f = 0; f < 6; ++f) {
        const double fij = ad[f * fvsize + i];
        if (fij > 0)
            pp += fij;
        else
            pm += fij;
        const double tj = TL[neighbour(n, nr, d, xc, yc, rc, f)];
        tmax = fmax(tmax, tj);
        tmin = fmin(tmin, tj);
    }
    Rp[i] = pp > 0 ? fmin(1.0, (tmax - ti) / pp) : 1.0;
    Rm[i] = pm < 0 ? fmin(1.0, (tmin - ti) / pm) : 1.0;
}

// limiter from the predictor's flux sums in Rp / Rm (each thread replaces its own):
// 40 instead of 72 B a cell
__global__ __launch_bounds__(FV_BLOCK) void k_fct_limiter_sums(int n, int nr, const double* __restrict__ TL,
                                                               double* __restrict__ Rp, double* __restrict__ Rm)
{
    const int64_t cells = 10LL * (n - 1) * (n - 1) * (nr - 1);
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= cells) return;
    int d, xc, yc, rc;
    cell_real(t, n, nr, d, xc, yc, rc);
    const int64_t i = fvi(n, nr, d, xc, yc, rc);
    const double pp = Rp[i], pm = Rm[i];
    const double ti = TL[i];
    double tmax = ti, tmin = ti;
#pragma unroll
    for (int f = 0; f < 6; ++f) {
        const double tj = TL[neighbour(n, nr, d, xc, yc, rc, f)];
        tmax = fmax(tmax, tj);
        tmin = fmin(tmin, tj);
    }
    Rp[i] = pp > 0 ? fmin(1.0, (tmax - ti) / pp) : 1.0;
    Rm[i] = pm < 0 ? fmin(1.0, (tmin - ti) / pm) : 1.0;
}

// correction (fct_advection_diffusion.hpp:604-658): T = T_L + sum_j alpha_ij f_ij
__global__ __launch_bounds__(FV_BLOCK) void k_fct_correction(int n, int nr, const double* __restrict__ TL,
                                                             const double* __restrict__ ad, int64_t fvsize,
                                                             const double* __restrict__ Rp,
                                                             const double* __restrict__ Rm, double* __restrict__ T)
{
    const int64_t cells = 10LL * (n - 1) * (n - 1) * (nr - 1);
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= cells) return;
    int d, xc, yc, rc;
    cell_real(t, n, nr, d, xc, yc, rc);
    const int64_t i = fvi(n, nr, d, xc, yc, rc);
    const double rpi = Rp[i], rmi = Rm[i];
    double corr = 0;
#pragma unroll
    for (int f = 0; f < 6; ++f) {
        const int64_t j = neighbour(n, nr, d, xc, yc, rc, f);
        const double fij = ad[f * fvsize + i];
        const double al = fij > 0 ? fmin(rpi, Rm[j]) : fmin(rmi, Rp[j]);
        corr += al * fij;
    }
    T[i] = TL[i] + corr;
}

// right-hand side of the FV -> FE L2 projection (conversion.hpp:151-200):
// b_i = sum over the cells K around node i of T_K int_K phi_i, gathered per
// node copy (no atomics); the interface sum follows.  The reference evaluates
// int_K phi_i |det J| with the Felippa 3x2 rule, which is exact: per wedge
//   |det(V0, V1, V2)| / 6 x (I_bot or I_top),  I = int rho^2 x radial hat drho,
//   I_bot = dr (r1^2/2 + r1 dr/3 + dr^2/12),  I_top = dr (r1^2/2 + 2 r1 dr/3 + dr^2/4)
// Tfv null: every T_K = 1, which gives the lumped diagonal D_i = int phi_i.
__global__ __launch_bounds__(FV_BLOCK) void k_fv_to_fe_rhs(FvArgs a, const double* __restrict__ Tfv,
                                                           double* __restrict__ b)
{
    const int n = a.n, nr = a.nr;
    const int64_t N = 10LL * n * n * nr;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= N) return;
    const int r = (int)(t % nr);
    const int y = (int)((t / nr) % n);
    const int x = (int)((t / ((int64_t)nr * n)) % n);
    const int d = (int)(t / ((int64_t)nr * n * n));
    double acc = 0;
    for (int cx = x - 1; cx <= x; ++cx) {
        if (cx < 0 || cx > n - 2) continue;
        for (int cy = y - 1; cy <= y; ++cy) {
            if (cy < 0 || cy > n - 2) continue;
            double P[2][3][3];
            wedge_corners(a.coords, n, d, cx, cy, P);
            double det[2];
#pragma unroll
            for (int w = 0; w < 2; ++w) {
                double v12[3];
                cross3(P[w][1], P[w][2], v12);
                det[w] = fabs(P[w][0][0] * v12[0] + P[w][0][1] * v12[1] + P[w][0][2] * v12[2]) / 6.0;
            }
            // the node's weight in this quad: the wedges that contain its lateral corner
            const int lx = x - cx, ly = y - cy;
            const double wlat = (lx == 0 && ly == 0) ? det[0] : ((lx == 1 && ly == 1) ? det[1] : det[0] + det[1]);
            for (int cr = r - 1; cr <= r; ++cr) {
                if (cr < 0 || cr > nr - 2) continue;
                const double r1 = a.radii[cr], dr = a.radii[cr + 1] - r1;
                const double irad = (r == cr + 1) ? dr * (0.5 * r1 * r1 + r1 * dr * (2.0 / 3.0) + 0.25 * dr * dr)
                                                  : dr * (0.5 * r1 * r1 + r1 * dr / 3.0 + dr * dr / 12.0);
                acc += wlat * irad * (Tfv ? Tfv[fvi(n, nr, d, cx + 1, cy + 1, cr + 1)] : 1.0);
            }
        }
    }
    b[t] = acc;
}

// u_i = b_i (1 / D_i): the lumped FV -> FE transfer's last step
// (conversion.hpp:337-340, invert_entries then scale_in_place)
__global__ __launch_bounds__(FV_BLOCK) void k_fv_lumped_scale(const double* __restrict__ D, double* __restrict__ u,
                                                             int64_t N)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < N) u[t] = u[t] * (1.0 / D[t]);
}

// FE -> FV cell averages (conversion.hpp:348-416): T_K = int_K u_h / |K| with
// the Felippa 3x2 rule on both wedges; wedge shape i = lateral hat (1 - xi -
// eta, xi, eta)[i % 3] x radial hat ((1 - zeta) / 2 for i < 3, else (1 + zeta) / 2)
__global__ __launch_bounds__(FV_BLOCK) void k_fe_to_fv(FvArgs a, const double* __restrict__ u,
                                                       double* __restrict__ Tfv)
{
    const int n = a.n, nr = a.nr;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 10LL * (n - 1) * (n - 1) * (nr - 1)) return;
    int d, xc, yc, rc;
    cell_real(t, n, nr, d, xc, yc, rc);
    const int x = xc - 1, y = yc - 1, r = rc - 1;
    double P[2][3][3];
    wedge_corners(a.coords, n, d, x, y, P);
    const double r1 = a.radii[r], r2 = a.radii[r + 1];
    double vol = 0, integral = 0;
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        double lu[6];
#pragma unroll
        for (int i = 0; i < 6; ++i)
            lu[i] = u[(((int64_t)d * n + x + FV_WOFF[w][i][0]) * n + y + FV_WOFF[w][i][1]) * nr + r + FV_WOFF[w][i][2]];
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            double xi, eta, zeta;
            qpoint(q, xi, eta, zeta);
            const double Jw = abs_det(P[w], r1, r2, xi, eta, zeta) * QW;
            vol += Jw;
            const double lat[3] = {1 - xi - eta, xi, eta};
            const double bot = 0.5 * (1 - zeta), top = 0.5 * (1 + zeta);
            double uq = 0;
#pragma unroll
            for (int i = 0; i < 6; ++i) uq += lu[i] * lat[i % 3] * (i < 3 ? bot : top);
            integral += uq * Jw;
        }
    }
    Tfv[fvi(n, nr, d, xc, yc, rc)] = integral / vol;
}

int blocks_for(int64_t work) { return (int)((work + FV_BLOCK - 1) / FV_BLOCK); }

}  // namespace

int64_t fv_real_cells(int n, int nr) { return 10LL * (n - 1) * (n - 1) * (nr - 1); }
int64_t fv_size(int n, int nr) { return 10LL * (n + 1) * (n + 1) * (nr + 1); }
// Blocks of the column walk: `per_cu` on every CU (what its registers allow), one
// column each on small meshes
static int walk_blocks(int n, int nr, int per_cu)
{
    return std::max(1, std::min(walk_groups(n, nr) * (n - 1), device_cus() * per_cu));
}
// Whether the column walk beats the form by cells: a chunk's lanes filled with `fill`
// layers or more on average, and four columns or more for each CU's first block (on
// fewer the walk has no columns to keep corners for).  Both forms measured at levels 3
// to 7 with 3 to 200 radial nodes.  The stable step reads little and breaks even at 24
// layers (level 7: 8 layers 104 us walked, 58 by cells; 24: 106, 108; 64: 120, 259), the
// predictor at 40 (8 layers 162, 50; 32: 252, 233; 40: 269, 287; 2 x 34.5: 491, 475; 64:
// 334, 445).  At level 4 the forms are within 4 us of each other.
constexpr int WALK_FILL_DT = 24, WALK_FILL_PREDICTOR = 40;
static bool walk_pays(int n, int nr, int fill)
{
    const int chunks = (nr - 1 + 63) / 64;
    return nr - 1 >= fill * chunks && walk_groups(n, nr) * (n - 1) >= 4 * device_cus();
}
// at most FV_DT_BLOCKS partial minima of the form by cells
constexpr int FV_DT_BLOCKS = 2048;
int fv_dt_blocks(int n, int nr)
{
    return walk_pays(n, nr, WALK_FILL_DT) ? walk_blocks(n, nr, 2) : std::min(blocks_for(fv_real_cells(n, nr)), FV_DT_BLOCKS);
}

void launch_fv_centers(const FvArgs& a, double* c, hipStream_t s)
{
    hipLaunchKernelGGL(k_fv_centers, dim3(blocks_for(fv_real_cells(a.n, a.nr))), dim3(FV_BLOCK), 0, s, a, c);
}

void launch_fv_centroids(const FvArgs& a, double* centroids, hipStream_t s)
{
    hipLaunchKernelGGL(k_fv_centroids, dim3(blocks_for(10LL * (a.n - 1) * (a.n - 1))), dim3(FV_BLOCK), 0, s, a,
                       centroids);
}

void launch_fv_ghost_columns(const int32_t* pairs, int cnt, double* centroids, hipStream_t s)
{
    if (cnt == 0) return;
    hipLaunchKernelGGL(k_fv_ghost_columns, dim3(blocks_for(cnt)), dim3(FV_BLOCK), 0, s, pairs, cnt, centroids);
}

void launch_fv_columns(const FvArgs& a, const double* centroids, double* columns, hipStream_t s)
{
    hipLaunchKernelGGL(k_fv_columns, dim3(blocks_for(10LL * (a.n - 1) * (a.n - 1))), dim3(FV_BLOCK), 0, s, a,
                       centroids, columns);
}

void launch_fv_ghost(const int32_t* pairs, int cnt, int nr, int ncomp, double* f, hipStream_t s)
{
    if (cnt == 0) return;
    hipLaunchKernelGGL(k_fv_ghost, dim3(blocks_for((int64_t)cnt * (nr - 1))), dim3(FV_BLOCK), 0, s, pairs, cnt, nr,
                       ncomp, f);
}

void launch_fv_ghost2(const int32_t* pairs, int cnt, int nr, double* f, double* g, hipStream_t s)
{
    if (cnt == 0) return;
    hipLaunchKernelGGL(k_fv_ghost2, dim3(blocks_for((int64_t)cnt * (nr - 1))), dim3(FV_BLOCK), 0, s, pairs, cnt, nr, f,
                       g);
}

void launch_fv_dt(const FvArgs& a, const double* vel, double kappa, double* part, double* out, hipStream_t s)
{
    const int nb = fv_dt_blocks(a.n, a.nr);
    if (walk_pays(a.n, a.nr, WALK_FILL_DT))
        hipLaunchKernelGGL(k_fv_dt, dim3(nb), dim3(64 * FV_STRIPS), 0, s, a, a.columns, vel, kappa, part);
    else
        hipLaunchKernelGGL(k_fv_dt_cells, dim3(nb), dim3(FV_BLOCK), 0, s, a, a.columns, vel, kappa, part);
    hipLaunchKernelGGL(k_min_finalize, dim3(1), dim3(256), 0, s, part, nb, out);
}

void launch_fct_predictor(const FvArgs& a, const double* vel, const double* T, double dt, double kappa,
                          const double* source, int subtract_div, double* TL, double* ad, const FctFused& fused,
                          hipStream_t s)
{
    if (walk_pays(a.n, a.nr, WALK_FILL_PREDICTOR))
        hipLaunchKernelGGL(k_fct_predictor, dim3(walk_blocks(a.n, a.nr, 1)), dim3(64 * FV_STRIPS), 0, s, a, a.columns, vel,
                           T, dt, kappa, source, subtract_div, TL, ad, fv_size(a.n, a.nr), fused);
    else
        hipLaunchKernelGGL(k_fct_predictor_cells, dim3(blocks_for(fv_real_cells(a.n, a.nr))), dim3(FV_BLOCK), 0, s, a,
                           a.columns, vel, T, dt, kappa, source, subtract_div, TL, ad, fv_size(a.n, a.nr), fused);
}

void launch_fv_dirichlet(int n, int nr, double* f, int apply_cmb, double t_cmb, int apply_surf, double t_surf,
                         hipStream_t s)
{
    hipLaunchKernelGGL(k_fv_dirichlet, dim3(blocks_for(10LL * (n - 1) * (n - 1))), dim3(FV_BLOCK), 0, s, n, nr, f,
                       apply_cmb, t_cmb, apply_surf, t_surf);
}

void launch_fct_limiter(int n, int nr, const double* TL, const double* ad, double* Rp, double* Rm, hipStream_t s)
{
    hipLaunchKernelGGL(k_fct_limiter, dim3(blocks_for(fv_real_cells(n, nr))), dim3(FV_BLOCK), 0, s, n, nr, TL, ad,
                       fv_size(n, nr), Rp, Rm);
}

void launch_fct_limiter_sums(int n, int nr, const double* TL, double* Rp, double* Rm, hipStream_t s)
{
    hipLaunchKernelGGL(k_fct_limiter_sums, dim3(blocks_for(fv_real_cells(n, nr))), dim3(FV_BLOCK), 0, s, n, nr, TL, Rp,
                       Rm);
}

void launch_fct_correction(int n, int nr, const double* TL, const double* ad, const double* Rp, const double* Rm,
                           double* T, hipStream_t s)
{
    hipLaunchKernelGGL(k_fct_correction, dim3(blocks_for(fv_real_cells(n, nr))), dim3(FV_BLOCK), 0, s, n, nr, TL, ad,
                       fv_size(n, nr), Rp, Rm, T);
}

void launch_fv_lumped_scale(const double* D, double* u, int64_t N, hipStream_t s)
{
    hipLaunchKernelGGL(k_fv_lumped_scale, dim3(blocks_for(N)), dim3(FV_BLOCK), 0, s, D, u, N);
}

void launch_fe_to_fv(const FvArgs& a, const double* u, double* Tfv, hipStream_t s)
{
    hipLaunchKernelGGL(k_fe_to_fv, dim3(blocks_for(fv_real_cells(a.n, a.nr))), dim3(FV_BLOCK), 0, s, a, u, Tfv);
}

void launch_fv_to_fe_rhs(const FvArgs& a, const double* Tfv, double* b, hipStream_t s)
{
    hipLaunchKernelGGL(k_fv_to_fe_rhs, dim3(blocks_for(10LL * a.n * a.n * a.nr)), dim3(FV_BLOCK), 0, s, a, Tfv, b);
}

}  // namespace tn
