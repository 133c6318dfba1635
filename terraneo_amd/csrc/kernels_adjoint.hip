// Adjoint viscosity gradient of the epsilon-div-div operator, CDNA4.
//
// With a per-hex-cell viscosity eta_c = exp(m_c) the viscous block is
// A(m) = sum_c eta_c A_c(1), A_c(1) the cell's two wedge matrices at unit
// viscosity.  For a misfit J(u(m)) and the adjoint state lam of the Stokes
// system (K lam = dJ/du, K symmetric),
//   dJ/dm_c = -lam_c^T (dK/dm_c) u_c = -eta_c (T lam)_c^T A_c(1) u_c,
// T the trial rule of the boundary shells (Dirichlet: zero, free-slip: project
// onto the tangent plane); u is the converged solution itself (its Dirichlet
// values are the boundary data, its free-slip normal component vanishes), so
// the boundary diagonal and normal terms of K drop out.  There is no
// counterpart in the reference.
//
// Per wedge the dot product needs no corner vectors: with the corner sums U1, U2, D of
// u and their counterparts V1, V2, E of lam it is p1 . V1 + p2 . V2 + q . E.
//
// A wave marches along runs of quads, its lanes the layers: P = 64 / layers runs side
// by side where the layers leave lanes over (at most six), else one run and a chunk
// of 64 layers.  A step takes over two lateral corners from the step before and loads
// the other two, the quad's wedge table (20 numbers per run, spread through LDS) and
// the viscosity one step ahead.  Bound by the latency of a step and its loads:
// 10 x 64 x 64 quads of 64 layers, FP64, free-slip 92 us as a thread per cell (eight
// corners and the table loaded by each, 64-bit divisions), 54 so (3.2 TB/s of the
// fields once).
#include <algorithm>

#include "tn_cell.hpp"
#include "tn_eps_march.hpp"
#include "tn_march.hpp"
#include "tn_objects.hpp"

namespace tn {
namespace {

using namespace cellops;

constexpr int ADJ_RUNS = 6;  // runs side by side, at most

// a node column at the lane's layer: sums and differences over its two levels
template <typename T>
struct AdjCorner {
    T S[3], D[3], V[3], E[3];  // of u, of lam (trial rule applied)
};

template <typename T>
struct AdjWalk {
    const T* u;
    const T* lam;
    const T* coords;
    int64_t N;
    int nr, rc;
    int bmode, tmode;
    bool slip;  // (uniform: a shell is free-slip)

    struct Raw {
        T ub[3], ut[3], lb[3], lt[3], n[3];
    };
    __device__ __forceinline__ void load(int lat, Raw& o) const
    {
        const int64_t ib = (int64_t)lat * nr + rc;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            o.ub[j] = u[j * N + ib];
            o.ut[j] = u[j * N + ib + 1];
            o.lb[j] = lam[j * N + ib];
            o.lt[j] = lam[j * N + ib + 1];
            o.n[j] = slip ? coords[3 * (int64_t)lat + j] : T(0);
        }
    }
    static __device__ __forceinline__ void trial(T (&v)[3], int mode, const T (&n)[3])
    {
        const T un = mode == TN_FREESLIP ? n[0] * v[0] + n[1] * v[1] + n[2] * v[2] : T(0);
#pragma unroll
        for (int j = 0; j < 3; ++j) v[j] = mode == TN_DIRICHLET ? T(0) : v[j] - un * n[j];
    }
    __device__ __forceinline__ void corner(Raw& o, AdjCorner<T>& c) const
    {
        trial(o.lb, bmode, o.n);
        trial(o.lt, tmode, o.n);
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            c.S[j] = o.ub[j] + o.ut[j];
            c.D[j] = o.ut[j] - o.ub[j];
            c.V[j] = o.lb[j] + o.lt[j];
            c.E[j] = o.lt[j] - o.lb[j];
        }
    }
};

// wedge with corners c0, c1, c2 and the shared difference sums of corners 1 and 2
template <typename T>
__device__ __forceinline__ T adj_wedge(const AdjCorner<T>& c0, const AdjCorner<T>& c1, const AdjCorner<T>& c2,
                                       const T d12[3], const T e12[3], const T* g, T alpha, T beta, T kr)
{
    T U1[3], U2[3], D[3], p1[3], p2[3], q[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        U1[k] = c1.S[k] - c0.S[k];
        U2[k] = c2.S[k] - c0.S[k];
        D[k] = c0.D[k] + d12[k];
    }
    wedge_products_g(U1, U2, D, T(6) * (kr * g[9]), g, alpha, beta, p1, p2, q);  // 6: unit viscosity at six nodes
    T acc = 0;
#pragma unroll
    for (int k = 0; k < 3; ++k)
        acc += p1[k] * (c1.V[k] - c0.V[k]) + p2[k] * (c2.V[k] - c0.V[k]) + q[k] * (c0.E[k] + e12[k]);
    return acc;
}

template <typename T>
__global__ __launch_bounds__(256) void k_grad_log_cell_eta(Geom<T> g, const T* __restrict__ eta_cell,
                                                           const T* __restrict__ u, const T* __restrict__ lam,
                                                           int bc_cmb, int bc_surf, T* __restrict__ grad, int P,
                                                           int chunks, int runs)
{
    constexpr int G = 2 * GEO_STRIDE;
    __shared__ T table[4][ADJ_RUNS * G];
    const int ncr = g.nr - 1, ncl = g.n - 1, quads = 10 * ncl * ncl;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int w = __builtin_amdgcn_readfirstlane(xcd_tile(blockIdx.x, gridDim.x) * 4 + wave);
    const int group = w / chunks, chunk = w % chunks;  // P runs, a chunk of the layers
    if (group * P >= runs) return;                     // (no block barrier follows)
    const int sub = P > 1 ? min(lane / ncr, P - 1) : 0;
    const int layer = P > 1 ? lane - sub * ncr : 64 * chunk + lane;
    const int run = group * P + sub;
    int pos = march::run_begin(quads, min(run, runs), runs);
    const int length = run < runs ? march::run_begin(quads, run + 1, runs) - pos : 0;
    const bool valid = layer < ncr;
    const int rc = valid ? layer : ncr - 1;
    AdjWalk<T> A{u, lam, g.coords, 10LL * g.n * g.n * g.nr, g.nr, rc, rc == 0 ? bc_cmb : (int)TN_NEUMANN,
                 rc == ncr - 1 ? bc_surf : (int)TN_NEUMANN, bc_cmb == TN_FREESLIP || bc_surf == TN_FREESLIP};
    const T r0 = g.radii[rc], r1 = g.radii[rc + 1];
    const T half_dr = T(0.5) * (r1 - r0), r_mid = T(0.5) * (r0 + r1);
    const T alpha = T(1) / r_mid, beta = T(1) / half_dr, kr = r_mid * r_mid * half_dr * T(1.0 / 6.0);
    // table entries this lane fetches: entry e of run e / G
    int gpos[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int r = min(group * P + min((lane + 64 * k) / G, P - 1), runs - 1);
        gpos[k] = march::run_begin(quads, r, runs);
    }
    const int steps = (quads + runs - 1) / runs;  // the longest run
    pos = min(pos, quads - 1);
    int y = pos % ncl, lat = ((pos / ncl / ncl) * g.n + (pos / ncl) % ncl) * g.n + y;
    auto geo = [&](int k, int step) {
        return g.geo[(int64_t)min(gpos[k] + step, quads - 1) * G + (lane + 64 * k) % G];
    };
    typename AdjWalk<T>::Raw na, nb;
    AdjCorner<T> c[4];
    T ng[2] = {geo(0, 0), P > 3 ? geo(1, 0) : T(0)};
    T ne = eta_cell[(int64_t)pos * ncr + rc];
    A.load(lat, na);
    A.load(lat + g.n, nb);
    A.corner(na, c[0]);
    A.corner(nb, c[1]);
    A.load(lat + 1, na);
    A.load(lat + g.n + 1, nb);
#pragma unroll 1
    for (int step = 0; step < steps; ++step) {
        __builtin_amdgcn_wave_barrier();
        if (lane < P * G) table[wave][lane] = ng[0];
        if (P > 3 && lane + 64 < P * G) table[wave][lane + 64] = ng[1];
        __builtin_amdgcn_wave_barrier();
        A.corner(na, c[2]);
        A.corner(nb, c[3]);
        const T e = ne;
        const int here = pos;
        // the next quad: along the strip, or the first of the next strip
        pos = min(pos + 1, quads - 1);
        int next = lat + 1;
        const bool wrap = y + 1 == ncl;
        if (wrap) {
            y = 0;
            next = ((pos / ncl / ncl) * g.n + (pos / ncl) % ncl) * g.n;
        } else {
            ++y;
        }
        ng[0] = geo(0, step + 1);
        if (P > 3) ng[1] = geo(1, step + 1);
        ne = eta_cell[(int64_t)pos * ncr + rc];
        A.load(next + 1, na);
        A.load(next + g.n + 1, nb);
        T d12[3], e12[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            d12[k] = c[1].D[k] + c[2].D[k];
            e12[k] = c[1].E[k] + c[2].E[k];
        }
        const T* t = table[wave] + sub * G;
        const T acc = adj_wedge(c[0], c[1], c[2], d12, e12, t, alpha, beta, kr) +
                      adj_wedge(c[3], c[2], c[1], d12, e12, t + GEO_STRIDE, alpha, beta, kr);
        if (valid && step < length) grad[(int64_t)here * ncr + rc] = -e * acc;
        c[0] = c[2];
        c[1] = c[3];
        if (wrap) {
            typename AdjWalk<T>::Raw fa, fb;
            A.load(next, fa);
            A.load(next + g.n, fb);
            A.corner(fa, c[0]);
            A.corner(fb, c[1]);
        }
        lat = next;
    }
}

// The same a thread per cell, with the march's arithmetic.
template <typename T>
__global__ __launch_bounds__(256) void k_grad_cells(Geom<T> g, const T* __restrict__ eta_cell, const T* __restrict__ u,
                                                    const T* __restrict__ lam, int bc_cmb, int bc_surf,
                                                    T* __restrict__ grad, int64_t cells)
{
    constexpr int G = 2 * GEO_STRIDE;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= cells) return;
    const int ncr = g.nr - 1, ncl = g.n - 1;
    const int q = (int)(t / ncr), rc = (int)(t - (int64_t)q * ncr);
    const int lat = ((q / ncl / ncl) * g.n + (q / ncl) % ncl) * g.n + q % ncl;
    AdjWalk<T> A{u, lam, g.coords, 10LL * g.n * g.n * g.nr, g.nr, rc, rc == 0 ? bc_cmb : (int)TN_NEUMANN,
                 rc == ncr - 1 ? bc_surf : (int)TN_NEUMANN, bc_cmb == TN_FREESLIP || bc_surf == TN_FREESLIP};
    typename AdjWalk<T>::Raw raw[4];
    A.load(lat, raw[0]);
    A.load(lat + g.n, raw[1]);
    A.load(lat + 1, raw[2]);
    A.load(lat + g.n + 1, raw[3]);
    T table[G];
#pragma unroll
    for (int k = 0; k < G; ++k) table[k] = g.geo[(int64_t)q * G + k];
    const T e = eta_cell[t];
    const T r0 = g.radii[rc], r1 = g.radii[rc + 1];
    const T half_dr = T(0.5) * (r1 - r0), r_mid = T(0.5) * (r0 + r1);
    const T alpha = T(1) / r_mid, beta = T(1) / half_dr, kr = r_mid * r_mid * half_dr * T(1.0 / 6.0);
    AdjCorner<T> c[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) A.corner(raw[k], c[k]);
    T d12[3], e12[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        d12[k] = c[1].D[k] + c[2].D[k];
        e12[k] = c[1].E[k] + c[2].E[k];
    }
    const T acc = adj_wedge(c[0], c[1], c[2], d12, e12, table, alpha, beta, kr) +
                  adj_wedge(c[3], c[2], c[1], d12, e12, table + GEO_STRIDE, alpha, beta, kr);
    grad[t] = -e * acc;
}

}  // namespace

template <typename T>
void launch_grad_log_cell_eta(const Geom<T>& g, const T* eta_cell, const T* u, const T* lam, int bc_cmb, int bc_surf,
                              T* grad, hipStream_t s)
{
    const int ncr = g.nr - 1, ncl = g.n - 1;
    const int64_t quads = 10LL * ncl * ncl;
    TN_REQUIRE(10LL * g.n * g.n < (1LL << 31), "gradient: mesh too large");
    const int P = ncr > 32 ? 1 : std::min(ADJ_RUNS, 64 / ncr), chunks = ncr > 32 ? (ncr + 63) / 64 : 1;
    // The march pays where a wave's lanes hold 40 layers or more on average and every lane
    // of one round of resident waves gets four cells; else a thread per cell, as fast or
    // faster than on all smaller or emptier meshes measured (levels 3 to 7, 3 to 200 radial
    // nodes).  FP64, free-slip, us by march and by cells: level 7 x 3 nodes 38 and 14, x 9
    // 43 and 43, x 17 59 and 80, x 70 355 and 352; level 6 x 9 18 and 12, x 33 27 and 39;
    // level 5 x 17 10.4 and 8.1, x 65 16 and 20.
    const int waves_simd = sizeof(T) == 8 ? 2 : 3;
    const int64_t cells = quads * ncr;
    if ((P > 1 ? P * ncr : ncr / chunks) < 40 || cells < 4LL * 64 * 4 * device_cus() * waves_simd) {
        hipLaunchKernelGGL(k_grad_cells<T>, dim3((unsigned)((cells + 255) / 256)), dim3(256), 0, s, g, eta_cell, u, lam,
                           bc_cmb, bc_surf, grad, cells);
        TN_HIP(hipGetLastError());
        return;
    }
    // Equal runs for one round of resident waves (two per SIMD in FP64, three in FP32), or
    // for further rounds so that no run is longer than 40 quads (10 x 128 x 128 quads of 99
    // layers, FP64: 461 us in one round, 417 in four).  Four runs side by side and more:
    // two rounds' worth (10 x 128 x 128 of 8 layers: 60 us in one, 47 in two, 57 in four; a
    // thread per cell took 54).
    const int64_t waves = std::max<int64_t>(1, 4LL * device_cus() * (P > 3 ? 4 : waves_simd) / chunks);
    const int64_t rounds = (quads + waves * P * 40 - 1) / (waves * P * 40);
    const int64_t runs = std::min<int64_t>(quads, waves * P * rounds);
    const int64_t groups = (runs + P - 1) / P;
    hipLaunchKernelGGL(k_grad_log_cell_eta<T>, dim3((unsigned)((groups * chunks + 3) / 4)), dim3(256), 0, s, g, eta_cell,
                       u, lam, bc_cmb, bc_surf, grad, P, chunks, (int)runs);
    TN_HIP(hipGetLastError());
}

template void launch_grad_log_cell_eta<double>(const Geom<double>&, const double*, const double*, const double*, int,
                                               int, double*, hipStream_t);
template void launch_grad_log_cell_eta<float>(const Geom<float>&, const float*, const float*, const float*, int, int,
                                              float*, hipStream_t);

}  // namespace tn
