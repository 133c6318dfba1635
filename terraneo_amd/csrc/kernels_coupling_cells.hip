// B and B^T by fine cells, for the solves: every cell forms its wedges' geometry and
// moments, its corner sums are gathered (B) or routed by a lateral march (B^T).
//
// The column stencils of kernels_stokes.hip are the same products in half the time and
// closer to 64 bits, and a single product takes them.  A solve does not: the CG on its
// preconditioner's coarsest level stops at a loose tolerance on an ill-conditioned
// operator and amplifies the last bits of everything before it -- one rounding in the
// right-hand side of a two-level Stokes step moved its velocity by 1e-9 -- so the
// Krylov operator and the preconditioner's B^T keep this form, and a solve its result.
//
// Moments as in kernels_stokes.hip: the divergence of u_h on a wedge is, per node level t,
//   |det J| div u_h = sgn(D) sum_t [ r g R_t (alpha_t - xi bx_t - eta be_t)
//                                    + r^2 R_t' (sigma_t + xi bx_t + eta be_t) ]
//   du1 = u_1t - u_0t, du2 = u_2t - u_0t,
//   alpha_t = v1.du1 + v3.du2, sigma_t = nv.u_0t, bx_t = nv.du1, be_t = nv.du2,
// so against the coarse shape (il, ir)
//   (B u)_i = -sgn(D) [ P0_ir M0_il + Px_ir Mx_il + Pe_ir Me_il ]
//   P0_ir = sum_t alpha_t A_(ir,t) + sigma_t C_(ir,t)
//   Px_ir = sum_t bx_t (C - A)_(ir,t),   Pe_ir = sum_t be_t (C - A)_(ir,t)
// and B^T is the transpose: with q0_ir = sum_il p_i M0_il (qx, qe likewise) and per level
//   X_t = sum_ir A q0, Y_t = sum_ir C q0, Zx_t = sum_ir (C - A) qx, Ze_t = sum_ir (C - A) qe,
// the node values are -sgn(D) times
//   (0, t): -X_t (v1 + v3) + (Y_t - Zx_t - Ze_t) nv
//   (1, t):  X_t v1 + Zx_t nv
//   (2, t):  X_t v3 + Ze_t nv.
// Velocity at 10 x 65 x 65 x 65 nodes, FP64, free-slip: B^T (Add) 85 us, B 74 with its gather.
#include "tn_cell.hpp"
#include "tn_coupling.hpp"
#include "tn_eps_march.hpp"
#include "tn_internal.hpp"
#include "tn_march.hpp"
#include "tn_stokes.hpp"

namespace tn {
namespace {

using cellops::dot3;
using cellops::V3;

template <typename T>
struct RadMoments {
    T A[2][2];  // [ir][t] int rad_ir r g R_t
    T C[2][2];  // [ir][t] R_t' int rad_ir r^2
};

// fine radial cell (r1, r2) in position frw (0 lower, 1 upper) of its coarse
// cell; scale 0 zeroes every moment (lanes past the last cell)
template <typename T>
__device__ inline RadMoments<T> radial_moments(double r1, double r2, int frw, double scale)
{
    const double g = 0.5 * (r2 - r1);
    double A[2][2] = {{0, 0}, {0, 0}}, rr[2] = {0, 0};
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const double z = s ? GAUSS2 : -GAUSS2;
        const double r = r1 + g * (1 + z);
        const double R[2] = {0.5 * (1 - z), 0.5 * (1 + z)};
        const double rad[2] = {frw ? 0.25 * (1 - z) : 0.25 * (3 - z), frw ? 0.25 * (3 + z) : 0.25 * (1 + z)};
#pragma unroll
        for (int ir = 0; ir < 2; ++ir) {
            A[ir][0] += rad[ir] * r * g * R[0];
            A[ir][1] += rad[ir] * r * g * R[1];
            rr[ir] += rad[ir] * r * r;
        }
    }
    RadMoments<T> m;
#pragma unroll
    for (int ir = 0; ir < 2; ++ir) {
        m.A[ir][0] = (T)(scale * A[ir][0]);
        m.A[ir][1] = (T)(scale * A[ir][1]);
        m.C[ir][0] = (T)(-0.5 * scale * rr[ir]);
        m.C[ir][1] = (T)(0.5 * scale * rr[ir]);
    }
    return m;
}

template <typename T>
struct LatWedge {
    V3<T> v1, v3, nv;
    T sg;  // -sgn(D): the sign of B folded in
};

template <typename T>
__device__ inline V3<T> cross3(const V3<T>& a, const V3<T>& b)
{
    return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}

template <typename T>
__device__ inline LatWedge<T> lat_wedge(const V3<T>& P0, const V3<T>& P1, const V3<T>& P2)
{
    const V3<T> a{P1.x - P0.x, P1.y - P0.y, P1.z - P0.z}, b{P2.x - P0.x, P2.y - P0.y, P2.z - P0.z};
    LatWedge<T> L;
    L.v1 = cross3(b, P0);
    L.v3 = cross3(P0, a);
    L.nv = cross3(a, b);
    L.sg = dot3(a, L.v1) > T(0) ? T(-1) : T(1);
    return L;
}

template <typename T>
__device__ inline V3<T> load_coord(const double* coords, int64_t lat)
{
    return {(T)coords[3 * lat], (T)coords[3 * lat + 1], (T)coords[3 * lat + 2]};
}

// trial-side boundary treatment of a shell node value: Dirichlet drops it,
// free-slip keeps its tangential part (normal: the node's radial direction)
template <typename T>
__device__ inline void trial_bc(V3<T>& u, int mode, const V3<T>& P)
{
    if (mode == TN_DIRICHLET) {
        u = {T(0), T(0), T(0)};
    } else if (mode == TN_FREESLIP) {
        const V3<T>& nn = P;  // lateral coordinates are unit vectors
        const T un = dot3(nn, u);
        u = {u.x - un * nn.x, u.y - un * nn.y, u.z - un * nn.z};
    }
}

// (B u) contributions of one fine wedge to its six coarse dofs:
// out[il][ir] += ..., u0/u1/u2 at node levels t = 0, 1
template <typename T>
__device__ inline void div_wedge(const LatWedge<T>& L, const T (*M)[3], const RadMoments<T>& rm, const V3<T> u0[2],
                                 const V3<T> u1[2], const V3<T> u2[2], T out[3][2])
{
    T al[2], sgm[2], bx[2], be[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const V3<T> du1{u1[t].x - u0[t].x, u1[t].y - u0[t].y, u1[t].z - u0[t].z};
        const V3<T> du2{u2[t].x - u0[t].x, u2[t].y - u0[t].y, u2[t].z - u0[t].z};
        al[t] = dot3(L.v1, du1) + dot3(L.v3, du2);
        sgm[t] = dot3(L.nv, u0[t]);
        bx[t] = dot3(L.nv, du1);
        be[t] = dot3(L.nv, du2);
    }
#pragma unroll
    for (int ir = 0; ir < 2; ++ir) {
        const T ca0 = rm.C[ir][0] - rm.A[ir][0], ca1 = rm.C[ir][1] - rm.A[ir][1];
        const T P0 = L.sg * (al[0] * rm.A[ir][0] + sgm[0] * rm.C[ir][0] + al[1] * rm.A[ir][1] + sgm[1] * rm.C[ir][1]);
        const T Px = L.sg * (bx[0] * ca0 + bx[1] * ca1);
        const T Pe = L.sg * (be[0] * ca0 + be[1] * ca1);
#pragma unroll
        for (int il = 0; il < 3; ++il) out[il][ir] += P0 * M[il][0] + Px * M[il][1] + Pe * M[il][2];
    }
}

// (B^T p) contributions of one fine wedge to its six velocity nodes:
// p[il][ir] coarse values, y0/y1/y2 at node levels t = 0, 1 (accumulated)
template <typename T>
__device__ inline void grad_wedge(const LatWedge<T>& L, const T (*M)[3], const RadMoments<T>& rm, const T p[3][2],
                                  T y0[2][3], T y1[2][3], T y2[2][3])
{
    T q0[2], qx[2], qe[2];
#pragma unroll
    for (int ir = 0; ir < 2; ++ir) {
        q0[ir] = L.sg * (p[0][ir] * M[0][0] + p[1][ir] * M[1][0] + p[2][ir] * M[2][0]);
        qx[ir] = L.sg * (p[0][ir] * M[0][1] + p[1][ir] * M[1][1] + p[2][ir] * M[2][1]);
        qe[ir] = L.sg * (p[0][ir] * M[0][2] + p[1][ir] * M[1][2] + p[2][ir] * M[2][2]);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const T X = rm.A[0][t] * q0[0] + rm.A[1][t] * q0[1];
        const T Y = rm.C[0][t] * q0[0] + rm.C[1][t] * q0[1];
        const T ca0 = rm.C[0][t] - rm.A[0][t], ca1 = rm.C[1][t] - rm.A[1][t];
        const T Zx = ca0 * qx[0] + ca1 * qx[1];
        const T Ze = ca0 * qe[0] + ca1 * qe[1];
        const T s0 = Y - Zx - Ze;
        y0[t][0] += s0 * L.nv.x - X * (L.v1.x + L.v3.x);
        y0[t][1] += s0 * L.nv.y - X * (L.v1.y + L.v3.y);
        y0[t][2] += s0 * L.nv.z - X * (L.v1.z + L.v3.z);
        y1[t][0] += X * L.v1.x + Zx * L.nv.x;
        y1[t][1] += X * L.v1.y + Zx * L.nv.y;
        y1[t][2] += X * L.v1.z + Zx * L.nv.z;
        y2[t][0] += X * L.v3.x + Ze * L.nv.x;
        y2[t][1] += X * L.v3.y + Ze * L.nv.y;
        y2[t][2] += X * L.v3.z + Ze * L.nv.z;
    }
}

// Lateral corners of a quad: k = 0 (x, y), 1 (x+1, y), 2 (x, y+1), 3 (x+1, y+1);
// wedge w's vertices 0, 1, 2 in that numbering (WOFF[w][0..2]).
__device__ constexpr int WK[2][3] = {{0, 1, 2}, {3, 2, 1}};

// B: a wave per coarse lateral quad (X, Y) and chunk of 64 coarse radial
// cells (one per lane).  A lane sums the 16 fine wedges of its coarse cell
// into the cell's 8 corners; the shared radial level is merged by a lane
// shuffle, so a lane writes its lower 4 corner sums per cell and the chunk's
// top lane the upper 4 once per chunk.  k_div_gather then sums, per pressure
// node copy, the (at most 4) lateral quads' values in a fixed order: no
// atomics, the same result on every run.
template <typename T>
__global__ __launch_bounds__(256) void k_div_cells(DivCellArgs<T> a)
{
    const int lane = threadIdx.x & 63;
    const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int nqc = a.nc - 1, ncrc = a.nrc - 1;
    const int nch = (ncrc + 63) >> 6;
    if (wave >= 10LL * nqc * nqc * nch) return;  // wave-uniform
    int64_t t = wave;
    const int h = (int)(t % nch);
    t /= nch;
    const int Y = (int)(t % nqc);
    t /= nqc;
    const int X = (int)(t % nqc);
    const int d = (int)(t / nqc);
    const int R = 64 * h + lane;
    const bool valid = R < ncrc;
    const int Rc = valid ? R : ncrc - 1;
    const int toplane = min(63, ncrc - 1 - 64 * h);
    const int nf = a.nf, nrf = a.nrf;
    const int64_t Nf = 10LL * nf * nf * nrf;
    const double sc = valid ? 1.0 : 0.0;
    const RadMoments<T> rm[2] = {radial_moments<T>(a.radii[2 * Rc], a.radii[2 * Rc + 1], 0, sc),
                                 radial_moments<T>(a.radii[2 * Rc + 1], a.radii[2 * Rc + 2], 1, sc)};
    const int bl = Rc == 0 ? a.bc_cmb : TN_NEUMANN;           // fine level 2R
    const int tl = Rc == ncrc - 1 ? a.bc_surf : TN_NEUMANN;  // fine level 2R + 2
    T acc[4][2] = {{0, 0}, {0, 0}, {0, 0}, {0, 0}};
    // one fine quad at a time (all four at once would exceed the register file in FP64)
#pragma unroll 1
    for (int dy = 0; dy < 2; ++dy)
#pragma unroll 1
        for (int dx = 0; dx < 2; ++dx) {
            const int fx = 2 * X + dx, fy = 2 * Y + dy;
            const int64_t l00 = ((int64_t)d * nf + fx) * nf + fy;
            const int64_t latc[4] = {l00, l00 + nf, l00 + 1, l00 + nf + 1};
            V3<T> u[4][3];
            V3<T> P[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int64_t ib = latc[k] * nrf + 2 * Rc;
#pragma unroll
                for (int l = 0; l < 3; ++l) u[k][l] = {a.u[ib + l], a.u[Nf + ib + l], a.u[2 * Nf + ib + l]};
                P[k] = load_coord<T>(a.coords, latc[k]);
            }
            if (bl != TN_NEUMANN || tl != TN_NEUMANN) {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    if (bl != TN_NEUMANN) trial_bc(u[k][0], bl, P[k]);
                    if (tl != TN_NEUMANN) trial_bc(u[k][2], tl, P[k]);
                }
            }
#pragma unroll
            for (int w = 0; w < 2; ++w) {
                const int k0 = WK[w][0], k1 = WK[w][1], k2 = WK[w][2];
                const LatWedge<T> L = lat_wedge(P[k0], P[k1], P[k2]);
                const int flw = fine_lateral_wedge_idx(dx, dy, w);
                T M[3][3];
#pragma unroll
                for (int il = 0; il < 3; ++il)
#pragma unroll
                    for (int j = 0; j < 3; ++j) M[il][j] = (T)LATM.m[flw][il][j];
                T out[3][2] = {{0, 0}, {0, 0}, {0, 0}};
#pragma unroll
                for (int frw = 0; frw < 2; ++frw) {
                    const V3<T> u0[2] = {u[k0][frw], u[k0][frw + 1]};
                    const V3<T> u1[2] = {u[k1][frw], u[k1][frw + 1]};
                    const V3<T> u2[2] = {u[k2][frw], u[k2][frw + 1]};
                    div_wedge(L, M, rm[frw], u0, u1, u2, out);
                }
                // coarse corners of wedge w: WOFF[w][il] in the k numbering
#pragma unroll
                for (int il = 0; il < 3; ++il) {
                    acc[WK[w][il]][0] += out[il][0];
                    acc[WK[w][il]][1] += out[il][1];
                }
            }
        }
    const int64_t ncol = 10LL * nqc * nqc, ncell = ncol * ncrc;
    const int64_t col = ((int64_t)d * nqc + X) * nqc + Y;
    T* ctop = a.csum + 4 * ncell;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        T below = __shfl_up(acc[k][1], 1, 64);
        if (lane == 0) below = T(0);
        if (valid) a.csum[k * ncell + col * ncrc + R] = acc[k][0] + below;
        if (lane == toplane) ctop[(k * ncol + col) * nch + h] = acc[k][1];
    }
}

// Pressure node copy (d, X, Y, level): corner k of quad (X - (k & 1), Y - (k >> 1)).
template <typename T>
__global__ __launch_bounds__(256) void k_div_gather(DivCellArgs<T> a)
{
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int nc = a.nc, nrc = a.nrc, nqc = nc - 1, ncrc = nrc - 1;
    if (tid >= 10LL * nc * nc * nrc) return;
    const int nch = (ncrc + 63) >> 6;
    const int64_t ncol = 10LL * nqc * nqc, ncell = ncol * ncrc;
    const T* ctop = a.csum + 4 * ncell;
    const int lev = (int)(tid % nrc);
    const int64_t lat = tid / nrc;
    const int Yn = (int)(lat % nc);
    const int Xn = (int)((lat / nc) % nc);
    const int d = (int)(lat / ((int64_t)nc * nc));
    T v = T(0);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int qx = Xn - (k & 1), qy = Yn - (k >> 1);
        if (qx < 0 || qy < 0 || qx > nqc - 1 || qy > nqc - 1) continue;
        const int64_t col = ((int64_t)d * nqc + qx) * nqc + qy;
        if (lev < ncrc) v += a.csum[k * ncell + col * ncrc + lev];
        // first level of a chunk > 0, or the top level: the previous chunk's top
        if ((lev > 0 && (lev & 63) == 0) || lev == ncrc) v += ctop[(k * ncol + col) * nch + ((lev - 1) >> 6)];
    }
    a.p[tid] = v;
}

// Decomposition.  A block of W waves owns W-1 lateral node rows of one
// diamond and one segment of `seg` node columns.  Wave w handles the quad
// strip x = x0 - 1 + w and marches over the quads of that strip in y; its 64
// lanes are 64 radial cells (a chunk; chunks of one column follow one after
// the other).  A quad's sums at its four lateral corners are routed
//   corner (x,   y)   own node row, column y   -> complete after this step
//   corner (x,   y+1) own node row, column y+1 -> carried in registers
//   corner (x+1, y)   next wave's row          -> LDS ring, read by wave w+1
//                                                 (LDS counters order producer and consumer)
//   corner (x+1, y+1)                          -> carried, sent next step
// and radially adjacent cells share their node level through a lane shuffle;
// the level above a chunk's last cell goes the same way through that lane and
// is either the top shell (finished) or the first level of the next chunk
// (kept in LDS until that chunk reaches the column).  Every node copy of the
// diamond is finished exactly once; the strip at a block edge is computed
// twice (as the halo wave 0 of the next block).
//
// The per-cell work is a functor Op with
//   void begin_chunk(int c, int cc, bool valid)      lane's radial cell c (cc: clamped)
//   void cell(int d, int x, int y, T yb[4][3], T yt[4][3])
//        adds the quad's corner sums (k = 0 (x,y), 1 (x+1,y), 2 (x,y+1),
//        3 (x+1,y+1); yb at node level c, yt at c+1); called for valid quads
//        only, lanes past the last cell must add zeros
//   void finish(int64_t lat, int level, V3<T> v)     the node copy's final sum
// number of blocks of a launch over a mesh of n x n lateral nodes
inline int march_blocks(int n, int seg, int waves)
{
    const int own = waves - 1;
    return 10 * ((n + own - 1) / own) * ((n + seg - 1) / seg);
}

template <typename T, int W, class Op>
__device__ __forceinline__ void cell_march(Op& op, int n, int nr, int seg, const MarchGuard& guard)
{
    constexpr int OWN = W - 1;
    constexpr int RING = 4;                  // hand-off slots: a producer may lead by RING - 1 steps
    __shared__ T ebuf[RING][W][3][65];       // corner (x+1, y) hand-off; slot 64: chunk-top level
    __shared__ T lvl[W][MARCH_SEG_MAX][3];   // chunk-top level values awaiting the next chunk
    __shared__ int done[W], used[W];         // steps whose hand-off wave w has written / has read
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int ncr = nr - 1;
    const int nxb = (n + OWN - 1) / OWN, nys = (n + seg - 1) / seg;
    int b = xcd_tile(blockIdx.x, gridDim.x);
    const int ys = b % nys;
    b /= nys;
    const int xb = b % nxb;
    const int d = b / nxb;
    const int x = xb * OWN - 1 + w;
    const bool strip_ok = x >= 0 && x <= n - 2;
    const bool row_own = w >= 1 && x <= n - 1;
    const int y0 = ys * seg, y1 = min(y0 + seg, n);
    const int nchunks = (ncr + 63) >> 6;
    if (lane == 0) done[w] = used[w] = 0;
    __syncthreads();
    int step = 0;  // hand-off ring position, continuous over chunks

    for (int h = 0; h < nchunks; ++h) {
        const int c = 64 * h + lane;
        const bool valid = c < ncr;
        const int toplane = min(63, ncr - 1 - 64 * h);
        const bool last = h == nchunks - 1;
        op.begin_chunk(c, valid ? c : ncr - 1, valid);
        T c01[3] = {0, 0, 0}, c11[3] = {0, 0, 0}, c01t[3] = {0, 0, 0}, c11t[3] = {0, 0, 0};

        for (int qy = y0 - 1; qy <= y1 - 1; ++qy, ++step) {
            const bool quad_ok = strip_ok && qy >= 0 && qy <= n - 2;
            T(*E)[65] = ebuf[step % RING][w];
            T yb[4][3], yt[4][3];
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int j = 0; j < 3; ++j) yb[k][j] = yt[k][j] = T(0);
            if (quad_ok) op.cell(d, x, qy, yb, yt);
            // radial merge (node level c = bottom of cell c + top of cell c-1) and routing;
            // the slot is free once the next wave has read what it held RING steps ago
            if (w + 1 < W) march::wait_counter(&used[w + 1], step - RING + 1, guard);
            T part[3], tp[3] = {0, 0, 0};
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                T Mg[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    T up = __shfl_up(yt[k][j], 1, 64);
                    if (lane == 0) up = T(0);
                    Mg[k] = yb[k][j] + up;
                }
                part[j] = Mg[0] + c01[j];
                c01[j] = Mg[2];
                E[j][lane] = Mg[1] + c11[j];
                c11[j] = Mg[3];
            }
            if (lane == toplane) {  // level above this chunk's last cell
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    tp[j] = yt[0][j] + c01t[j];
                    c01t[j] = yt[2][j];
                    E[j][64] = yt[1][j] + c11t[j];
                    c11t[j] = yt[3][j];
                }
            }
            march::post_counter(&done[w], step + 1, lane);
            if (w >= 1) march::wait_counter(&done[w - 1], step + 1, guard);
            if (row_own && qy >= y0) {
                const T(*Ein)[65] = ebuf[step % RING][w - 1];
                const int64_t lat = ((int64_t)d * n + x) * n + qy;
                const int slot = qy - y0;
                if (valid) {
                    V3<T> v{part[0] + Ein[0][lane], part[1] + Ein[1][lane], part[2] + Ein[2][lane]};
                    if (lane == 0 && h > 0) {
                        v.x += lvl[w][slot][0];
                        v.y += lvl[w][slot][1];
                        v.z += lvl[w][slot][2];
                    }
                    op.finish(lat, c, v);
                }
                if (lane == toplane) {
                    const V3<T> v{tp[0] + Ein[0][64], tp[1] + Ein[1][64], tp[2] + Ein[2][64]};
                    if (last) {
                        op.finish(lat, ncr, v);
                    } else {
                        lvl[w][slot][0] = v.x;
                        lvl[w][slot][1] = v.y;
                        lvl[w][slot][2] = v.z;
                    }
                }
            }
            march::post_counter(&used[w], step + 1, lane);
        }
    }
}

// B^T: the lateral march over fine cells: each
// fine cell evaluates its two wedges from the 8 coarse values of its coarse
// cell.  Every velocity node copy is written once (store or read-modify-
// write); Dirichlet shells are left out and free-slip shells projected
// tangentially on the summed value (the test-side masks and rotations of
// gradient.hpp:115-325).
template <typename T>
struct GradCell {
    const GradCellArgs<T> a;  // by value: a reference would put the kernel argument in scratch
    // the arrays, taken from restrict kernel parameters: loads at wave-uniform
    // addresses (the lateral coordinates) can then go through the scalar unit
    const double* coords;
    const T* p;
    T* u;
    int64_t N;
    RadMoments<T> rm;
    int R;
    __device__ GradCell(const GradCellArgs<T>& args, const double* c, const T* pp, T* uu)
        : a(args), coords(c), p(pp), u(uu), N(10LL * args.nf * args.nf * args.nrf)
    {
    }
    __device__ void begin_chunk(int, int cc, bool valid)
    {
        rm = radial_moments<T>(a.radii[cc], a.radii[cc + 1], cc & 1, valid ? 1.0 : 0.0);
        R = cc >> 1;
    }
    __device__ void cell(int d, int x, int qy, T yb[4][3], T yt[4][3])
    {
        const int n = a.nf, nc = a.nc, nrc = a.nrc;
        const int64_t c00 = ((int64_t)d * nc + (x >> 1)) * nc + (qy >> 1);
        const int64_t cl[4] = {c00, c00 + nc, c00 + 1, c00 + nc + 1};
        T pc[4][2];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            pc[k][0] = p[cl[k] * nrc + R];
            pc[k][1] = p[cl[k] * nrc + R + 1];
        }
        const int64_t lat00 = ((int64_t)d * n + x) * n + qy;
        const int64_t latc[4] = {lat00, lat00 + n, lat00 + 1, lat00 + n + 1};
        V3<T> P[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) P[k] = load_coord<T>(coords, latc[k]);
#pragma unroll
        for (int w2 = 0; w2 < 2; ++w2) {
            const int k0 = WK[w2][0], k1 = WK[w2][1], k2 = WK[w2][2];
            const LatWedge<T> L = lat_wedge(P[k0], P[k1], P[k2]);
            const int flw = fine_lateral_wedge_idx(x & 1, qy & 1, w2);
            T M[3][3];
#pragma unroll
            for (int il = 0; il < 3; ++il)
#pragma unroll
                for (int j = 0; j < 3; ++j) M[il][j] = (T)LATM.m[flw][il][j];
            const T p[3][2] = {{pc[k0][0], pc[k0][1]}, {pc[k1][0], pc[k1][1]}, {pc[k2][0], pc[k2][1]}};
            T o0[2][3] = {{0, 0, 0}, {0, 0, 0}}, o1[2][3] = {{0, 0, 0}, {0, 0, 0}}, o2[2][3] = {{0, 0, 0}, {0, 0, 0}};
            grad_wedge(L, M, rm, p, o0, o1, o2);
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                yb[k0][j] += o0[0][j];
                yt[k0][j] += o0[1][j];
                yb[k1][j] += o1[0][j];
                yt[k1][j] += o1[1][j];
                yb[k2][j] += o2[0][j];
                yt[k2][j] += o2[1][j];
            }
        }
    }
    __device__ void finish(int64_t lat, int level, V3<T> v)
    {
        const int mode = level == 0 ? a.bc_cmb : (level == a.nrf - 1 ? a.bc_surf : TN_NEUMANN);
        const int64_t idx = lat * a.nrf + level;
        if (mode == TN_DIRICHLET) {
            if (a.add) return;
            v = {T(0), T(0), T(0)};
        } else if (mode == TN_FREESLIP) {
            const V3<T> nn = load_coord<T>(coords, lat);  // unit vector
            const T vn = dot3(nn, v);
            v = {v.x - vn * nn.x, v.y - vn * nn.y, v.z - vn * nn.z};
        }
        if (a.add) {
            u[idx] += v.x;
            u[N + idx] += v.y;
            u[2 * N + idx] += v.z;
        } else {
            u[idx] = v.x;
            u[N + idx] = v.y;
            u[2 * N + idx] = v.z;
        }
    }
};

template <typename T, int W>
// (3 waves per SIMD: the FP64 build fits 168 VGPRs without spills)
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(3))) void k_grad_march(GradCellArgs<T> a, const double* __restrict__ coords,
                                                         const T* __restrict__ p, T* __restrict__ u)
{
    GradCell<T> op(a, coords, p, u);
    cell_march<T, W>(op, a.nf, a.nrf, a.seg, a.guard);
}

}  // namespace

template <typename T>
void launch_div_cells(const DivCellArgs<T>& a, hipStream_t s)
{
    TN_REQUIRE(a.nf == 2 * a.nc - 1 && a.nrf == 2 * a.nrc - 1 && a.nrc >= 2 && a.nc >= 2,
               "B: velocity mesh must be the pressure mesh refined once");
    TN_REQUIRE(a.csum, "B: corner-sum scratch missing");
    const int64_t waves = 10LL * (a.nc - 1) * (a.nc - 1) * ((a.nrc - 1 + 63) / 64);
    hipLaunchKernelGGL(k_div_cells<T>, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, s, a);
    TN_HIP(hipGetLastError());
    const int64_t Nc = 10LL * a.nc * a.nc * a.nrc;
    hipLaunchKernelGGL(k_div_gather<T>, dim3((unsigned)((Nc + 255) / 256)), dim3(256), 0, s, a);
    TN_HIP(hipGetLastError());
}

template <typename T>
void launch_grad_cells(const GradCellArgs<T>& a, hipStream_t s)
{
    TN_REQUIRE(a.nf == 2 * a.nc - 1 && a.nrf == 2 * a.nrc - 1 && a.nrc >= 2 && a.nc >= 2,
               "B^T: velocity mesh must be the pressure mesh refined once");
    TN_REQUIRE(a.seg >= 1 && a.seg <= MARCH_SEG_MAX, "B^T: segment length out of range");
    constexpr int W = grad_march_waves<T>();
    hipLaunchKernelGGL((k_grad_march<T, W>), dim3((unsigned)march_blocks(a.nf, a.seg, W)), dim3(64 * W), 0, s, a,
                       a.coords, a.p, a.u);
    TN_HIP(hipGetLastError());
}

template void launch_div_cells<double>(const DivCellArgs<double>&, hipStream_t);
template void launch_div_cells<float>(const DivCellArgs<float>&, hipStream_t);
template void launch_grad_cells<double>(const GradCellArgs<double>&, hipStream_t);
template void launch_grad_cells<float>(const GradCellArgs<float>&, hipStream_t);

}  // namespace tn
