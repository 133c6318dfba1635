// Stokes coupling: B (Divergence, divergence.hpp:117-323), p_c += -int div(u_h) q_H,
// and its transpose B^T (Gradient, gradient.hpp:115-325), u += -int p_H div(v_h): the
// products that a program asks for.  The solves keep the form by cells, whose roundings
// their results rest on (kernels_coupling_cells.hip).
//
// Velocity lives on the fine mesh, pressure on the mesh one level coarser; each
// fine wedge integrates with the 6-point Felippa 3x2 rule and the coarse shape
// functions evaluated on the fine wedge (integrands.hpp:103-243).  The coarse dofs
// a fine wedge couples to are those of coarse cell (x/2, y/2, r/2) in the node
// pattern of the FINE wedge index, exactly as the reference scatters them
// (kernel_helpers.hpp:396-424); for the two centre fine wedges this is the
// neighbouring coarse wedge.
//
// Wedge moments.  A fine wedge with lateral unit-sphere vertices P0, P1, P2
// (a = P1 - P0, b = P2 - P0) between radii r1 < r2 is x = r(zeta) c(xi, eta) with
// c = P0 + xi a + eta b, r = r1 + g (1 + zeta), g = (r2 - r1) / 2.  Its Jacobian
// [r a, r b, g c] has det J = r^2 g D, D = det[a, b, P0], constant over the
// triangle, and for a shape N
//   |det J| grad N = sgn(D) [ r g (N_xi (v1 - xi nv) + N_eta (v3 - eta nv))
//                             + r^2 N_zeta nv ],
//   v1 = b x P0,  v3 = P0 x a,  nv = a x b.
// Against a coarse shape lat_il(xi, eta) rad_ir(zeta) the integrand has lateral
// degree <= 2 and radial degree <= 3, which the rule integrates exactly, so the sum
// is a moment formula.  With the lateral moments M0, Mx, Me = int lat_il (1, xi,
// eta) and the radial ones A_(ir,t) = int rad_ir r g R_t, C_(ir,t) = R_t' int rad_ir
// r^2 over [-1, 1], the coupling of velocity node (m, t) (lateral vertex m, level t)
// with coarse dof (il, ir) is the vector  A_(ir,t) al + C_(ir,t) ga,
//   m = 0: al = s [(Mx + Me) nv - M0 (v1 + v3)],  ga = s (M0 - Mx - Me) nv
//   m = 1: al = s [M0 v1 - Mx nv],                ga = s Mx nv
//   m = 2: al = s [M0 v3 - Me nv],                ga = s Me nv,    s = -sgn(D).
//
// Column stencil.  al and ga depend on the lateral position only, so summed over
// the wedges of a fine node column F and a coarse node column K they are two vectors
// per pair (F, K), and the radial moments summed over the layers of a level are
// three weights of A and of C:
//   B^T: u_F(r) = sum_K [ al_FK sum_q wA_q(r) p_K(q) + ga_FK sum_q wC_q(r) p_K(q) ]
//   B:   p_K(q) = sum_F [ al_FK . sum_r wA_q(r) u_F(r) + ga_FK . sum_r wC_q(r) u_F(r) ]
// with at most 7 coarse columns per fine one.  The vectors are tabulated once per
// operator (48 numbers a fine column: a quarter of a velocity vector at 65 levels); no
// geometry, no scatter and no order of waves is left in either product, and every
// output is written once, in a fixed order.  A wave keeps one x and walks y, its
// lanes are 64 levels; B^T holds the radial sums of the coarse columns in reach in
// registers, B the open sums of three coarse columns.
//
// Both are bound by the latency of a step's loads.  The table entries of a column are
// loaded like a vector (a lane each) one step ahead and spread over the lanes through
// LDS: as scalar loads, ready only when needed, B took 80 us where it now takes 37.
// Velocity at 10 x 65 x 65 x 65 nodes, FP64, free-slip, kernels in us: B^T (Add) 89 as a
// march over cells with hand-offs between waves, 38 now where its velocity is still in
// the caches (repeated alone: 66 + 66 MB read and written, 16 MB of table: 3.9 TB/s) and
// 48 in the block apply, behind the viscous block (103 as a march); B 73 + 6 as a cell
// pass with a gather, 37 now.  At 10 x 9 x 9 x 9 nodes 25 -> 5 and 16 -> 10.  FP32 against FP64 (relative L2): 9.4e-7
// as cell geometry in FP32, 0.8e-7 with vectors made in FP64 and rounded once (B 1.2e-7).
#include <algorithm>
#include <type_traits>

#include "tn_cell.hpp"
#include "tn_coupling.hpp"
#include "tn_eps_march.hpp"
#include "tn_march.hpp"
#include "tn_stokes.hpp"

namespace tn {
namespace {

// Table slot of coarse column offset (dx, dy) from (x >> 1, y >> 1) for a fine
// column of parities (xo, yo); the offsets in reach:
//   even, even: the node and its six neighbours along the edges
//   even, odd:  dx in -1..1, dy in 0..1    odd, even: dx in 0..1, dy in -1..1
//   odd, odd:   dx, dy in 0..1
__host__ __device__ constexpr int coupling_slot(int xo, int yo, int dx, int dy)
{
    if (!xo && !yo)
        return dx == -1 ? (dy == 0 ? 0 : 1) : dx == 0 ? 3 + dy : (dy == -1 ? 5 : 6);
    if (!xo) return (dx + 1) * 2 + dy;
    if (!yo) return dx * 3 + dy + 1;
    return dx * 2 + dy;
}
__host__ __device__ constexpr bool coupling_has(int xo, int yo, int dx, int dy)
{
    if (!xo && !yo) return dx >= -1 && dx <= 1 && dy >= -1 && dy <= 1 && dx + dy >= -1 && dx + dy <= 1 && !(dx && dx == dy);
    return dx >= (xo ? 0 : -1) && dx <= 1 && dy >= (yo ? 0 : -1) && dy <= 1;
}

// lateral table: a thread per fine node column and slot (slot values al[3], ga[3]; the
// thread past the last slot writes the normal).  A thread with all seven slots kept them
// in scratch and took 36 us for 42250 columns, 22 so.
template <typename T>
__global__ __launch_bounds__(256) void k_coupling_table(const double* __restrict__ coords, int n, T* __restrict__ tab)
{
    constexpr int OFF[2][3][2] = {{{0, 0}, {1, 0}, {0, 1}}, {{1, 1}, {0, 1}, {1, 0}}};
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t t = tid >> 3;
    const int slot = (int)(tid & 7);
    static_assert(COUPLING_SLOTS == 7 && COUPLING_ENTRIES == 6 * (COUPLING_SLOTS + 1), "eight threads per column");
    if (t >= 10LL * n * n) return;
    T* o = tab + t * COUPLING_ENTRIES + 6 * slot;
    if (slot == COUPLING_SLOTS) {
        for (int j = 0; j < 6; ++j) o[j] = j < 3 ? (T)coords[3 * t + j] : T(0);
        return;
    }
    const int y = (int)(t % n), x = (int)((t / n) % n), d = (int)(t / ((int64_t)n * n));
    double v[6] = {0, 0, 0, 0, 0, 0};
    for (int qx = x - 1; qx <= x; ++qx)
        for (int qy = y - 1; qy <= y; ++qy) {
            if (qx < 0 || qy < 0 || qx > n - 2 || qy > n - 2) continue;
#pragma unroll
            for (int w = 0; w < 2; ++w) {
                int m = -1, il = -1;  // vertex of the wedge here, coarse shape of the slot
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    if (qx + OFF[w][i][0] == x && qy + OFF[w][i][1] == y) m = i;
                    if (coupling_slot(x & 1, y & 1, (qx >> 1) + OFF[w][i][0] - (x >> 1),
                                      (qy >> 1) + OFF[w][i][1] - (y >> 1)) == slot)
                        il = i;
                }
                if (m < 0 || il < 0) continue;
                double P[3][3];
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    const double* c = coords + 3 * (((int64_t)d * n + qx + OFF[w][i][0]) * n + qy + OFF[w][i][1]);
#pragma unroll
                    for (int j = 0; j < 3; ++j) P[i][j] = c[j];
                }
                double a[3], b[3];
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    a[j] = P[1][j] - P[0][j];
                    b[j] = P[2][j] - P[0][j];
                }
                const double v1[3] = {b[1] * P[0][2] - b[2] * P[0][1], b[2] * P[0][0] - b[0] * P[0][2],
                                      b[0] * P[0][1] - b[1] * P[0][0]};
                const double v3[3] = {P[0][1] * a[2] - P[0][2] * a[1], P[0][2] * a[0] - P[0][0] * a[2],
                                      P[0][0] * a[1] - P[0][1] * a[0]};
                const double nv[3] = {a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]};
                const double s = a[0] * v1[0] + a[1] * v1[1] + a[2] * v1[2] > 0.0 ? -1.0 : 1.0;
                const double* M = LATM.m[fine_lateral_wedge_idx(qx & 1, qy & 1, w)][il];
                const double M0 = M[0], Mx = M[1], Me = M[2];
                const double n0 = m == 0 ? Mx + Me : (m == 1 ? -Mx : -Me);
                const double n1 = m == 0 ? M0 - Mx - Me : (m == 1 ? Mx : Me);
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    const double vv = m == 0 ? -(v1[j] + v3[j]) : (m == 1 ? v1[j] : v3[j]);
                    v[j] += s * (n0 * nv[j] + M0 * vv);
                    v[3 + j] += s * n1 * nv[j];
                }
            }
        }
#pragma unroll
    for (int j = 0; j < 6; ++j) o[j] = (T)v[j];
}

// radial weights: [6][nr], wA_0..2 and wC_0..2 of fine level r for the coarse levels
// b, b + 1, b + 2 with b = r/2 - 1 (r even) or (r - 1)/2 (r odd, third weight 0)
template <typename T>
__global__ __launch_bounds__(256) void k_coupling_radial(const double* __restrict__ radii, int nr, T* __restrict__ w)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nr) return;
    double o[6] = {0, 0, 0, 0, 0, 0};
    for (int below = 0; below < 2; ++below) {  // layer r (the level is its bottom), layer r - 1 (its top)
        const int layer = r - below, t = below;
        if (layer < 0 || layer > nr - 2) continue;
        const double r1 = radii[layer], g = 0.5 * (radii[layer + 1] - r1);
        const int frw = layer & 1;
        double A[2] = {0, 0}, C[2] = {0, 0};
        for (int s = 0; s < 2; ++s) {
            const double z = s ? GAUSS2 : -GAUSS2;
            const double rr = r1 + g * (1 + z);
            const double R = t ? 0.5 * (1 + z) : 0.5 * (1 - z);
            const double rad[2] = {frw ? 0.25 * (1 - z) : 0.25 * (3 - z), frw ? 0.25 * (3 + z) : 0.25 * (1 + z)};
            for (int ir = 0; ir < 2; ++ir) {
                A[ir] += rad[ir] * rr * g * R;
                C[ir] += (t ? 0.5 : -0.5) * rad[ir] * rr * rr;
            }
        }
        const int base = (r & 1) ? (r >> 1) : (r >> 1) - 1;
        const int q = (layer >> 1) - base;
        for (int ir = 0; ir < 2; ++ir) {
            o[q + ir] += A[ir];
            o[3 + q + ir] += C[ir];
        }
    }
    for (int k = 0; k < 6; ++k) w[(int64_t)k * nr + r] = (T)o[k];
}

// Levels past whole chunks of B^T that go to a thread each: the top level of 64 k + 1
// as a chunk of its own takes a second wave per column (65 levels: 52 us, not 38).
constexpr int TAIL = 4;
// ---------------------------------------------------------------- B^T
// one node's value: Dirichlet left out, free-slip projected
template <typename T>
__device__ __forceinline__ void mask_node(int mode, const T* nv, T (&v)[3])
{
    if (mode == TN_DIRICHLET) {
        v[0] = v[1] = v[2] = T(0);
    } else if (mode == TN_FREESLIP) {
        const T vn = nv[0] * v[0] + nv[1] * v[1] + nv[2] * v[2];
#pragma unroll
        for (int j = 0; j < 3; ++j) v[j] -= vn * nv[j];
    }
}

// A wave takes `run` columns (even) of one x, its lanes 64 levels.
template <typename T, int XO>
__device__ __forceinline__ void grad_strip(const GradArgs<T>& a, const T* __restrict__ tab, const T* __restrict__ wr,
                                           const T* __restrict__ p, T* __restrict__ u, T (*lds)[COUPLING_ENTRIES],
                                           int d, int x, int y0, int y1, int rbase)
{
    constexpr int X0 = XO ? 0 : -1, NX = XO ? 2 : 3;  // coarse columns X + X0 .. X + 1
    const int n = a.nf, nr = a.nrf, nc = a.nc, nrc = a.nrc;
    const int64_t N = 10LL * n * n * nr;
    const int lane = threadIdx.x & 63;
    const bool valid = rbase + lane < nr;
    const int r = valid ? rbase + lane : nr - 1;
    T wA[3], wC[3];
    int lev[3];
    {
        const int base = (r & 1) ? (r >> 1) : (r >> 1) - 1;
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            // a level of weight 0 is replaced by one the node does couple to
            lev[q] = min(max(base + min(q, (r & 1) ? 1 : 2), 0), nrc - 1);
            wA[q] = wr[q * nr + r];
            wC[q] = wr[(3 + q) * nr + r];
        }
    }
    const int mode = r == 0 ? a.bc_cmb : (r == nr - 1 ? a.bc_surf : (int)TN_NEUMANN);
    const int X = x >> 1;
    // Coarse columns (X + X0 + i, Y) of row Y: values, then radial sums.  A column
    // outside the diamond is replaced by one in reach, so that no load waits for a
    // branch, and its sums by 0.
    struct Raw {
        T p[NX][3];
    };
    auto raw = [&](int Y, Raw& o) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NX; ++i) {
            const int cx = min(max(X + X0 + i, 0), nc - 1), cy = min(max(Y, 0), nc - 1);
            const T* pc = p + (((int64_t)d * nc + cx) * nc + cy) * nrc;
#pragma unroll
            for (int q = 0; q < 3; ++q) o.p[i][q] = pc[lev[q]];
        }
    };
    T SA[NX][3], SC[NX][3];  // rows Y - 1, Y, Y + 1
    auto sums = [&](int j, int Y, const Raw& o) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NX; ++i) {
            const bool in = X + X0 + i >= 0 && X + X0 + i < nc && Y >= 0 && Y < nc;  // wave-uniform
            const T sa = wA[0] * o.p[i][0] + wA[1] * o.p[i][1] + wA[2] * o.p[i][2];
            const T sc = wC[0] * o.p[i][0] + wC[1] * o.p[i][1] + wC[2] * o.p[i][2];
            SA[i][j] = in ? sa : T(0);
            SC[i][j] = in ? sc : T(0);
        }
    };
    struct Node {
        T tab, old[3];
    };
    auto load = [&](int y, Node& o) __attribute__((always_inline)) {
        const int64_t lat = __builtin_amdgcn_readfirstlane((d * n + x) * n + min(y, n - 1));
        o.tab = tab[lat * COUPLING_ENTRIES + min(lane, COUPLING_ENTRIES - 1)];
#pragma unroll
        for (int j = 0; j < 3; ++j) o.old[j] = a.add ? u[j * N + lat * nr + r] : T(0);
    };
    auto node = [&](int y, auto yo, const Node& o, const T* e) __attribute__((always_inline)) {
        constexpr int YO = decltype(yo)::value;
        const int64_t lat = __builtin_amdgcn_readfirstlane((d * n + x) * n + y);
        T v[3] = {0, 0, 0};
#pragma unroll
        for (int dx = X0; dx <= 1; ++dx)
#pragma unroll
            for (int dy = -1; dy <= 1; ++dy) {
                if (!coupling_has(XO, YO, dx, dy)) continue;
                const T* s = e + 6 * coupling_slot(XO, YO, dx, dy);
                const T sa = SA[dx - X0][dy + 1], sc = SC[dx - X0][dy + 1];
#pragma unroll
                for (int j = 0; j < 3; ++j) v[j] += s[j] * sa + s[3 + j] * sc;
            }
        const T nv[3] = {e[COUPLING_NORMAL], e[COUPLING_NORMAL + 1], e[COUPLING_NORMAL + 2]};
        mask_node(mode, nv, v);
        if (valid) {
#pragma unroll
            for (int j = 0; j < 3; ++j) u[j * N + lat * nr + r] = o.old[j] + v[j];
        }
    };
    Raw next;
    raw((y0 >> 1) - 1, next);
    sums(0, (y0 >> 1) - 1, next);
    raw(y0 >> 1, next);
    sums(1, y0 >> 1, next);
    raw((y0 >> 1) + 1, next);
    Node ne, no;
    load(y0, ne);
    load(y0 + 1, no);
    // y0 is even: an even column, then the odd one beside it; the loads of the next
    // pair are under way meanwhile
#pragma unroll 1
    for (int y = y0; y < y1; y += 2) {
        sums(2, (y >> 1) + 1, next);
        const Node e = ne, o = no;
        __builtin_amdgcn_wave_barrier();
        if (lane < COUPLING_ENTRIES) {
            lds[0][lane] = e.tab;
            lds[1][lane] = o.tab;
        }
        __builtin_amdgcn_wave_barrier();
        if (y + 2 < y1) {
            raw((y >> 1) + 2, next);
            load(y + 2, ne);
            load(y + 3, no);
        }
        node(y, std::integral_constant<int, 0>{}, e, lds[0]);
        if (y + 1 < y1) node(y + 1, std::integral_constant<int, 1>{}, o, lds[1]);
#pragma unroll
        for (int i = 0; i < NX; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                SA[i][j] = SA[i][j + 1];
                SC[i][j] = SC[i][j + 1];
            }
    }
}

// Levels past the last whole chunk of 64, where they are few (the top level of
// 64 k + 1): a thread per node, so that they take no wave per column of their own.
template <typename T>
__device__ __forceinline__ void grad_tail(const GradArgs<T>& a, const T* __restrict__ tab, const T* __restrict__ wr,
                                          const T* __restrict__ p, T* __restrict__ u, int64_t t)
{
    const int n = a.nf, nr = a.nrf, nc = a.nc, nrc = a.nrc;
    const int64_t N = 10LL * n * n * nr;
    if (t >= 10LL * n * n * a.tail) return;
    const int r = nr - a.tail + (int)(t % a.tail);
    const int64_t lat = t / a.tail;
    const int y = (int)(lat % n), x = (int)((lat / n) % n), d = (int)(lat / ((int64_t)n * n));
    const int base = (r & 1) ? (r >> 1) : (r >> 1) - 1;
    const T* e = tab + lat * COUPLING_ENTRIES;
    T v[3] = {0, 0, 0};
#pragma unroll
    for (int dx = -1; dx <= 1; ++dx)
#pragma unroll
        for (int dy = -1; dy <= 1; ++dy) {
            const int cx = (x >> 1) + dx, cy = (y >> 1) + dy;
            if (!coupling_has(x & 1, y & 1, dx, dy) || cx < 0 || cy < 0 || cx >= nc || cy >= nc) continue;
            const T* pc = p + (((int64_t)d * nc + cx) * nc + cy) * nrc;
            T sa = T(0), sc = T(0);
            for (int q = 0; q < ((r & 1) ? 2 : 3); ++q) {
                if (base + q < 0 || base + q >= nrc) continue;
                sa += wr[q * nr + r] * pc[base + q];
                sc += wr[(3 + q) * nr + r] * pc[base + q];
            }
            const T* s = e + 6 * coupling_slot(x & 1, y & 1, dx, dy);
#pragma unroll
            for (int j = 0; j < 3; ++j) v[j] += s[j] * sa + s[3 + j] * sc;
        }
    mask_node(r == 0 ? a.bc_cmb : (r == nr - 1 ? a.bc_surf : (int)TN_NEUMANN), e + COUPLING_NORMAL, v);
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const int64_t i = j * N + lat * nr + r;
        u[i] = a.add ? u[i] + v[j] : v[j];
    }
}

template <typename T>
__global__ __launch_bounds__(256) void k_grad(GradArgs<T> a, const T* __restrict__ tab, const T* __restrict__ wr,
                                              const T* __restrict__ p, T* __restrict__ u)
{
    __shared__ alignas(16) T entries[4][2][COUPLING_ENTRIES];
    const int n = a.nf;
    if ((int)blockIdx.x < a.tail_blocks) return grad_tail<T>(a, tab, wr, p, u, (int64_t)blockIdx.x * 256 + threadIdx.x);
    const int pieces = (n + a.run - 1) / a.run, chunks = (a.nrf - a.tail + 63) >> 6;
    const int wave = threadIdx.x >> 6;
    // consecutive waves: chunks of a piece, pieces of a strip, strips of a diamond
    int w = __builtin_amdgcn_readfirstlane(
        xcd_tile(blockIdx.x - a.tail_blocks, gridDim.x - a.tail_blocks) * 4 + wave);
    if (w >= 10 * n * pieces * chunks) return;  // (no block barrier follows)
    const int rbase = 64 * (w % chunks);
    w /= chunks;
    const int y0 = (w % pieces) * a.run, y1 = min(n, y0 + a.run);
    w /= pieces;
    const int x = w % n, d = w / n;
    if (x & 1)
        grad_strip<T, 1>(a, tab, wr, p, u, entries[wave], d, x, y0, y1, rbase);
    else
        grad_strip<T, 0>(a, tab, wr, p, u, entries[wave], d, x, y0, y1, rbase);
}

// ---------------------------------------------------------------- B
// A wave takes `run` coarse columns of one X and walks the fine rows y below them:
// the five fine columns 2X - 2 .. 2X + 2 of a row add al . u and ga . u to the open
// sums of up to three coarse columns, per fine level (the lanes); the radial weights
// come last, once per coarse column, through the wave's own piece of LDS.  Velocity
// and table entries are loaded one row ahead.  The 64 fine levels from 60 c on give
// the coarse levels 30 c + 1 .. 30 c + 30, and level 0 where c = 0.  Up to 12 levels
// past the last window (one at 65 levels, five at 129) take lanes (fine column, level)
// of one more register each instead of a window of their own (65 levels: 57 us with a
// second register for all 64 lanes, 35 so).
constexpr int DIV_WINDOW = 30, DIV_EXTRA = 12;

template <typename T, bool FS>
struct DivWalk {
    struct Row {
        T u[5][3], ux[3], tab[5];
    };
    const T* tab;
    const T* u;
    T (*lds)[COUPLING_ENTRIES];
    int n, nr, d, X, lane;
    int64_t N;
    int r;
    bool in, slip;
    T sA[3], sC[3];  // coarse columns Y - 1, Y, Y + 1
    // the extra level of this lane: fine column xi, level rx; partial sums
    int xi, rx;
    bool extra, xin, xslip;  // (extra: wave-uniform)
    T xA[3], xC[3];

    __device__ __forceinline__ void load(int y, Row& v) const
    {
        y = min(y, n - 1);
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            const int x = min(max(2 * X - 2 + i, 0), n - 1);
            const int64_t la = __builtin_amdgcn_readfirstlane((d * n + x) * n + y);
            v.tab[i] = tab[la * COUPLING_ENTRIES + min(lane, COUPLING_ENTRIES - 1)];
#pragma unroll
            for (int j = 0; j < 3; ++j) v.u[i][j] = u[j * N + la * nr + r];
        }
        if (extra) {
            const int x = min(max(2 * X - 2 + xi, 0), n - 1);
#pragma unroll
            for (int j = 0; j < 3; ++j) v.ux[j] = u[j * N + ((int64_t)(d * n + x) * n + y) * nr + rx];
        }
    }
    __device__ __forceinline__ void mask(const T* e, bool sl, bool keep, T (&v)[3]) const
    {
        if constexpr (FS) {
            const T nx = e[COUPLING_NORMAL], ny = e[COUPLING_NORMAL + 1], nz = e[COUPLING_NORMAL + 2];
            const T vn = sl ? nx * v[0] + ny * v[1] + nz * v[2] : T(0);
            v[0] -= vn * nx;
            v[1] -= vn * ny;
            v[2] -= vn * nz;
        }
#pragma unroll
        for (int j = 0; j < 3; ++j) v[j] = keep ? v[j] : T(0);
    }
    template <int YO>
    __device__ __forceinline__ void row(Row& o)
    {
        __builtin_amdgcn_wave_barrier();
        if (lane < COUPLING_ENTRIES) {
#pragma unroll
            for (int i = 0; i < 5; ++i) lds[i][lane] = o.tab[i];
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            const int x = 2 * X - 2 + i, XO = i & 1, dx = 1 - (i >> 1);  // offset of X from x >> 1
            if (x < 0 || x >= n) continue;  // wave-uniform; the clamped column's load is unused
            const T* e = lds[i];
            T v[3] = {o.u[i][0], o.u[i][1], o.u[i][2]};
            mask(e, slip, in, v);
#pragma unroll
            for (int dy = -1; dy <= 1; ++dy) {
                if (!coupling_has(XO, YO, dx, dy)) continue;
                const T* s = e + 6 * coupling_slot(XO, YO, dx, dy);
                sA[dy + 1] += s[0] * v[0] + s[1] * v[1] + s[2] * v[2];
                sC[dy + 1] += s[3] * v[0] + s[4] * v[1] + s[5] * v[2];
            }
        }
        if (extra) {
            const T* e = lds[xi];
            mask(e, xslip, xin, o.ux);
#pragma unroll
            for (int dy = -1; dy <= 1; ++dy) {
                const bool has = coupling_has(xi & 1, YO, 1 - (xi >> 1), dy);
                const T* s = e + (has ? 6 * coupling_slot(xi & 1, YO, 1 - (xi >> 1), dy) : 0);
                const T dA = s[0] * o.ux[0] + s[1] * o.ux[1] + s[2] * o.ux[2];
                const T dC = s[3] * o.ux[0] + s[4] * o.ux[1] + s[5] * o.ux[2];
                xA[dy + 1] += has ? dA : T(0);
                xC[dy + 1] += has ? dC : T(0);
            }
        }
    }
};

// windows of a mesh of nr fine levels
__host__ __device__ constexpr int div_windows(int nr)
{
    return nr <= 64 + DIV_EXTRA ? 1 : (nr - 64 - DIV_EXTRA + 2 * DIV_WINDOW - 1) / (2 * DIV_WINDOW) + 1;
}

// coarse level Q takes the fine levels 2Q - 2 + i with the weights of slot ..
__device__ constexpr int DIV_SLOT[5] = {2, 1, 1, 0, 0};

template <typename T, bool FS>
__global__ __launch_bounds__(256) void k_div(DivArgs<T> a, const T* __restrict__ tab, const T* __restrict__ wr,
                                             const T* __restrict__ u, T* __restrict__ p)
{
    using Op = DivWalk<T, FS>;
    __shared__ T window[4][2][64 + DIV_EXTRA], partial[4][2][64];
    __shared__ alignas(16) T entries[4][5][COUPLING_ENTRIES];
    const int n = a.nf, nr = a.nrf, nc = a.nc, nrc = a.nrc;
    const int chunks = div_windows(nr), pieces = (nc + a.run - 1) / a.run;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // consecutive waves: strips of a diamond (neighbours share fine columns), chunks, pieces
    int w = __builtin_amdgcn_readfirstlane(xcd_tile(blockIdx.x, gridDim.x) * 4 + wave);
    if (w >= 10 * nc * pieces * chunks) return;  // (no block barrier follows)
    Op op;
    op.tab = tab;
    op.u = u;
    op.lds = entries[wave];
    op.lane = lane;
    op.n = n;
    op.nr = nr;
    op.N = 10LL * n * n * nr;
    op.X = w % nc;
    w /= nc;
    const int c = w % chunks, rbase = 2 * DIV_WINDOW * c;
    w /= chunks;
    const int y0 = (w % pieces) * a.run, y1 = min(nc, y0 + a.run);
    op.d = w / pieces;
    op.in = rbase + lane < nr;
    op.r = op.in ? rbase + lane : nr - 1;
    const int mode = op.r == 0 ? a.bc_cmb : (op.r == nr - 1 ? a.bc_surf : (int)TN_NEUMANN);
    op.slip = mode == TN_FREESLIP;
    if (mode == TN_DIRICHLET) op.in = false;
#pragma unroll
    for (int k = 0; k < 3; ++k) op.sA[k] = op.sC[k] = op.xA[k] = op.xC[k] = T(0);
    const int nx = c == chunks - 1 ? max(0, nr - rbase - 64) : 0;  // extra levels
    op.extra = nx > 0;
    op.xi = min(lane / max(nx, 1), 4);
    op.rx = min(rbase + 64 + lane % max(nx, 1), nr - 1);
    {
        const int x = 2 * op.X - 2 + op.xi;
        const int xmode = op.rx == nr - 1 ? a.bc_surf : (int)TN_NEUMANN;
        op.xslip = xmode == TN_FREESLIP;
        op.xin = lane < 5 * nx && x >= 0 && x < n && xmode != TN_DIRICHLET;
    }
    // the coarse level of this lane in the window, and its weights
    const int q = lane + (c > 0), Q = DIV_WINDOW * c + q;
    const bool out = Q < nrc && (q <= DIV_WINDOW || c == chunks - 1);
    T wA[5], wC[5];
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        const int rr = 2 * Q - 2 + i;
        const bool ok = out && rr >= 0 && rr < nr;
        wA[i] = ok ? wr[DIV_SLOT[i] * nr + rr] : T(0);
        wC[i] = ok ? wr[(3 + DIV_SLOT[i]) * nr + rr] : T(0);
    }
    T* pcol = p + ((int64_t)op.d * nc + op.X) * nc * a.nrc;
    auto store = [&](int Y) __attribute__((always_inline)) {
        window[wave][0][lane] = op.sA[0];
        window[wave][1][lane] = op.sC[0];
        if (op.extra) {
            partial[wave][0][lane] = op.xA[0];
            partial[wave][1][lane] = op.xC[0];
            __builtin_amdgcn_wave_barrier();
            if (lane < nx) {
                T ta = T(0), tc = T(0);
#pragma unroll
                for (int i = 0; i < 5; ++i) {
                    ta += partial[wave][0][lane + i * nx];
                    tc += partial[wave][1][lane + i * nx];
                }
                window[wave][0][64 + lane] = ta;
                window[wave][1][64 + lane] = tc;
            }
        }
        __builtin_amdgcn_wave_barrier();
        T v = T(0);
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            // (levels outside the mesh: weight 0 on a level the node does couple to)
            const int rr = min(max(2 * Q - 2 + i, 0), nr - 1) - rbase;
            const int k = min(max(rr, 0), 63 + nx);
            v += wA[i] * window[wave][0][k] + wC[i] * window[wave][1][k];
        }
        if (out) pcol[(int64_t)Y * a.nrc + Q] = v;
        __builtin_amdgcn_wave_barrier();
    };
    // rows 2Y (into Y - 1, Y, Y + 1) and 2Y + 1 (into Y, Y + 1); the run's first column
    // also takes the rows 2 y0 - 2 and 2 y0 - 1, its last one the row 2 y1
    typename Op::Row even, odd;
    int Y = max(0, y0 - 1);
    op.load(2 * Y, even);
#pragma unroll 1
    for (; Y < y1; ++Y) {
        op.load(2 * Y + 1, odd);
        op.template row<0>(even);
        if (Y - 1 >= y0) store(Y - 1);
        op.load(2 * Y + 2, even);
        if (2 * Y + 1 < n) op.template row<1>(odd);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            op.sA[k] = op.sA[k + 1];
            op.sC[k] = op.sC[k + 1];
            op.xA[k] = op.xA[k + 1];
            op.xC[k] = op.xC[k + 1];
        }
        op.sA[2] = op.sC[2] = op.xA[2] = op.xC[2] = T(0);
    }
    if (y1 < nc) op.template row<0>(even);
    store(y1 - 1);
}

// Columns per run: one round of resident waves, with runs of at most 8 (a run reads one
// or two columns more than it writes; B at 65 levels: 35 us in one round of runs of 6,
// 46 in runs of 5 that need a second round, 41 in runs of 8).
int coupling_run(int64_t columns, int waves_per_simd)
{
    const int64_t waves = 4LL * device_cus() * waves_per_simd;
    return (int)std::min<int64_t>(8, (columns + waves - 1) / waves);
}

}  // namespace

template <typename T>
void launch_coupling_tables(const double* coords, const double* radii, int n, int nr, T* lat, T* rad, hipStream_t s)
{
    const int64_t threads = 8 * 10LL * n * n;
    hipLaunchKernelGGL(k_coupling_table<T>, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, coords, n, lat);
    TN_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_coupling_radial<T>, dim3((unsigned)((nr + 255) / 256)), dim3(256), 0, s, radii, nr, rad);
    TN_HIP(hipGetLastError());
}

template <typename T>
void launch_div(const DivArgs<T>& a, hipStream_t s)
{
    TN_REQUIRE(a.nf == 2 * a.nc - 1 && a.nrf == 2 * a.nrc - 1 && a.nrc >= 2 && a.nc >= 2,
               "B: velocity mesh must be the pressure mesh refined once");
    TN_REQUIRE(a.tab && a.rad, "B: coupling tables missing");
    DivArgs<T> g = a;
    const int64_t chunks = div_windows(a.nrf);
    g.run = coupling_run(10LL * a.nc * a.nc * chunks, sizeof(T) == 8 ? 2 : 4);
    const int64_t waves = 10LL * a.nc * ((a.nc + g.run - 1) / g.run) * chunks;
    const bool fs = a.bc_cmb == TN_FREESLIP || a.bc_surf == TN_FREESLIP;
    hipLaunchKernelGGL(fs ? (k_div<T, true>) : (k_div<T, false>), dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, s, g,
                       g.tab, g.rad, g.u, g.p);
    TN_HIP(hipGetLastError());
}

template <typename T>
void launch_grad(const GradArgs<T>& a, hipStream_t s)
{
    TN_REQUIRE(a.nf == 2 * a.nc - 1 && a.nrf == 2 * a.nrc - 1 && a.nrc >= 2 && a.nc >= 2,
               "B^T: velocity mesh must be the pressure mesh refined once");
    TN_REQUIRE(a.tab && a.rad, "B^T: coupling tables missing");
    GradArgs<T> g = a;
    g.tail = a.nrf > 64 && (a.nrf & 63) <= TAIL ? a.nrf & 63 : 0;
    g.run = (coupling_run(10LL * a.nf * a.nf * ((a.nrf - g.tail + 63) >> 6), sizeof(T) == 8 ? 3 : 4) + 1) & ~1;
    g.tail_blocks = (int)((10LL * a.nf * a.nf * g.tail + 255) / 256);
    const int64_t waves = 10LL * a.nf * ((a.nf + g.run - 1) / g.run) * ((a.nrf - g.tail + 63) >> 6);
    hipLaunchKernelGGL(k_grad<T>, dim3((unsigned)(g.tail_blocks + (waves + 3) / 4)), dim3(256), 0, s, g, g.tab, g.rad,
                       g.p, g.u);
    TN_HIP(hipGetLastError());
}

#define TN_INST(T)                                                                                                  \
    template void launch_coupling_tables<T>(const double*, const double*, int, int, T*, T*, hipStream_t);         \
    template void launch_div<T>(const DivArgs<T>&, hipStream_t);                                                     \
    template void launch_grad<T>(const GradArgs<T>&, hipStream_t);
TN_INST(double)
TN_INST(float)
#undef TN_INST

}  // namespace tn
