// Mass operators on wedges: VectorMass (vector_mass.hpp:83-153), lumped KMass
// (kmass.hpp:97-185).
#include <algorithm>
#include <type_traits>

#include "tn_eps_march.hpp"
#include "tn_internal.hpp"
#include "tn_march.hpp"
#include "tn_reduce.hpp"
#include "tn_stokes.hpp"

namespace tn {
namespace {

// VectorMass as a gather: every node copy is written once, y_i = sum over the wedges
// of its diamond that contain it of (M_w x)_i; no atomics, so the result repeats bit
// for bit.  The
// reference's Felippa 3x2 rule factors into the 3-point triangle rule, exact for
// the lateral products (the P1 triangle mass (1 + delta_ij) / 24 times
// |det(V0, V1, V2)|), and the 2-point Gauss rule in zeta for rho^2 hat_a hat_b,
// which is not exact (degree 4) and is kept:
//   M_w[i][j] = |det_w| (1 + delta_ij) / 24 x h sum_{g = -+1/sqrt 3} rho(g)^2 hat_a(g) hat_b(g).
// Summed over the six wedges around a lateral node this is a 7-point lateral
// stencil (the node and its neighbours (x+-1, y), (x, y+-1), (x-1, y+1),
// (x+1, y-1)) times a 3-point radial stencil; |det_w| comes from the mesh's
// wedge table (geo[..][9]).
//
// Vectors: a thread per node.
template <typename T>
__global__ __launch_bounds__(256) void k_mass_stencil(MassArgs<T> a)
{
    const int n = a.n, nr = a.nr, nc = n - 1;
    const int64_t N = 10LL * n * n * nr;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= N) return;
    const int r = (int)(t % nr);
    const int y = (int)((t / nr) % n);
    const int x = (int)((t / ((int64_t)nr * n)) % n);
    const int d = (int)(t / ((int64_t)nr * n * n));
    auto det = [&](int qx, int qy, int w) -> double {
        if (qx < 0 || qy < 0 || qx >= nc || qy >= nc) return 0.0;
        return a.geo[((((int64_t)d * nc + qx) * nc + qy) * 2 + w) * GEO_STRIDE + 9];
    };
    // the six wedges around (x, y): quad (x, y) w0; (x-1, y) w0, w1; (x, y-1) w0, w1; (x-1, y-1) w1
    const double a0 = det(x, y, 0), b0 = det(x - 1, y, 0), b1 = det(x - 1, y, 1);
    const double c0 = det(x, y - 1, 0), c1 = det(x, y - 1, 1), d1 = det(x - 1, y - 1, 1);
    constexpr double s = 1.0 / 24.0;
    constexpr int NB = 7;
    const int ox[NB] = {0, 1, 0, -1, 0, -1, 1}, oy[NB] = {0, 0, 1, 0, -1, 1, -1};
    const double wl[NB] = {2.0 * s * (a0 + b0 + b1 + c0 + c1 + d1), s * (a0 + c1), s * (a0 + b1),
                           s * (b0 + d1),                          s * (c0 + d1), s * (b0 + b1), s * (c0 + c1)};
    // radial stencil: the node's own level and the levels below / above
    constexpr double g = 0.57735026918962584;  // 1/sqrt(3)
    constexpr double hm = 0.5 * (1.0 + g), hp = 0.5 * (1.0 - g);  // bottom hat at zeta = -g, +g
    double cm = 0.0, c0r = 0.0, cp = 0.0;
    if (r > 0) {  // layer (r-1, r): the node is its top level
        const double r1 = a.radii[r - 1], h = 0.5 * (a.radii[r] - r1);
        const double rm = r1 + h * (1.0 - g), rp = r1 + h * (1.0 + g);
        c0r += h * (rm * rm * hp * hp + rp * rp * hm * hm);
        cm = h * (rm * rm + rp * rp) * hm * hp;
    }
    if (r < nr - 1) {  // layer (r, r+1): the node is its bottom level
        const double r1 = a.radii[r], h = 0.5 * (a.radii[r + 1] - r1);
        const double rm = r1 + h * (1.0 - g), rp = r1 + h * (1.0 + g);
        c0r += h * (rm * rm * hm * hm + rp * rp * hp * hp);
        cp = h * (rm * rm + rp * rp) * hm * hp;
    }
    double acc[3] = {0, 0, 0};
#pragma unroll
    for (int k = 0; k < NB; ++k) {
        if (wl[k] == 0.0) continue;  // a neighbour outside the diamond (no wedge holds it)
        const int64_t col = (((int64_t)d * n + x + ox[k]) * n + y + oy[k]) * nr + r;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const T* xc = a.x + c * N + col;
            double v = c0r * (double)xc[0];
            if (r > 0) v += cm * (double)xc[-1];
            if (r < nr - 1) v += cp * (double)xc[1];
            acc[c] += wl[k] * v;
        }
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) a.y[c * N + t] = (T)acc[c];
}

// One component (the projection's CG): a wave walks an even
// run of consecutive radial columns, its lanes on 64 levels.  The radial weights
// stay in registers for the whole run, the lateral ones are wave-uniform, and the
// next column is loaded while one is summed.  A lane loads its own level and takes
// the two beside it from the neighbouring lanes, so a window of 64 levels gives the
// levels between its first and last (past 64 levels the windows overlap by two); with
// 21 loads per node instead of 7 the vector cache was what bound it.  With dot != null it also leaves the
// block's part of the sum over all node copies of x . y, which for x equal on a
// node's copies is the owned dot of x with the interface-summed y.
// With its part of the dot, FP64: level 7 x 129 314 us, level 6 x 65 44 us, level 5 x 33
// 11 us (13 without the determinants a column ahead); a thread per node, without the
// dot, 456, 58 and 13 us.
// lane i receives lane i-1's (UP) or i+1's value, 0 at the end
constexpr int LANE_UP = 0x138, LANE_DOWN = 0x130;  // DPP wave_shr:1, wave_shl:1
template <int CTRL>
__device__ __forceinline__ float lane_shift(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ __forceinline__ double lane_shift(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffLL), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}
constexpr int MASS_WAVES = 4;
template <typename T>
__global__ __launch_bounds__(64 * MASS_WAVES) void k_mass_columns(MassArgs<T> a)
{
    constexpr int NB = 7;
    const int n = a.n, nr = a.nr, nc = n - 1;
    const int nlat = 10 * n * n;
    const int lane = threadIdx.x & 63;
    const int waves = gridDim.x * MASS_WAVES;
    const int wave =
        __builtin_amdgcn_readfirstlane(xcd_tile(blockIdx.x, gridDim.x) * MASS_WAVES + (int)(threadIdx.x >> 6));
    const int lat0 = march::run_begin(nlat, wave, waves), lat1 = march::run_begin(nlat, wave + 1, waves);
    struct Col {
        T v[NB];        // the node's column and its six lateral neighbours
        double det[6];  // the six wedges around it
    };
    double sum = 0.0;
    for (int r0 = 0;; r0 += 62) {
        const int r = min(r0 + lane, nr - 1);
        const bool on = r0 + lane < nr && (lane > 0 || r0 == 0) && (lane < 63 || r == nr - 1);
        // column lat's values; neighbours and wedges outside the diamond count 0: not read
        auto load = [&](int lat, Col& q) {
            const int y = lat % n, x = (lat / n) % n, d = lat / (n * n);
            const int off[NB] = {0, n, 1, -n, -1, 1 - n, n - 1};
            const bool in[NB] = {true,  x < n - 1, y < n - 1, x > 0, y > 0, x > 0 && y < n - 1, x < n - 1 && y > 0};
#pragma unroll
            for (int k = 0; k < NB; ++k) q.v[k] = in[k] ? a.x[(int64_t)(lat + off[k]) * nr + r] : T(0);
            auto det = [&](int qx, int qy, int w) -> double {
                if (qx < 0 || qy < 0 || qx >= nc || qy >= nc) return 0.0;
                return a.geo[((((int64_t)d * nc + qx) * nc + qy) * 2 + w) * GEO_STRIDE + 9];
            };
            // quad (x, y) w0; (x-1, y) w0, w1; (x, y-1) w0, w1; (x-1, y-1) w1
            q.det[0] = det(x, y, 0);
            q.det[1] = det(x - 1, y, 0);
            q.det[2] = det(x - 1, y, 1);
            q.det[3] = det(x, y - 1, 0);
            q.det[4] = det(x, y - 1, 1);
            q.det[5] = det(x - 1, y - 1, 1);
        };
        const double ra = a.radii[r > 0 ? r - 1 : r], rb = a.radii[r], rc = a.radii[r < nr - 1 ? r + 1 : r];
        Col q[2];
        if (lat0 < lat1) load(lat0, q[0]);
        // radial stencil: the node's own level and the levels below / above
        constexpr double g = 0.57735026918962584;  // 1/sqrt(3)
        constexpr double hm = 0.5 * (1.0 + g), hp = 0.5 * (1.0 - g);  // bottom hat at zeta = -g, +g
        double cm = 0.0, c0r = 0.0, cp = 0.0;
        if (r > 0) {  // layer (r-1, r): the node is its top level
            const double r1 = ra, h = 0.5 * (rb - r1);
            const double rm = r1 + h * (1.0 - g), rp = r1 + h * (1.0 + g);
            c0r += h * (rm * rm * hp * hp + rp * rp * hm * hm);
            cm = h * (rm * rm + rp * rp) * hm * hp;
        }
        if (r < nr - 1) {  // layer (r, r+1): the node is its bottom level
            const double r1 = rb, h = 0.5 * (rc - r1);
            const double rm = r1 + h * (1.0 - g), rp = r1 + h * (1.0 + g);
            c0r += h * (rm * rm * hm * hm + rp * rp * hp * hp);
            cp = h * (rm * rm + rp * rp) * hm * hp;
        }
        auto finish = [&](int lat, const Col& q) {
            const double a0 = q.det[0], b0 = q.det[1], b1 = q.det[2], c0 = q.det[3], c1 = q.det[4], d1 = q.det[5];
            constexpr double s = 1.0 / 24.0;
            const double wl[NB] = {2.0 * s * (a0 + b0 + b1 + c0 + c1 + d1), s * (a0 + c1), s * (a0 + b1),
                                   s * (b0 + d1),                          s * (c0 + d1), s * (b0 + b1), s * (c0 + c1)};
            double acc = 0.0;
#pragma unroll
            for (int k = 0; k < NB; ++k) {
                const T vm = lane_shift<LANE_UP>(q.v[k]), vp = lane_shift<LANE_DOWN>(q.v[k]);
                const double v0 = r > 0 ? (double)vm : 0.0, v2 = r < nr - 1 ? (double)vp : 0.0;
                acc += wl[k] * (c0r * (double)q.v[k] + cm * v0 + cp * v2);
            }
            if (on) {
                a.y[(int64_t)lat * nr + r] = (T)acc;
                sum += (double)q.v[0] * acc;
            }
        };
        int lat = lat0;
        for (; lat + 1 < lat1; lat += 2) {
            load(lat + 1, q[1]);
            finish(lat, q[0]);
            if (lat + 2 < lat1) load(lat + 2, q[0]);
            finish(lat + 1, q[1]);
        }
        if (lat < lat1) finish(lat, q[0]);
        if (r0 + 64 >= nr) break;
    }
    if (a.dot) block_partial(sum, a.dot);
}

// Lumped k-weighted mass: row sums of the k-weighted wedge mass matrices in the
// reference's 6-point quadrature, a thread per node copy that adds the rows of the
// wedges of its diamond that contain it, in a fixed order.  In exact arithmetic this
// is the mass product above with the nodal k (sum_j N_j = 1), but it is the Schur
// diagonal of the solves, whose coarsest-level CG amplifies its last bits, so the
// quadrature's own sums are kept.  0.36 M pressure nodes: 426 us with the whole 6x6
// matrix per row in local arrays, 37 us with the row alone, its index a constant.
__device__ constexpr double Q6P[6][3] = {{0.6666666666666666, 0.1666666666666667, -0.5773502691896257},
                                        {0.1666666666666667, 0.6666666666666666, -0.5773502691896257},
                                        {0.1666666666666667, 0.1666666666666667, -0.5773502691896257},
                                        {0.6666666666666666, 0.1666666666666667, 0.5773502691896257},
                                        {0.1666666666666667, 0.6666666666666666, 0.5773502691896257},
                                        {0.1666666666666667, 0.1666666666666667, 0.5773502691896257}};
__device__ constexpr double Q6W = 0.1666666666666667;

__device__ constexpr double shape6(int q, int j)
{
    const double lat = j % 3 == 0 ? 1.0 - Q6P[q][0] - Q6P[q][1] : (j % 3 == 1 ? Q6P[q][0] : Q6P[q][1]);
    return lat * (j < 3 ? 0.5 * (1 - Q6P[q][2]) : 0.5 * (1 + Q6P[q][2]));
}

// row ROW of wedge W of quad (qx, qy), layer rc
template <typename T, int W, int ROW>
__device__ __forceinline__ double kmass_row(const double* __restrict__ coords, const double* __restrict__ radii,
                                            const T* __restrict__ k, int n, int nr, int d, int qx, int qy, int rc)
{
    constexpr int OFF[2][3][2] = {{{0, 0}, {1, 0}, {0, 1}}, {{1, 1}, {0, 1}, {1, 0}}};
    double P[3][3], kv[6];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int64_t lat = ((int64_t)d * n + qx + OFF[W][i][0]) * n + qy + OFF[W][i][1];
#pragma unroll
        for (int c = 0; c < 3; ++c) P[i][c] = coords[3 * lat + c];
        kv[i] = (double)k[lat * nr + rc];
        kv[i + 3] = (double)k[lat * nr + rc + 1];
    }
    const double r1 = radii[rc], r2 = radii[rc + 1], gr = 0.5 * (r2 - r1);
    double M[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        double J[3][3];  // lateral Jacobian (kernel_helpers.hpp:153-176)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            J[c][0] = P[1][c] - P[0][c];
            J[c][1] = P[2][c] - P[0][c];
            J[c][2] = (1 - Q6P[q][0] - Q6P[q][1]) * P[0][c] + Q6P[q][0] * P[1][c] + Q6P[q][1] * P[2][c];
        }
        const double det = fabs(J[0][0] * (J[1][1] * J[2][2] - J[1][2] * J[2][1]) -
                                J[0][1] * (J[1][0] * J[2][2] - J[1][2] * J[2][0]) +
                                J[0][2] * (J[1][0] * J[2][1] - J[1][1] * J[2][0]));
        const double rr = r1 + 0.5 * (r2 - r1) * (1 + Q6P[q][2]);
        double kq = 0.0;
#pragma unroll
        for (int j = 0; j < 6; ++j) kq += shape6(q, j) * kv[j];
        const double f = Q6W * kq * rr * rr * gr * det;
#pragma unroll
        for (int j = 0; j < 6; ++j) M[j] += f * shape6(q, ROW) * shape6(q, j);
    }
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < 6; ++j) s += M[j];
    return s;
}

template <typename T>
__global__ __launch_bounds__(256) void k_kmass_lumped(const double* __restrict__ coords, const double* __restrict__ radii,
                                                      const T* __restrict__ k, T* __restrict__ out, int n, int nr)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 10LL * n * n * nr) return;
    const int lat = (int)(t / nr), lev = (int)(t - (int64_t)lat * nr);
    const int Y = lat % n, X = (lat / n) % n, d = lat / (n * n), nc = n - 1;
    double acc = 0.0;
    // the six wedges around (X, Y) of layer rc: (X-1, Y-1) w1; (X-1, Y) w0, w1; (X, Y-1) w0, w1; (X, Y) w0
    auto layer = [&](int rc, auto top) {
        constexpr int B = decltype(top)::value ? 3 : 0;
        if (X > 0 && Y > 0) acc += kmass_row<T, 1, B>(coords, radii, k, n, nr, d, X - 1, Y - 1, rc);
        if (X > 0 && Y < nc) {
            acc += kmass_row<T, 0, B + 1>(coords, radii, k, n, nr, d, X - 1, Y, rc);
            acc += kmass_row<T, 1, B + 2>(coords, radii, k, n, nr, d, X - 1, Y, rc);
        }
        if (X < nc && Y > 0) {
            acc += kmass_row<T, 0, B + 2>(coords, radii, k, n, nr, d, X, Y - 1, rc);
            acc += kmass_row<T, 1, B + 1>(coords, radii, k, n, nr, d, X, Y - 1, rc);
        }
        if (X < nc && Y < nc) acc += kmass_row<T, 0, B>(coords, radii, k, n, nr, d, X, Y, rc);
    };
    if (lev > 0) layer(lev - 1, std::true_type{});
    if (lev < nr - 1) layer(lev, std::false_type{});
    out[t] = (T)acc;
}

}  // namespace

int mass_blocks(int n)
{
    // a wave per column on small meshes, runs of columns on large ones; 1024 blocks hold
    // every SIMD's four waves, and the users of the dot add up a partial sum per block
    const int nlat = 10 * n * n;
    return std::max(1, std::min((nlat + MASS_WAVES - 1) / MASS_WAVES, REDUCE_MAX_BLOCKS / 2));
}

template <typename T>
void launch_mass(const MassArgs<T>& a, hipStream_t s)
{
    TN_REQUIRE(a.ncomp == 1 || (a.ncomp == 3 && !a.dot), "mass: ncomp must be 1, or 3 without the dot");
    TN_REQUIRE(a.geo, "mass: wedge table missing");
    const int64_t N = 10LL * a.n * a.n * a.nr;
    if (a.ncomp == 3)
        hipLaunchKernelGGL((k_mass_stencil<T>), dim3((unsigned)((N + 255) / 256)), dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((k_mass_columns<T>), dim3((unsigned)mass_blocks(a.n)), dim3(64 * MASS_WAVES), 0, s, a);
    TN_HIP(hipGetLastError());
}

template <typename T>
void launch_kmass_lumped(const double* coords, const double* radii, int n, int nr, const T* k, T* out, hipStream_t s)
{
    const int64_t N = 10LL * n * n * nr;
    hipLaunchKernelGGL((k_kmass_lumped<T>), dim3((unsigned)((N + 255) / 256)), dim3(256), 0, s, coords, radii, k, out, n,
                       nr);
    TN_HIP(hipGetLastError());
}
template void launch_kmass_lumped<double>(const double*, const double*, int, int, const double*, double*, hipStream_t);
template void launch_kmass_lumped<float>(const double*, const double*, int, int, const float*, float*, hipStream_t);

template void launch_mass<double>(const MassArgs<double>&, hipStream_t);
template void launch_mass<float>(const MassArgs<float>&, hipStream_t);

}  // namespace tn
