// Conjugate gradients on a small stored-matrix operator in one workgroup: the
// multigrid's coarsest-level solve (pcg.hpp:78-153 without preconditioner).
//
// On the coarsest level (80 to 640 cells) an iteration by separate launches is six
// kernels of 2 to 14 us, each waiting for memory with an almost empty chip: 34 us an
// iteration at lateral level 1 x 3 radial nodes, 136 with a host wait per reduction.
// Here one workgroup of 8 waves runs the whole solve: the search direction and the
// cells' corner sums live in LDS, a thread's node copies (x, r, p, A p) in registers,
// the matrices stream from the XCD's L2 (220 KB at level 1, 1.8 MB at level 2) with 16
// or 8 loads in flight per lane, and a reduction is two barriers.  Measured per
// iteration (FP64, no-slip; the wall time of 50 iterations less that of 10): 7.8 us at
// level 1 x 3, 21 us at 1 x 9, 28 us at level 2 x 5, where the one CU's L2 bandwidth
// binds.  Past the sizes that fit (coarse_cg_fits) the queued launches are used; they
// fill the chip.
//
// The operator is the stored apply's (kernels_mg.hip): trial side on the boundary
// levels, cells, gather, test side from the boundary-node forms, fs/fs penalty,
// interface sum.  Every sum -- products, gather, copies, penalty moment, dots -- is
// formed in the order of the separate launches, so a solve has their bits: this CG
// stops at a loose tolerance on an ill-conditioned operator, and roundings in another
// order moved a two-level Stokes step's velocity by up to 5e-7.
#include "tn_coarse_cg.hpp"
#include "tn_reduce.hpp"

namespace tn {
namespace {

constexpr int THREADS = 512, WAVES = THREADS / 64;

template <typename S>
struct Vec16;
template <>
struct Vec16<float> {
    using type = float4;
    static __device__ float get(const float4& v, int i) { return i == 0 ? v.x : (i == 1 ? v.y : (i == 2 ? v.z : v.w)); }
};
template <>
struct Vec16<double> {
    using type = double2;
    static __device__ double get(const double2& v, int i) { return i == 0 ? v.x : v.y; }
};

// lane i receives lane i + N's value, within rows of 16 lanes
template <int N>
__device__ __forceinline__ double row_down(double v)
{
    constexpr int CTRL = 0x100 + N;  // DPP row_shl:N
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffLL), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

// The sum over `ncol` columns' values in LDS (NV fields, `stride` apart), the same
// bits in every thread and those of a reduction over the whole chip: blocks of four
// columns, then the blocks' sums over the 256 threads of a finalize, each a wave's
// butterfly.  The values must be in place and the last call's be read: two barriers.
template <int NV>
__device__ __forceinline__ void columns_total(const double* col, int ncol, int stride, double (*red)[NV], double (&out)[NV])
{
    const int tid = threadIdx.x;
    __syncthreads();
    if (tid < 256) {
#pragma unroll
        for (int f = 0; f < NV; ++f) {
            double s = 0.0;
            for (int c = 4 * tid; c < ncol; c += 1024) {
                const double* v = col + f * stride + c;
                const double v1 = c + 1 < ncol ? v[1] : 0.0, v2 = c + 2 < ncol ? v[2] : 0.0, v3 = c + 3 < ncol ? v[3] : 0.0;
                s += (v[0] + v2) + (v1 + v3);
            }
            s = wave_sum(s);
            if ((tid & 63) == 0) red[tid >> 6][f] = s;
        }
    }
    __syncthreads();
#pragma unroll
    for (int f = 0; f < NV; ++f) out[f] = (red[0][f] + red[2][f]) + (red[1][f] + red[3][f]);
}

// NPT: node copies per thread (1 on the smallest levels, whose matrices' loads then
// find registers; 4 up to COARSE_CG_NODES).  A column's copies take `1 << lg` adjacent
// lanes, at least its levels.
template <typename T, typename S, int NPT, bool PEN>
__global__ __launch_bounds__(THREADS) void k_coarse_cg(CoarseCgArgs<T, S> g)
{
    constexpr int PD = NPT == 1 ? 16 : 8;  // 16-byte matrix vectors in flight per lane
    const StoredArgs<T, S>& a = g.op;
    __shared__ __align__(16) unsigned char raw[COARSE_CG_LDS];
    __shared__ double red3[4][3], red1[4][1];
    const int n = a.n, nr = a.nr, ncl = n - 1, ncr = nr - 1, nlat = 10 * n * n;
    const int N = nlat * nr, cells = 10 * ncl * ncl * ncr;
    T* pt = reinterpret_cast<T*>(raw);  // [3][N] search direction after the trial rule; between products a reduction's columns
    T* cs = pt + 3 * N;                 // [24][cells] corner sums, then [3][N] the copies' A p
    double* col = reinterpret_cast<double*>(raw);  // [3][nlat]
    // (opaque again in every iteration: else the addresses of all copies' corners are
    // kept, and spilled, across the whole solve)
    int tid = threadIdx.x;
    const int lg = g.lanes_log2;

    // this thread's node copies (x stays in memory: it is read and written once per iteration)
    T r[NPT][3], p[NPT][3], ap[NPT][3];
    unsigned owned = 0;  // bit k: copy k is its node's owned one
    auto lat_of = [&](int k) { return (tid + k * THREADS) >> lg; };
    const int lev = threadIdx.x & ((1 << lg) - 1);  // (THREADS is a multiple of the lanes)
    auto has = [&](int k) { return lev < nr && lat_of(k) < nlat; };
#pragma unroll
    for (int k = 0; k < NPT; ++k) {
        const bool on = has(k);
        const int lat = on ? lat_of(k) : 0, j = lat * nr + lev;
        owned |= on && g.owned_lat[lat] ? 1u << k : 0u;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            r[k][c] = on ? g.b[c * N + j] : T(0);
            p[k][c] = g.zero ? r[k][c] : (on ? g.x[c * N + j] : T(0));
            if (g.zero && on) g.x[c * N + j] = T(0);
        }
    }
    // the sums of v[f] over each column's levels into col[f][lat], in a butterfly's order
    auto columns = [&](int k, const double (&v)[3]) {
#pragma unroll
        for (int f = 0; f < 3; ++f) {
            double s = v[f];
            if (lg > 4) s += __shfl_xor(s, 16, 64);
            if (lg > 3) s += row_down<8>(s);
            if (lg > 2) s += row_down<4>(s);
            s += row_down<2>(s);
            s += row_down<1>(s);
            if (lev == 0 && lat_of(k) < nlat) col[f * nlat + lat_of(k)] = s;
        }
    };
    auto mode_of = [&](int lev) { return lev == 0 ? a.bc_cmb : (lev == ncr ? a.bc_surf : (int)TN_NEUMANN); };

    // ap = A p (p equal on a node's copies)
    auto apply = [&]() {
        double gam[3] = {0, 0, 0};
        if constexpr (PEN) {
#pragma unroll
            for (int k = 0; k < NPT; ++k) {
                double m[3] = {0.0, 0.0, 0.0};
                if (owned >> k & 1) {
                    const int lat = lat_of(k);
                    const double rr = a.radii[lev];
                    const double px = a.coords[3 * lat] * rr, py = a.coords[3 * lat + 1] * rr,
                                 pz = a.coords[3 * lat + 2] * rr;
                    const double ax = p[k][0], ay = p[k][1], az = p[k][2];
                    m[0] += py * az - pz * ay;
                    m[1] += pz * ax - px * az;
                    m[2] += px * ay - py * ax;
                }
                columns(k, m);
            }
            double bk[3];
            columns_total<3>(col, nlat, nlat, red3, bk);
            const double* Sm = a.pen + 4;
            for (int i = 0; i < 3; ++i) gam[i] = Sm[3 * i] * bk[0] + Sm[3 * i + 1] * bk[1] + Sm[3 * i + 2] * bk[2];
        }
#pragma unroll
        for (int k = 0; k < NPT; ++k) {
            if (!has(k)) continue;
            const int lat = lat_of(k), j = lat * nr + lev, mode = mode_of(lev);
            T v[3] = {p[k][0], p[k][1], p[k][2]};
            if (mode == TN_DIRICHLET) {
                v[0] = v[1] = v[2] = T(0);
            } else if (mode == TN_FREESLIP) {
                const T nx = (T)a.coords[3 * lat], ny = (T)a.coords[3 * lat + 1], nz = (T)a.coords[3 * lat + 2];
                const T un = nx * v[0] + ny * v[1] + nz * v[2];
                v[0] -= un * nx;
                v[1] -= un * ny;
                v[2] -= un * nz;
            }
#pragma unroll
            for (int c = 0; c < 3; ++c) pt[c * N + j] = v[c];
        }
        __syncthreads();
        // cells: both wedges' products into the 8 corner sums (corner k: bottom, top)
        for (int cell = tid; cell < cells; cell += THREADS) {
            constexpr int WC[2][3] = {{0, 1, 2}, {3, 2, 1}};
            const int rc = cell % ncr, col = cell / ncr;
            const int y = col % ncl, xq = (col / ncl) % ncl, d = col / (ncl * ncl);
            const int l00 = (d * n + xq) * n + y;
            const int latc[4] = {l00, l00 + n, l00 + 1, l00 + n + 1};
            T y8[8][3];
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int c = 0; c < 3; ++c) y8[i][c] = T(0);
#pragma unroll
            for (int w = 0; w < 2; ++w) {
                T xs[18];
#pragma unroll
                for (int i = 0; i < 6; ++i)
#pragma unroll
                    for (int c = 0; c < 3; ++c) xs[c * 6 + i] = pt[c * N + latc[WC[w][i % 3]] * nr + rc + (i >= 3)];
                constexpr int V = stored_vec<S>(), NV = WEDGE_SLOTS / V;
                using Vec = typename Vec16<S>::type;
                const Vec* vp = reinterpret_cast<const Vec*>(a.stored + stored_at<S>(cell, w, 0));
                Vec buf[NV];
#pragma unroll
                for (int q = 0; q < PD; ++q) buf[q] = vp[q * 64];
                int e = 0;
#pragma unroll
                for (int i = 0; i < 18; ++i) {
#pragma unroll
                    for (int j = i; j < 18; ++j, ++e) {
                        if (e % V == 0 && e / V + PD < NV) buf[e / V + PD] = vp[(e / V + PD) * 64];
                        const T aij = (T)Vec16<S>::get(buf[e / V], e % V);
                        const int ni = i % 6, nj = j % 6;
                        y8[WC[w][ni % 3] + (ni >= 3 ? 4 : 0)][i / 6] += aij * xs[j];
                        if (j != i) y8[WC[w][nj % 3] + (nj >= 3 ? 4 : 0)][j / 6] += aij * xs[i];
                    }
                }
                // (keeps the second wedge's loads behind the first one's arithmetic)
                asm volatile("" ::: "memory");
            }
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int c = 0; c < 3; ++c) cs[(i * 3 + c) * cells + cell] = y8[i][c];
        }
        __syncthreads();
        // node copies: the up to four quads' bottom and top sums, then the test side (into ap)
#pragma unroll
        for (int k = 0; k < NPT; ++k) {
            T part[3] = {T(0), T(0), T(0)};
            if (has(k)) {
                const int lat = lat_of(k), mode = mode_of(lev);
                const int Y = lat % n, X = (lat / n) % n, d = lat / (n * n);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int qx = X - (q & 1), qy = Y - (q >> 1);
                    if (qx < 0 || qy < 0 || qx >= ncl || qy >= ncl) continue;
                    const int cell = ((d * ncl + qx) * ncl + qy) * ncr + lev;
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        const T below = lev > 0 ? cs[((q + 4) * 3 + c) * cells + cell - 1] : T(0);
                        part[c] += lev < ncr ? cs[(q * 3 + c) * cells + cell] + below : below;
                    }
                }
                if (mode != TN_NEUMANN) {
                    const T* bk = a.blk + ((lev == 0 ? 0 : 10 * n * n) + lat) * 3;
                    if (mode == TN_DIRICHLET) {
#pragma unroll
                        for (int c = 0; c < 3; ++c) part[c] = bk[c] * p[k][c];
                    } else {
                        const T nx = (T)a.coords[3 * lat], ny = (T)a.coords[3 * lat + 1], nz = (T)a.coords[3 * lat + 2];
                        const T corr = bk[0] * (nx * p[k][0] + ny * p[k][1] + nz * p[k][2]) -
                                       (nx * part[0] + ny * part[1] + nz * part[2]);
                        part[0] += corr * nx;
                        part[1] += corr * ny;
                        part[2] += corr * nz;
                    }
                }
                if constexpr (PEN) {
                    const double rr = a.radii[lev];
                    const double px = a.pen_coords[3 * lat] * rr, py = a.pen_coords[3 * lat + 1] * rr,
                                 pz = a.pen_coords[3 * lat + 2] * rr;
                    part[0] += (T)(gam[1] * pz - gam[2] * py);
                    part[1] += (T)(gam[2] * px - gam[0] * pz);
                    part[2] += (T)(gam[0] * py - gam[1] * px);
                }
            }
#pragma unroll
            for (int c = 0; c < 3; ++c) ap[k][c] = part[c];
        }
        __syncthreads();  // the corner sums are read: their space takes the copies' sums
#pragma unroll
        for (int k = 0; k < NPT; ++k) {
            if (has(k))
#pragma unroll
                for (int c = 0; c < 3; ++c) cs[c * N + lat_of(k) * nr + lev] = ap[k][c];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < NPT; ++k) {
            const int grp = has(k) ? g.group_of[lat_of(k)] : -1;
            if (grp < 0) continue;  // no other copies: ap holds the sum
            double s[3] = {0.0, 0.0, 0.0};
#pragma unroll 1
            for (int m = 0; m < MeshLevel::GRP_PAD; ++m) {
                const int q = g.groups[MeshLevel::GRP_PAD * grp + m];
                if (q < 0) break;
#pragma unroll
                for (int c = 0; c < 3; ++c) s[c] += (double)cs[c * N + q * nr + lev];
            }
#pragma unroll
            for (int c = 0; c < 3; ++c) ap[k][c] = (T)s[c];
        }
        // (the next use of raw is a reduction's columns, in pt, with a barrier before cs is written)
    };
    // a dot is a sum over the columns of all three components, one after the other
    auto dot = [&](const T(&u)[NPT][3], const T(&v)[NPT][3]) {
#pragma unroll
        for (int k = 0; k < NPT; ++k) {
            double s[3];
#pragma unroll
            for (int c = 0; c < 3; ++c) s[c] = owned >> k & 1 ? (double)u[k][c] * (double)v[k][c] : 0.0;
            columns(k, s);
        }
        double t[1];
        columns_total<1>(col, 3 * nlat, 0, red1, t);
        return t[0];
    };

    // iteration 0 (a given start only): r = b - A x with x in p, then p = r
    double rr = 0.0, r0 = 0.0;
    if (g.zero) {
        rr = dot(r, r);
        r0 = sqrt(rr);
        if (r0 < g.atol) return;
    }
    for (int it = g.zero ? 1 : 0; it <= g.max_iterations; ++it) {
        if constexpr (NPT > 1 || PEN) asm volatile("" : "+v"(tid));
        apply();
        const T alpha = it == 0 ? T(1) : (T)(rr / dot(ap, p));
#pragma unroll
        for (int k = 0; k < NPT; ++k) {
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                if (it > 0 && has(k)) g.x[c * N + lat_of(k) * nr + lev] += alpha * p[k][c];
                r[k][c] -= alpha * ap[k][c];
            }
        }
        const double rn = dot(r, r);
        const double res = sqrt(rn);
        if (it == 0) {
            r0 = res;
            if (r0 < g.atol) return;
        } else if (res / r0 <= g.rtol || res < g.atol) {
            return;
        }
        const T beta = it == 0 ? T(0) : (T)(rn / rr);
        rr = rn;
#pragma unroll
        for (int k = 0; k < NPT; ++k)
#pragma unroll
            for (int c = 0; c < 3; ++c) p[k][c] = it == 0 ? r[k][c] : r[k][c] + beta * p[k][c];
    }
}

}  // namespace

// lanes of a column: a power of two, its levels at least
static int lanes_log2(int nr)
{
    int lg = 2;
    while ((1 << lg) < nr) ++lg;
    return lg;
}

bool coarse_cg_fits(int n, int nr, int esize)
{
    const int64_t nlat = 10LL * n * n, N = nlat * nr, cells = 10LL * (n - 1) * (n - 1) * (nr - 1);
    return nr >= 3 && nr <= 32 && (nlat << lanes_log2(nr)) <= COARSE_CG_NODES &&
           (3 * N + std::max<int64_t>(24 * cells, 3 * N)) * esize <= COARSE_CG_LDS;
}

template <typename T, typename S>
void launch_coarse_cg(CoarseCgArgs<T, S> g, hipStream_t s)
{
    TN_REQUIRE(coarse_cg_fits(g.op.n, g.op.nr, (int)sizeof(T)), "coarse CG: operator too large for one workgroup");
    TN_REQUIRE(g.op.blk || (g.op.bc_cmb == TN_NEUMANN && g.op.bc_surf == TN_NEUMANN), "coarse CG: no boundary forms");
    g.lanes_log2 = lanes_log2(g.op.nr);
    const bool one = (10 * g.op.n * g.op.n) << g.lanes_log2 <= THREADS;
    constexpr int MOST = COARSE_CG_NODES / THREADS;
    auto kernel = g.op.pen ? (one ? k_coarse_cg<T, S, 1, true> : k_coarse_cg<T, S, MOST, true>)
                           : (one ? k_coarse_cg<T, S, 1, false> : k_coarse_cg<T, S, MOST, false>);
    hipLaunchKernelGGL(kernel, dim3(1), dim3(THREADS), 0, s, g);
    TN_HIP(hipGetLastError());
}
template void launch_coarse_cg<double, double>(CoarseCgArgs<double, double>, hipStream_t);
template void launch_coarse_cg<double, float>(CoarseCgArgs<double, float>, hipStream_t);
template void launch_coarse_cg<float, float>(CoarseCgArgs<float, float>, hipStream_t);
template void launch_coarse_cg<float, double>(CoarseCgArgs<float, double>, hipStream_t);

}  // namespace tn
