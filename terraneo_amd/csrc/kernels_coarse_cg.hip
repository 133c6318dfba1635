// Conjugate gradients on a small stored-matrix operator in one workgroup: the
// multigrid's coarsest-level solve (pcg.hpp:78-153 without preconditioner).
//
// On the coarsest level (80 to 640 cells) an iteration by separate launches is six
// kernels of 2 to 14 us, each waiting for memory with an almost empty chip: 34 us an
// iteration at lateral level 1 x 3 radial nodes.  Here one workgroup of 8 waves
// runs the whole solve: the search direction and the cells' corner sums live in
// LDS, a thread's node copies (x, r, p, A p) in registers, the matrices stream from
// the XCD's L2 (220 KB at level 1, 1.8 MB at level 2) with 16 or 8 loads in flight
// per lane, and a reduction is one barrier.  Measured per iteration: 9 us at level
// 1 x 3, 29 us at level 2 x 5, where the one CU's L2 bandwidth binds.  Past the
// sizes that fit (coarse_cg_fits) the queued launches are used; they fill the chip.
//
// The operator is the stored apply's (kernels_mg.hip): trial side on the boundary
// levels, cells, gather, test side from the boundary-node forms, fs/fs penalty,
// interface sum; sums run in a fixed order, so a solve repeats bit for bit.
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

// Sum over the block, the same bits in every thread; `slot` alternates between
// calls, so one barrier per call suffices.
struct BlockSum {
    double (*buf)[WAVES];
    int slot = 0;
    __device__ double operator()(double v)
    {
        v = wave_sum(v);
        const int lane = threadIdx.x & 63;
        if (lane == 0) buf[slot][threadIdx.x >> 6] = v;
        __syncthreads();
        const double t = wave_sum(lane < WAVES ? buf[slot][lane] : 0.0);
        slot = slot == 3 ? 0 : slot + 1;
        return t;
    }
};

// NPT: node copies per thread (1 on the smallest levels, whose matrices' loads then
// find registers; 4 up to COARSE_CG_NODES)
template <typename T, typename S, int NPT>
__global__ __launch_bounds__(THREADS) void k_coarse_cg(CoarseCgArgs<T, S> g)
{
    constexpr int PD = NPT == 1 ? 16 : 8;  // 16-byte matrix vectors in flight per lane
    const StoredArgs<T, S>& a = g.op;
    __shared__ __align__(16) unsigned char raw[COARSE_CG_LDS];
    __shared__ double red[4][WAVES];
    const int n = a.n, nr = a.nr, ncl = n - 1, ncr = nr - 1;
    const int N = 10 * n * n * nr, cells = 10 * ncl * ncl * ncr;
    T* pt = reinterpret_cast<T*>(raw);  // [3][N] search direction after the trial rule
    T* cs = pt + 3 * N;                 // [24][cells] corner sums, then [3][N] the copies' A p
    const int tid = threadIdx.x;
    BlockSum sum{red};

    // this thread's node copies (x stays in memory: it is read and written once per iteration)
    T r[NPT][3], p[NPT][3], ap[NPT][3];
    bool own[NPT];
#pragma unroll
    for (int k = 0; k < NPT; ++k) {
        const int j = tid + k * THREADS;
        const bool on = j < N;
        own[k] = on && g.owned_lat[on ? j / nr : 0];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            r[k][c] = on ? g.b[c * N + j] : T(0);
            p[k][c] = g.zero ? r[k][c] : (on ? g.x[c * N + j] : T(0));
            if (g.zero && on) g.x[c * N + j] = T(0);
        }
    }
    auto mode_of = [&](int lev) { return lev == 0 ? a.bc_cmb : (lev == ncr ? a.bc_surf : (int)TN_NEUMANN); };

    // ap = A p (p equal on a node's copies)
    auto apply = [&]() {
        double gam[3] = {0, 0, 0};
        if (a.pen) {
            double m0 = 0, m1 = 0, m2 = 0;
#pragma unroll
            for (int k = 0; k < NPT; ++k) {
                const int j = tid + k * THREADS;
                if (own[k]) {
                    const int lat = j / nr;
                    const double rr = a.radii[j - lat * nr];
                    const double px = a.coords[3 * lat] * rr, py = a.coords[3 * lat + 1] * rr,
                                 pz = a.coords[3 * lat + 2] * rr;
                    m0 += py * (double)p[k][2] - pz * (double)p[k][1];
                    m1 += pz * (double)p[k][0] - px * (double)p[k][2];
                    m2 += px * (double)p[k][1] - py * (double)p[k][0];
                }
            }
            m0 = sum(m0);
            m1 = sum(m1);
            m2 = sum(m2);
            const double* Sm = a.pen + 4;
            for (int i = 0; i < 3; ++i) gam[i] = Sm[3 * i] * m0 + Sm[3 * i + 1] * m1 + Sm[3 * i + 2] * m2;
        }
#pragma unroll
        for (int k = 0; k < NPT; ++k) {
            const int j = tid + k * THREADS;
            if (j >= N) continue;
            const int lat = j / nr, mode = mode_of(j - lat * nr);
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
            const int j = tid + k * THREADS;
            T part[3] = {T(0), T(0), T(0)};
            if (j < N) {
                const int lat = j / nr, lev = j - lat * nr, mode = mode_of(lev);
                const int Y = lat % n, X = (lat / n) % n, d = lat / (n * n);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int qx = X - (q & 1), qy = Y - (q >> 1);
                    if (qx < 0 || qy < 0 || qx >= ncl || qy >= ncl) continue;
                    const int cell = ((d * ncl + qx) * ncl + qy) * ncr + lev;
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        if (lev < ncr) part[c] += cs[(q * 3 + c) * cells + cell];
                        if (lev > 0) part[c] += cs[((q + 4) * 3 + c) * cells + cell - 1];
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
                if (a.pen) {
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
            const int j = tid + k * THREADS;
            if (j < N)
#pragma unroll
                for (int c = 0; c < 3; ++c) cs[c * N + j] = ap[k][c];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < NPT; ++k) {
            const int j = tid + k * THREADS;
            const int lat = j < N ? j / nr : 0, lev = j - lat * nr;
            const int grp = j < N ? g.group_of[lat] : -1;
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
        // (the next apply writes pt first and reaches a barrier before the corner sums)
    };
    auto dot = [&](const T(&u)[NPT][3], const T(&v)[NPT][3]) {
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < NPT; ++k)
            if (own[k])
#pragma unroll
                for (int c = 0; c < 3; ++c) s += (double)u[k][c] * (double)v[k][c];
        return sum(s);
    };

    // iteration 0 (a given start only): r = b - A x with x in p, then p = r
    double rr = 0.0, r0 = 0.0;
    if (g.zero) {
        rr = dot(r, r);
        r0 = sqrt(rr);
        if (r0 < g.atol) return;
    }
    for (int it = g.zero ? 1 : 0; it <= g.max_iterations; ++it) {
        apply();
        const T alpha = it == 0 ? T(1) : (T)(rr / dot(ap, p));
#pragma unroll
        for (int k = 0; k < NPT; ++k) {
            const int j = tid + k * THREADS;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                if (it > 0 && j < N) g.x[c * N + j] += alpha * p[k][c];
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

bool coarse_cg_fits(int n, int nr, int esize)
{
    const int64_t N = 10LL * n * n * nr, cells = 10LL * (n - 1) * (n - 1) * (nr - 1);
    return N <= COARSE_CG_NODES && nr >= 3 &&
           (3 * N + std::max<int64_t>(24 * cells, 3 * N)) * esize <= COARSE_CG_LDS;
}

template <typename T, typename S>
void launch_coarse_cg(const CoarseCgArgs<T, S>& g, hipStream_t s)
{
    TN_REQUIRE(coarse_cg_fits(g.op.n, g.op.nr, (int)sizeof(T)), "coarse CG: operator too large for one workgroup");
    TN_REQUIRE(g.op.blk || (g.op.bc_cmb == TN_NEUMANN && g.op.bc_surf == TN_NEUMANN), "coarse CG: no boundary forms");
    if (10 * g.op.n * g.op.n * g.op.nr <= THREADS)
        hipLaunchKernelGGL((k_coarse_cg<T, S, 1>), dim3(1), dim3(THREADS), 0, s, g);
    else
        hipLaunchKernelGGL((k_coarse_cg<T, S, COARSE_CG_NODES / THREADS>), dim3(1), dim3(THREADS), 0, s, g);
    TN_HIP(hipGetLastError());
}
template void launch_coarse_cg<double, double>(const CoarseCgArgs<double, double>&, hipStream_t);
template void launch_coarse_cg<double, float>(const CoarseCgArgs<double, float>&, hipStream_t);
template void launch_coarse_cg<float, float>(const CoarseCgArgs<float, float>&, hipStream_t);
template void launch_coarse_cg<float, double>(const CoarseCgArgs<float, double>&, hipStream_t);

}  // namespace tn
