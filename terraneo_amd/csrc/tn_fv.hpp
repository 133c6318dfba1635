// Hex finite-volume energy step (FCT advection-diffusion): argument block,
// launchers and the state object behind tn_fv.
#pragma once

#include "tn_internal.hpp"

namespace tn {

struct FvArgs {
    const double* coords;   // [10][n][n][3] unit lateral positions
    const double* radii;    // [nr]
    const double* columns;  // [10][n-1][n-1][FV_COLUMN] lateral geometry of each hex column
    const double* layers;   // [nr+1] radial part of the cell centres (ghost layers at the shells: 0)
    int n, nr;
};

// Per hex column (d, x, y).  A cell centre is s(layer) c(column) and a lateral
// face vector a radial factor times the column's normal N, so orientation and
// diffusion split into a column and a layer part:
//   [0, 12)  the four lateral face normals, oriented towards the neighbour's centre
//   [12, 18) the two triangles' (V1 - V0) x (V2 - V0)
//   [18]     the sum of the two wedges' |det(V0, V1, V2)|
//   [19]     sign of a = (n0 + n1) . c   (radial faces)
//   [20, 24) |N|^2 / |N . (c_neighbour - c)| of the lateral faces
//   [24]     |n0 + n1|^2 / |a|
//   [25]     pad (rows of 208 bytes, 16-byte aligned)
constexpr int FV_COLUMN = 26;

int64_t fv_real_cells(int n, int nr);
int64_t fv_size(int n, int nr);  // FV scalar elements, ghost layers included
int fv_dt_blocks(int n, int nr);

void launch_fv_centers(const FvArgs& a, double* c, hipStream_t s);
// centroids: [10][n+1][n+1][3], the column parts c of the cell centres; real
// columns written, the lateral ghosts to be exchanged (launch_fv_ghost_columns)
// before launch_fv_columns
void launch_fv_centroids(const FvArgs& a, double* centroids, hipStream_t s);
void launch_fv_ghost_columns(const int32_t* pairs, int cnt, double* centroids, hipStream_t s);
void launch_fv_columns(const FvArgs& a, const double* centroids, double* columns, hipStream_t s);
// pairs[k] = (ghost lateral index, source lateral index), lateral index (d (n+1) + x) (n+1) + y
void launch_fv_ghost(const int32_t* pairs, int cnt, int nr, int ncomp, double* f, hipStream_t s);
void launch_fv_ghost2(const int32_t* pairs, int cnt, int nr, double* f, double* g, hipStream_t s);
void launch_fv_dt(const FvArgs& a, const double* vel, double kappa, double* part, double* out, hipStream_t s);
// Values on the shells that the predictor writes into T_L itself (the real
// boundary cell and the ghost beyond), and where it leaves the sums of the
// positive and negative fluxes for launch_fct_limiter_sums (null: not wanted)
struct FctFused {
    int apply_cmb = 0, apply_surf = 0;
    double t_cmb = 0.0, t_surf = 0.0;
    double *pp = nullptr, *pm = nullptr;
};
void launch_fct_predictor(const FvArgs& a, const double* vel, const double* T, double dt, double kappa,
                          const double* source, int subtract_div, double* TL, double* ad, const FctFused& fused,
                          hipStream_t s);
void launch_fv_dirichlet(int n, int nr, double* f, int apply_cmb, double t_cmb, int apply_surf, double t_surf,
                         hipStream_t s);
void launch_fct_limiter(int n, int nr, const double* TL, const double* ad, double* Rp, double* Rm, hipStream_t s);
// the same from the predictor's flux sums, held in Rp / Rm and replaced
void launch_fct_limiter_sums(int n, int nr, const double* TL, double* Rp, double* Rm, hipStream_t s);
void launch_fct_correction(int n, int nr, const double* TL, const double* ad, const double* Rp, const double* Rm,
                           double* T, hipStream_t s);
void launch_fv_to_fe_rhs(const FvArgs& a, const double* Tfv, double* b, hipStream_t s);  // Tfv null: all ones
void launch_fv_lumped_scale(const double* D, double* u, int64_t N, hipStream_t s);      // u *= 1 / D
void launch_fe_to_fv(const FvArgs& a, const double* u, double* Tfv, hipStream_t s);    // real cells only

}  // namespace tn

// FV state on one velocity mesh: cell centres, the ghost-layer map and the
// FCT work arrays (the reference's FVFCTBuffers), allocated once
struct tn_fv {
    tn_mesh* mesh = nullptr;
    int n = 0, nr = 0;
    int64_t size = 0;                 // FV scalar elements (ghosts included)
    tn::DevBuf<double> centers;       // [size][3], for tn_fv_cell_centers
    tn::DevBuf<double> columns;       // [10 (n-1)^2][FV_COLUMN] lateral column geometry
    tn::DevBuf<double> layers;        // [nr+1] radial part of the cell centres
    tn::DevBuf<double> TL, Rp, Rm;    // FV scalars; their radial ghost cells at the shells stay zero
    tn::DevBuf<double> ad;            // [6][size] antidiffusive fluxes
    tn::DevBuf<int32_t> pairs;        // [npairs][2]
    int npairs = 0;
    tn::DevBuf<double> part;          // per-block minima of the stable step
    tn::DevBuf<double> result;        // [1]
    tn::FvArgs args() const;
};
