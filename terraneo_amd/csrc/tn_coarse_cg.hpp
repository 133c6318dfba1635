// The coarsest-level CG in one workgroup (kernels_coarse_cg.hip).
#pragma once

#include <algorithm>

#include "tn_mg.hpp"

namespace tn {

constexpr int COARSE_CG_NODES = 2048;   // node copies, columns padded to a power of two of lanes: 4 per thread
constexpr int COARSE_CG_LDS = 155 * 1024;  // of 160 KB

template <typename T, typename S>
struct CoarseCgArgs {
    StoredArgs<T, S> op;       // the operator (src, dst, csum, ctop, add unused)
    T* x;                      // initial guess (unless zero) and solution
    const T* b;
    const uint8_t* owned_lat;  // [10][n][n]
    const int32_t* groups;     // MeshLevel::d_grp_pad
    const int32_t* group_of;   // MeshLevel::d_grp_of
    int zero;                  // 1: start from x = 0
    int max_iterations;
    double rtol, atol;
    int lanes_log2 = 0;        // lanes of a column (set by the launcher)
};
// whether an n x n x nr operator with elements of esize bytes fits
bool coarse_cg_fits(int n, int nr, int esize);
template <typename T, typename S>
void launch_coarse_cg(CoarseCgArgs<T, S> g, hipStream_t s);

}  // namespace tn
