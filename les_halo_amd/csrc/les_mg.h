// The multigrid preconditioner of the mixed-precision correction solve (les_mg.hip).
#pragma once
#include <vector>

#include "les_mixed.h"

namespace les {

constexpr int MG_MAX = 20;

// One coarse grid: nx x ny columns of kp levels, arrays [k][j][i].
struct MgLevel {
  int nx, ny;
  const float2 *cx, *cy;  // coupling to the i - 1, i + 1 and j - 1, j + 1 neighbour (0: none)
  const int *kx, *ky;     // kx(i) + ky(j): offset of the column's tables below
  float *b, *e, *t;     // right-hand side, solution, scratch of the line solves
  const float* inv;     // 1 / pivot of a column's tridiagonal system, by k
  const float* up;      // its upper factor
  const float *gf, *gb; // products of its recurrences' coefficients within a segment of levels
  // restriction from the next finer grid: coarse index -> up to four fine ones and weights
  const int4 *ri, *rj;
  const float4 *wi, *wj;
  // prolongation to it: fine index -> two coarse ones and weights
  const int2 *pi, *pj;
  const float2 *vi, *vj;
};

struct MgPlan {
  int nl = 0;  // coarse grids; 0: not set up
  MgLevel l[MG_MAX];
  const float *c4l = nullptr, *c4s = nullptr;  // cn4l, cn4s, zero across k = kp and k = 1
  float* mem = nullptr;
};

// Sets up the coarse grids of a uniform horizontal grid (host tables uploaded, synchronises).
hipError_t mg_setup(Dims d, float c2, float c3, const std::vector<float>& cn4l,
                    const std::vector<float>& cn4s, MgPlan& mg);
void mg_release(MgPlan& mg);
// z += P (V-cycle) R s on colour 0, s = colour 0's residual in mx.q[0] (colour 1's is zero);
// nothing once *stopped is nonzero
void launch_mg_correct(hipStream_t st, Dims d, SplitSOR sp, Mixed mx, const MgPlan& mg);

}  // namespace les
