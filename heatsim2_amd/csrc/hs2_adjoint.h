// Adjoint kernels of the ADI step (defined in hs2_adjoint.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "hs2_device.h"

namespace hs2 {

// Fields of one adjoint step.  Inputs: the forward states of the step
// (T^n, T*, T**, T^{n+1}), the transposed-solve results u_x, u_y, u_z, and
// optionally the readout adjoint ghist (ny, nx) of T^n.  Outputs: lam_out =
// dJ/dT^n, gM and gg[axis] (accumulated), gsrc = w u_x (written if non-null).
struct AdjFields {
  const double *Tn, *Tx, *Ty, *Tn1;
  const double *ux, *uy, *uz;
  const double *ghist;
  double *lam_out, *gM;
  double *gg[3];
  double *gsrc;
};

// Up to kAdjGroup adjoint steps whose sensitivities are added in one pass
// (per-voxel coefficients), latest first.  Step s of the group has T^t at
// T - s N, T^{t+1} at T + N - s N, T* and T** at Tx - s N and Ty - s N, and the
// transposed solves u_z, u_y, u_x at u + 3 s N, + N and + 2 N; gsrc[s] takes w u_x
// when non-null.
constexpr int kAdjGroup = 4;
struct AdjGroup {
  const double *T, *Tx, *Ty, *u;
  double *gM;
  double *gg[3];
  double *gsrc[kAdjGroup];
  long long N;
};

struct AdjLineConfig {
  int seg, cw;  // seg 0: unsupported line length
};

AdjLineConfig adj_line_config(int L);

// U = A_axis^{-T} (scale_m ? M R : R) along every line of `axis`
hipError_t launch_adj_line(const Grid &g, const ClassView &v, int axis, const double *R,
                           int scale_m, double *U, hipStream_t s);
hipError_t launch_adj_line(const Grid &g, const DenseView &v, int axis, const double *R,
                           int scale_m, double *U, hipStream_t s);
hipError_t launch_adj_stencil(const Grid &g, const ClassView &v, const AdjFields &f,
                              hipStream_t s);
hipError_t launch_adj_stencil(const Grid &g, const DenseView &v, const AdjFields &f,
                              hipStream_t s);
// per-voxel coefficients, where dense_cols_ok(g, 0): lambda of the step before
// from the solves of the step after (ux null: none) and the readout adjoint gh
// (null: none), and its transposed z solve (solve false: lambda itself)
hipError_t launch_dense_lambda(const Grid &g, const DenseView &v, const double *ux,
                               const double *uy, const double *uz, const double *gh, bool solve,
                               double *U, hipStream_t s);
hipError_t launch_dense_sens(const Grid &g, const DenseView &v, const AdjGroup &f, int cnt,
                             hipStream_t s);
hipError_t launch_lam_from_readout(const Grid &g, const double *ghist, double *lam,
                                   hipStream_t s);
hipError_t launch_fill(double *a, size_t n, double v, hipStream_t s);

}  // namespace hs2
