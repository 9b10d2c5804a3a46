// Sweeps on per-voxel coefficients (DenseView, AsymView) and the transposed
// solves of their adjoint, for single plans and for batches (gfx950, FP64).
//
// Rows (x): a row over G lanes x CPL consecutive cells, everything in
// registers.  Columns (y, z): a thread per segment of SEG cells, neighbouring
// columns side by side, the segments' end rows reduced in LDS.
//
// All of it is bound by memory traffic once the chip is full: per cell the x
// sweep moves 49 bytes (T, M, three conductances, w in; out), y and z 41 (33
// where y gets its right-hand side from x), a transposed solve 33.  Times in
// us, the kernels before (rows staged through LDS, both end rows of every
// segment reduced) | now:
//                      64x128x128      48x96x120 (per side)   24 of 32..128^3
//                                                             (in one launch)
//   x                  13.1 | 10.4     13.3 | 9.5             121 | 73
//   y after x / alone  10.5 | 7.3/8.4   9.3 | 7.5              68 | 49/64
//   z                   9.3 | 9.3      10.3 | 7.4              61 | 58
//   transposed x        16.5 | 6.8      -                      74 | 41
//   transposed y        10.8 | 8.5      -                      59 | 52
// 10.4 us for 51 MB is 4.9 TB/s, what a copy between arrays larger than the
// Infinity Cache reaches; 29x45x51 (3.5 to 5.2 us a launch) is bound by the
// latency of one chain of load, solve and store.
#include <algorithm>

#include "hs2_adjoint.h"
#include "hs2_batch.h"
#include "hs2_dense.h"
#include "hs2_launch.h"

namespace hs2 {

// ---------------------------------------------------------------- rows
// x sweep: a wave holds 64/G neighbouring rows and walks KC planes; its own
// cells, the plane's before and the z faces are carried.  Unit `unit` of the
// grid's (row groups) x (chunks of KC planes).  RY: writes y's right-hand side
// M T* - w/2 (Ly T^n) instead of T*.  ck: receives T^n as it passes.
template <class V, int CPL, int G, bool SRC, bool RY>
__device__ __forceinline__ void row_sweep(const Grid &g, const V &v, const double *__restrict__ Tn,
                                          double *__restrict__ Ts,
                                          const uint8_t *__restrict__ vmap, const double *vtab,
                                          const double *__restrict__ sfield,
                                          double *__restrict__ ck, int unit, int KC) {
  constexpr int LPW = kWave / G;
  const int nx = g.nx, ny = g.ny, nz = g.nz;
  const int n = nx * ny * nz;
  const int lane = threadIdx.x & (kWave - 1), lig = lane % G;
  const int nj = (ny + LPW - 1) / LPW;
  const int kc = unit / nj, jg = unit - kc * nj;
  const int jr = jg * LPW + lane / G;
  const int j = min(jr, ny - 1);
  const int i0 = lig * CPL;
  const int left = jr < ny ? nx - i0 : 0;  // cells of the row from this lane on
  const int ir = i0 < nx ? i0 : max(0, nx - CPL);
  const int ym = j > 0 ? j - 1 : j, yp = min(j + 1, ny - 1);
  const int k0 = kc * KC, k1 = min(k0 + KC, nz);
  auto load = [&](const double *__restrict__ a, int k, int jj, double(&o)[CPL]) {
    load_cells<CPL>(a, (k * ny + jj) * nx + ir, n, o);
  };
  double Tm[CPL], T[CPL], Tp[CPL], gz[CPL], gzp[CPL];
  load(Tn, k0 > 0 ? k0 - 1 : k0, j, Tm);
  load(Tn, k0, j, T);
  load(v.g[0], k0, j, gz);
  for (int k = k0; k < k1; k++) {
    const int o = (k * ny + j) * nx + i0;
    // differences across faces that are not there are 0: their neighbour is
    // the cell itself, whatever conductance is read
    double Tym[CPL], Typ[CPL], M[CPL], gx[CPL], gy[CPL], gyp[CPL];
    [[maybe_unused]] double gxp[CPL], S[CPL] = {};
    load(Tn, k, ym, Tym);
    load(Tn, k, yp, Typ);
    load(Tn, min(k + 1, nz - 1), j, Tp);
    load(v.M, k, j, M);
    load(v.g[2], k, j, gx);
    load(v.g[1], k, j, gy);
    if constexpr (V::kAsym) {
      load(v.gp[2], k, j, gxp);
      load(v.gp[1], k, j, gyp);
      load(v.gp[0], k, j, gzp);
    } else {
      load(v.g[1], k, yp, gyp);
      load(v.g[0], min(k + 1, nz - 1), j, gzp);
    }
    const uint64_t wb = load_bytes<CPL>(v.w, (k * ny + j) * nx + ir, n);
    if constexpr (SRC) {
      if (sfield) load(sfield, k, j, S);
      if (vmap) {
        const uint64_t cls = load_bytes<CPL>(vmap, (k * ny + j) * nx + ir, n);
#pragma unroll
        for (int q = 0; q < CPL; q++) S[q] += vtab[(cls >> (8 * q)) & 0xffu];
      }
    }
    const double TL = wave_up(T[CPL - 1]), TR = wave_down(T[0]);
    [[maybe_unused]] const double gR = wave_down(gx[0]);
    double hly[CPL];
    Seg<CPL> seg;
#pragma unroll
    for (int q = 0; q < CPL; q++) {
      const int i = i0 + q;
      const bool in = q < left;
      const double w = (double)(unsigned)((wb >> (8 * q)) & 0xffu);
      const double gm = i > 0 ? gx[q] : 0.0;
      double gp;
      if constexpr (V::kAsym) gp = gxp[q];
      else gp = q < CPL - 1 ? gx[q + 1] : gR;
      if (i + 1 >= nx) gp = 0.0;
      const double Tc = T[q];
      const double dm = (q > 0 ? T[q - 1] : TL) - Tc;
      const double dp = (q < CPL - 1 ? T[q + 1] : TR) - Tc;
      const double ly = __builtin_fma(gyp[q], Typ[q] - Tc, gy[q] * (Tym[q] - Tc));
      double e = __builtin_fma(gzp[q], Tp[q] - Tc, gz[q] * (Tm[q] - Tc)) + ly;
      if (i > 0) e = __builtin_fma(0.5 * gm, dm, e);
      if (i + 1 < nx) e = __builtin_fma(0.5 * gp, dp, e);
      if constexpr (SRC) e += S[q];
      hly[q] = 0.5 * w * ly;
      const double am = -0.5 * w * gm, cp = -0.5 * w * gp;
      seg.row(q, in ? am : 0.0, in ? M[q] - am - cp : 1.0, in ? cp : 0.0,
              in ? __builtin_fma(M[q], Tc, w * e) : 0.0);
    }
    double x[CPL];
    row_solve<CPL, G>(seg, x, lig);
    if constexpr (RY) {
#pragma unroll
      for (int q = 0; q < CPL; q++) x[q] = __builtin_fma(M[q], x[q], -hly[q]);
    }
    if (ck) store_cells<CPL>(ck, o, left, T);
    store_cells<CPL>(Ts, o, left, x);
#pragma unroll
    for (int q = 0; q < CPL; q++) {
      Tm[q] = T[q];
      T[q] = Tp[q];
      if constexpr (!V::kAsym) gz[q] = gzp[q];
    }
    if constexpr (V::kAsym) load(v.g[0], min(k + 1, nz - 1), j, gz);
  }
}

// Transposed x solve: A_x^T U = (scale_m ? M R : R), one row group per unit.
template <class V, int CPL, int G>
__device__ __forceinline__ void row_adjoint(const Grid &g, const V &v, const double *__restrict__ R,
                                            int scale_m, double *__restrict__ U, int unit) {
  constexpr int LPW = kWave / G;
  const int nx = g.nx, rows = g.ny * g.nz, n = nx * rows;
  const int lane = threadIdx.x & (kWave - 1), lig = lane % G;
  const int rr = unit * LPW + lane / G, row = min(rr, rows - 1);
  const int i0 = lig * CPL, left = rr < rows ? nx - i0 : 0;
  const int c = row * nx + (i0 < nx ? i0 : max(0, nx - CPL));
  double M[CPL], gx[CPL], r[CPL], w[CPL];
  load_cells<CPL>(R, c, n, r);
  load_cells<CPL>(v.M, c, n, M);
  load_cells<CPL>(v.g[2], c, n, gx);
  const uint64_t wb = load_bytes<CPL>(v.w, c, n);
#pragma unroll
  for (int q = 0; q < CPL; q++) w[q] = (double)(unsigned)((wb >> (8 * q)) & 0xffu);
  const double wL = wave_up(w[CPL - 1]), wR = wave_down(w[0]), gR = wave_down(gx[0]);
  Seg<CPL> seg;
#pragma unroll
  for (int q = 0; q < CPL; q++) {
    const int i = i0 + q;
    const bool in = q < left;
    const double gm = i > 0 ? gx[q] : 0.0;
    const double gp = i + 1 < nx ? (q < CPL - 1 ? gx[q + 1] : gR) : 0.0;
    const double a = i > 0 ? -0.5 * (q > 0 ? w[q - 1] : wL) * gm : 0.0;
    const double cc = i + 1 < nx ? -0.5 * (q < CPL - 1 ? w[q + 1] : wR) * gp : 0.0;
    const double b = M[q] + 0.5 * w[q] * (gm + gp);
    const double rhs = scale_m ? M[q] * r[q] : r[q];
    seg.row(q, in ? a : 0.0, in ? b : 1.0, in ? cc : 0.0, in ? rhs : 0.0);
  }
  double x[CPL];
  row_solve<CPL, G>(seg, x, lig);
  store_cells<CPL>(U, row * nx + i0, left, x);
}

// ------------------------------------------------------------- columns
// A block's CW neighbouring columns (all of the grid's in memory order) x P
// segments of SEG cells; threads past P x CW only take part in the barriers.
// Rows past a column's end read what follows it (or 0 past the array's end,
// the buffers' bound on the lane's offset) and become identity rows.
struct ColPlace {
  int p, cl, base, L, t0;
  bool act, valid;
  unsigned vo, so;  // byte offsets: the segment's first cell; a row of the column
};
template <int AXIS>
__device__ __forceinline__ ColPlace col_place(const Grid &g, int seg, int P, int CW, int blk) {
  ColPlace c;
  c.p = threadIdx.x / CW;
  c.cl = threadIdx.x - c.p * CW;
  c.act = c.p < P;
  c.L = AXIS == 1 ? g.ny : g.nz;
  const int ncol = g.nx * (AXIS == 1 ? g.nz : g.ny), col = blk * CW + c.cl;
  c.valid = c.act && col < ncol;
  c.base = min(col, ncol - 1);
  if (AXIS == 1) {
    const int k = c.base / g.nx;
    c.base = k * g.ny * g.nx + (c.base - k * g.nx);
  }
  c.t0 = min(c.p, P - 1) * seg;
  c.so = (unsigned)(AXIS == 1 ? g.nx : g.nx * g.ny);
  c.vo = (unsigned)c.base + (unsigned)c.t0 * c.so;
  return c;
}

// y and z sweeps: (M - La/2) X = M Y - (La/2) T^n, or = Y with RY.  X may alias
// Y or T^n: a block owns whole columns, and all of its loads happen before its
// first barrier and all of its stores after its last.
template <class V, int SEG, int AXIS, bool RY>
__device__ __forceinline__ void col_sweep(const Grid &g, const V &v, int P, int CW,
                                          const double *Tn, const double *Y, double *X,
                                          double *surf, double dz, int blk) {
  extern __shared__ double lds[];
  const ColPlace c = col_place<AXIS>(g, SEG, P, CW, blk);
  const unsigned n = (unsigned)g.nx * (unsigned)g.ny * (unsigned)g.nz;
  const BufRsrc bT = make_buf(Tn, n * 8u), bY = make_buf(Y, n * 8u), bX = make_buf(X, n * 8u),
                bM = make_buf(v.M, n * 8u), bG = make_buf(v.g[AXIS], n * 8u),
                bW = make_buf(v.w, n);
  const unsigned so = c.so * 8u, vo = c.vo * 8u;
  double Yv[SEG], M[SEG], G[SEG + 1];
  [[maybe_unused]] double T[SEG + 2], Gp[SEG];
  uint32_t w[SEG];
  if constexpr (!RY) {
    T[0] = buf_load_d(bT, c.t0 > 0 ? vo - so : vo);
#pragma unroll
    for (int q = 0; q <= SEG; q++) T[q + 1] = buf_load_d(bT, vo + q * so);
  }
#pragma unroll
  for (int q = 0; q < SEG; q++) Yv[q] = buf_load_d(bY, vo + q * so);
#pragma unroll
  for (int q = 0; q < SEG; q++) M[q] = buf_load_d(bM, vo + q * so);
#pragma unroll
  for (int q = 0; q < (V::kAsym ? SEG : SEG + 1); q++) G[q] = buf_load_d(bG, vo + q * so);
  if constexpr (V::kAsym) {
    const BufRsrc bP = make_buf(v.gp[AXIS], n * 8u);
#pragma unroll
    for (int q = 0; q < SEG; q++) Gp[q] = buf_load_d(bP, vo + q * so);
  }
#pragma unroll
  for (int q = 0; q < SEG; q++) w[q] = buf_load_u8(bW, c.vo + q * c.so);
  Seg<SEG> seg;
#pragma unroll
  for (int q = 0; q < SEG; q++) {
    const int t = c.t0 + q;
    const bool in = t < c.L;
    const double wd = (double)w[q];
    const double gm = t > 0 ? G[q] : 0.0;
    double gp;
    if constexpr (V::kAsym) gp = Gp[q];
    else gp = G[q + 1];
    if (t + 1 >= c.L) gp = 0.0;
    double rhs;
    if constexpr (RY) {
      rhs = Yv[q];
    } else {  // the order of the x sweep's right-hand side for y (RY there)
      const double dm = t > 0 ? T[q] - T[q + 1] : 0.0;
      const double dp = t + 1 < c.L ? T[q + 2] - T[q + 1] : 0.0;
      const double h = 0.5 * wd * __builtin_fma(gp, dp, gm * dm);
      rhs = __builtin_fma(M[q], Yv[q], -h);
    }
    const double am = -0.5 * wd * gm, cp = -0.5 * wd * gp;
    seg.row(q, in ? am : 0.0, in ? M[q] - am - cp : 1.0, in ? cp : 0.0, in ? rhs : 0.0);
  }
  double As, Cs, Rs, Ae, Ce, Re, xs = 0.0, xe = 0.0;
  seg.finish(As, Cs, Rs, Ae, Ce, Re);
  block_ends(lds, c.p, P, CW, c.cl, c.act, As, Cs, Rs, Ae, Ce, Re, xs, xe);
  if (!c.valid) return;
  double x1 = xe;
#pragma unroll
  for (int q = 0; q < SEG; q++) {
    const double x = q == 0 ? xs : q == SEG - 1 ? xe : seg.interior(q, xs, xe);
    if (q == 1) x1 = x;
    if (c.t0 + q < c.L) buf_store_ds(x, bX, vo, q * so);
  }
  if (AXIS == 0 && surf && c.p == 0 && c.L >= 2) surf[c.base] = surface_readout(xs, x1, dz);
}

// Transposed y solve: A_y^T U = (scale_m ? M R : R).  U must not alias R.  (z's is
// col_lambda's.)
template <class V, int SEG>
__device__ __forceinline__ void col_adjoint(const Grid &g, const V &v, int P, int CW,
                                            const double *R, int scale_m, double *U, int blk) {
  extern __shared__ double lds[];
  const ColPlace c = col_place<1>(g, SEG, P, CW, blk);
  const unsigned n = (unsigned)g.nx * (unsigned)g.ny * (unsigned)g.nz;
  const BufRsrc bR = make_buf(R, n * 8u), bU = make_buf(U, n * 8u), bM = make_buf(v.M, n * 8u),
                bG = make_buf(v.g[1], n * 8u), bW = make_buf(v.w, n);
  const unsigned so = c.so * 8u, vo = c.vo * 8u;
  double r[SEG], M[SEG], G[SEG + 1];
  uint32_t w[SEG + 2];
#pragma unroll
  for (int q = 0; q < SEG; q++) r[q] = buf_load_d(bR, vo + q * so);
#pragma unroll
  for (int q = 0; q < SEG; q++) M[q] = buf_load_d(bM, vo + q * so);
#pragma unroll
  for (int q = 0; q <= SEG; q++) G[q] = buf_load_d(bG, vo + q * so);
  w[0] = buf_load_u8(bW, c.t0 > 0 ? c.vo - c.so : c.vo);
#pragma unroll
  for (int q = 0; q <= SEG; q++) w[q + 1] = buf_load_u8(bW, c.vo + q * c.so);
  Seg<SEG> seg;
#pragma unroll
  for (int q = 0; q < SEG; q++) {
    const int t = c.t0 + q;
    const bool in = t < c.L;
    const double gm = t > 0 ? G[q] : 0.0;
    const double gp = t + 1 < c.L ? G[q + 1] : 0.0;
    const double b = M[q] + 0.5 * (double)w[q + 1] * (gm + gp);
    const double rhs = scale_m ? M[q] * r[q] : r[q];
    seg.row(q, in ? -0.5 * (double)w[q] * gm : 0.0, in ? b : 1.0,
            in ? -0.5 * (double)w[q + 2] * gp : 0.0, in ? rhs : 0.0);
  }
  double As, Cs, Rs, Ae, Ce, Re, xs = 0.0, xe = 0.0;
  seg.finish(As, Cs, Rs, Ae, Ce, Re);
  block_ends(lds, c.p, P, CW, c.cl, c.act, As, Cs, Rs, Ae, Ce, Re, xs, xe);
  if (!c.valid) return;
#pragma unroll
  for (int q = 0; q < SEG; q++) {
    const double x = q == 0 ? xs : q == SEG - 1 ? xe : seg.interior(q, xs, xe);
    if (c.t0 + q < c.L) buf_store_ds(x, bU, vo, q * so);
  }
}

// dJ/dT^{t+1} (lambda) of the cells of a block's z columns, and its transposed
// z solve: A_z^T U = lambda.  lambda is the adjoint stencil of the step after
// (its transposed solves ux, uy, uz; null: no such step) plus the readout
// adjoint `gh` of T^{t+1} on the top two layers.  U may be uz: a block reads uz
// in its own columns only, before its first barrier.  SOLVE false: lambda is
// the result.
//
// One pass instead of the adjoint stencil's lambda and the z solve that read it
// back (65 bytes a cell; those moved 98).  Memory and latency bound at three
// waves a SIMD: all of a segment's loads are issued together (about 160
// registers).  Fewer registers lose: 128 by spilling 24.2 us, 150 by loading
// the y faces after the x faces are done 18.3, as it stands 15.3 (64x128x128).
template <int SEG, bool SOLVE>
__device__ __forceinline__ void col_lambda(const Grid &g, const DenseView &v, int P, int CW,
                                           const double *ux, const double *uy, const double *uz,
                                           const double *gh, double *U, int blk) {
  extern __shared__ double lds[];
  const ColPlace c = col_place<0>(g, SEG, P, CW, blk);
  const int nx = g.nx, j = c.base / nx, i = c.base - j * nx;
  const unsigned n = (unsigned)nx * (unsigned)g.ny * (unsigned)g.nz;
  const BufRsrc bU = make_buf(U, n * 8u), bM = make_buf(v.M, n * 8u),
                bGz = make_buf(v.g[0], n * 8u), bW = make_buf(v.w, n);
  const unsigned so = c.so * 8u, vo = c.vo * 8u, row = (unsigned)nx;
  double M[SEG], G[SEG + 1], lam[SEG];
  uint32_t w[SEG + 2];
#pragma unroll
  for (int q = 0; q < SEG; q++) M[q] = buf_load_d(bM, vo + q * so);
#pragma unroll
  for (int q = 0; q <= SEG; q++) G[q] = buf_load_d(bGz, vo + q * so);
  w[0] = buf_load_u8(bW, c.t0 > 0 ? c.vo - c.so : c.vo);
#pragma unroll
  for (int q = 0; q <= SEG; q++) w[q + 1] = buf_load_u8(bW, c.vo + q * c.so);
  if (ux) {
    // v across the faces of each axis: x: w ux / 2, y: w (ux - uy / 2), z:
    // w (ux - uz / 2); faces that are not there add nothing (an offset before
    // the array or behind it reads 0)
    const BufRsrc bX = make_buf(ux, n * 8u), bY = make_buf(uy, n * 8u), bZ = make_buf(uz, n * 8u),
                  bGx = make_buf(v.g[2], n * 8u), bGy = make_buf(v.g[1], n * 8u);
    double x[SEG], vz[SEG + 2];
    {
      const unsigned om = c.t0 > 0 ? vo - so : vo;
      vz[0] = (double)w[0] * (buf_load_d(bX, om) - 0.5 * buf_load_d(bZ, om));
    }
#pragma unroll
    for (int q = 0; q <= SEG; q++) {
      const double xq = buf_load_d(bX, vo + q * so);
      if (q < SEG) x[q] = xq;
      vz[q + 1] = (double)w[q + 1] * (xq - 0.5 * buf_load_d(bZ, vo + q * so));
    }
#pragma unroll
    for (int q = 0; q < SEG; q++) {
      const int t = c.t0 + q;
      const double dm = t > 0 ? vz[q] - vz[q + 1] : 0.0;
      const double dp = t + 1 < c.L ? vz[q + 2] - vz[q + 1] : 0.0;
      lam[q] = __builtin_fma(G[q + 1], dp, __builtin_fma(G[q], dm, M[q] * x[q]));
    }
#pragma unroll
    for (int q = 0; q < SEG; q++) {
      const unsigned o = vo + q * so, ow = c.vo + q * c.so;
      const double vc = 0.5 * (double)w[q + 1] * x[q];
      const double vm = 0.5 * (double)buf_load_u8(bW, ow - 1u) * buf_load_d(bX, o - 8u);
      const double vp = 0.5 * (double)buf_load_u8(bW, ow + 1u) * buf_load_d(bX, o + 8u);
      const double dm = i > 0 ? vm - vc : 0.0, dp = i + 1 < nx ? vp - vc : 0.0;
      lam[q] = __builtin_fma(buf_load_d(bGx, o + 8u), dp,
                             __builtin_fma(buf_load_d(bGx, o), dm, lam[q]));
    }
#pragma unroll
    for (int q = 0; q < SEG; q++) {
      const unsigned o = vo + q * so, ow = c.vo + q * c.so;
      const double vc = (double)w[q + 1] * (x[q] - 0.5 * buf_load_d(bY, o));
      const double vm = (double)buf_load_u8(bW, ow - row) *
                        (buf_load_d(bX, o - 8u * row) - 0.5 * buf_load_d(bY, o - 8u * row));
      const double vp = (double)buf_load_u8(bW, ow + row) *
                        (buf_load_d(bX, o + 8u * row) - 0.5 * buf_load_d(bY, o + 8u * row));
      const double dm = j > 0 ? vm - vc : 0.0, dp = j + 1 < g.ny ? vp - vc : 0.0;
      lam[q] = __builtin_fma(buf_load_d(bGy, o + 8u * row), dp,
                             __builtin_fma(buf_load_d(bGy, o), dm, lam[q]));
    }
  } else {
#pragma unroll
    for (int q = 0; q < SEG; q++) lam[q] = 0.0;
  }
  if (gh && c.t0 == 0) {
    const double s = gh[c.base];
    lam[0] = __builtin_fma(21.0 / 16.0, s, lam[0]);
    lam[1] = __builtin_fma(-5.0 / 16.0, s, lam[1]);
  }
  if constexpr (!SOLVE) {
    if (!c.valid) return;
#pragma unroll
    for (int q = 0; q < SEG; q++)
      if (c.t0 + q < c.L) buf_store_ds(lam[q], bU, vo, q * so);
  } else {
    Seg<SEG> seg;
#pragma unroll
    for (int q = 0; q < SEG; q++) {
      const int t = c.t0 + q;
      const bool in = t < c.L;
      const double gm = t > 0 ? G[q] : 0.0;
      const double gp = t + 1 < c.L ? G[q + 1] : 0.0;
      const double b = M[q] + 0.5 * (double)w[q + 1] * (gm + gp);
      seg.row(q, in ? -0.5 * (double)w[q] * gm : 0.0, in ? b : 1.0,
              in ? -0.5 * (double)w[q + 2] * gp : 0.0, in ? lam[q] : 0.0);
    }
    double As, Cs, Rs, Ae, Ce, Re, xs = 0.0, xe = 0.0;
    seg.finish(As, Cs, Rs, Ae, Ce, Re);
    block_ends(lds, c.p, P, CW, c.cl, c.act, As, Cs, Rs, Ae, Ce, Re, xs, xe);
    if (!c.valid) return;
#pragma unroll
    for (int q = 0; q < SEG; q++) {
      const double y = q == 0 ? xs : q == SEG - 1 ? xe : seg.interior(q, xs, xe);
      if (c.t0 + q < c.L) buf_store_ds(y, bU, vo, q * so);
    }
  }
}

// Sensitivities of up to kAdjGroup adjoint steps added to the four gradient
// fields, latest step first: one pass over the fields for the group instead of
// one for every step.  A thread owns one column of planes k0 .. k1 - 1 and
// carries the plane before in registers.
//
// Bound by memory: (25 fields read, 4 of them read and written, and w for four
// steps) 265 bytes a cell in 52 us at 64x128x128, 5.3 TB/s.  lambda, the z
// solve and this take 28 us a step there, where a stencil that added every
// step by itself took 35.3 and the z solve 7.9; a batch of 24 instances of
// 32..128^3 went from 298 to 243.  Groups of eight read 13% less a step but
// run slower at 64x128x128 (102 us) and gain 1% of the whole in the batch,
// for 12 more fields of workspace.
__device__ __forceinline__ void add_sensitivities(const Grid &g, const uint8_t *__restrict__ w,
                                                  const AdjGroup &f, int cnt, int col, int k0,
                                                  int k1) {
  constexpr int S = kAdjGroup;
  const int nx = g.nx, sxy = nx * g.ny;
  if (col >= sxy) return;
  const int j = col / nx, i = col - j * nx;
  const double *__restrict__ T = f.T, *__restrict__ Tx = f.Tx, *__restrict__ Ty = f.Ty,
               *__restrict__ u = f.u;
  const long long N = f.N;
  // of the plane before: T^{t+1} of the latest step and every T^t, w ux, w uz
  double bT[S + 1] = {}, bX[S] = {}, bZ[S] = {};
  if (k0 > 0) {
    const int c = (k0 - 1) * sxy + col;
    const double wc = w[c];
    bT[0] = T[N + c];
#pragma unroll
    for (int s = 0; s < S; s++)
      if (s < cnt) {
        bT[s + 1] = T[c - s * N];
        bZ[s] = wc * u[3 * s * N + c];
        bX[s] = wc * u[(3 * s + 2) * N + c];
      }
  }
  for (int k = k0; k < k1; k++) {
    const int c = k * sxy + col, cx = i > 0 ? c - 1 : c, cy = j > 0 ? c - nx : c;
    const double wc = w[c], wx = w[cx], wy = w[cy];
    double aM = f.gM[c], az = f.gg[0][c], ay = f.gg[1][c], ax = f.gg[2][c];
    double T1 = T[N + c], T1b = bT[0];
    bT[0] = T1;
#pragma unroll
    for (int s = 0; s < S; s++)
      if (s < cnt) {
        const double *Ts = T - s * N, *Xs = Tx - s * N, *Ys = Ty - s * N;
        const double *uz = u + 3 * s * N, *uy = uz + N, *ux = uy + N;
        const double Tn = Ts[c], X = Xs[c], Y = Ys[c], z = uz[c], y = uy[c], x = ux[c];
        const double wz_ = wc * z, wy_ = wc * y, wx_ = wc * x;
        aM -= x * (X - Tn) + y * (Y - X) + z * (T1 - Y);
        const double gx = 0.5 * ((X + Tn) - (Xs[cx] + Ts[cx])) * (wx * ux[cx] - wx_);
        ax += i > 0 ? gx : 0.0;
        const double Tm = Ts[cy];
        const double gy = (Tn - Tm) * (wy * ux[cy] - wx_) +
                          0.5 * ((Y - Tn) - (Ys[cy] - Tm)) * (wy * uy[cy] - wy_);
        ay += j > 0 ? gy : 0.0;
        const double Tb = bT[s + 1];
        const double gz =
            (Tn - Tb) * (bX[s] - wx_) + 0.5 * ((T1 - Tn) - (T1b - Tb)) * (bZ[s] - wz_);
        az += k > 0 ? gz : 0.0;
        if (f.gsrc[s]) f.gsrc[s][c] = wx_;
        T1 = Tn;
        T1b = Tb;
        bT[s + 1] = Tn;
        bX[s] = wx_;
        bZ[s] = wz_;
      }
    f.gM[c] = aM;
    f.gg[0][c] = az;
    f.gg[1][c] = ay;
    f.gg[2][c] = ax;
  }
}

// -------------------------------------------------------- single plans
template <class V, int CPL, int G, bool SRC, bool RY>
__global__ __launch_bounds__(256) void k_drows(Grid g, V v, const double *Tn, double *Ts,
                                               const uint8_t *vmap, const double *vtab_g,
                                               const double *sfield, int KC, int units) {
  __shared__ double vtab[SRC ? kMaxVtab : 1];
  if (SRC && vmap) {
    for (int e = threadIdx.x; e < kMaxVtab; e += 256) vtab[e] = vtab_g[e];
    __syncthreads();
  }
  const int unit = xcd_remap(blockIdx.x, gridDim.x) * (256 / kWave) +
                   __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  if (unit >= units) return;
  row_sweep<V, CPL, G, SRC, RY>(g, v, Tn, Ts, vmap, vtab, sfield, nullptr, unit, KC);
}

template <class V, int SEG, int AXIS, bool RY>
__global__ __launch_bounds__(512) void k_dcols(Grid g, V v, int P, int CW, const double *Tn,
                                               const double *Y, double *X, double *surf,
                                               double dz) {
  col_sweep<V, SEG, AXIS, RY>(g, v, P, CW, Tn, Y, X, surf, dz,
                              xcd_remap_chunks<32>(blockIdx.x, gridDim.x));
}

template <class V, int CPL, int G>
__global__ __launch_bounds__(256) void k_drows_adj(Grid g, V v, const double *R, int scale_m,
                                                   double *U, int units) {
  const int unit = xcd_remap(blockIdx.x, gridDim.x) * (256 / kWave) +
                   __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  if (unit < units) row_adjoint<V, CPL, G>(g, v, R, scale_m, U, unit);
}

template <class V, int SEG>
__global__ __launch_bounds__(512) void k_dcols_adj(Grid g, V v, int P, int CW, const double *R,
                                                   int scale_m, double *U) {
  col_adjoint<V, SEG>(g, v, P, CW, R, scale_m, U,
                            xcd_remap_chunks<32>(blockIdx.x, gridDim.x));
}

template <int SEG, bool SOLVE>
__global__ __launch_bounds__(512) void k_dlambda(Grid g, DenseView v, int P, int CW,
                                                 const double *ux, const double *uy,
                                                 const double *uz, const double *gh, double *U) {
  col_lambda<SEG, SOLVE>(g, v, P, CW, ux, uy, uz, gh, U,
                         xcd_remap_chunks<32>(blockIdx.x, gridDim.x));
}

__global__ __launch_bounds__(256) void k_dsens(Grid g, const uint8_t *w, AdjGroup f, int cnt,
                                               int KZ, int nbp) {
  const int b = xcd_remap_chunks<32>(blockIdx.x, gridDim.x), kc = b / nbp;
  add_sensitivities(g, w, f, cnt, (b - kc * nbp) * 256 + (int)threadIdx.x, kc * KZ,
                    min(kc * KZ + KZ, g.nz));
}

// cells per lane and lanes of a row of nx cells (0: none).  Twice the lanes at
// half the cells was measured at 29x45x51 (4.4 against 4.4 us) and at
// 64x128x128 (11.6 against 10.5).
static void drow_shape(int nx, int *cpl, int *G) {
  *G = nx <= 64 ? 16 : nx <= 128 ? 32 : 64;
  *cpl = std::max((nx + *G - 1) / *G, *G == 16 ? 2 : 3);
  if (nx > 256) *cpl = *G = 0;
}
// Columns: segments of 8 cells up to 256 (16 beyond), and blocks of whole
// 128-byte lines, P x CW <= 512 threads: 32 columns where that leaves a block
// for every CU, 16 where it does not.  Measured (us, 8 cells x 16 | 8 x 32 |
// 16 x 32 | 4 x 16): y at 64x128x128 10.0 | 8.5 | 8.9 | 11.0, z 9.6 | 9.4 |
// 10.9 | 10.2; y at 48x96x120 7.5 | 8.6 | 8.5 | 9.4, at 29x45x51 5.2 | 5.5 |
// 6.0 | 5.3; column counts that are not whole lines cost more: 8 x 21 8.6 and
// 4 x 21 9.1 at 48x96x120.
static void dcol_shape(int L, long long ncol, int *seg, int *P, int *CW) {
  *seg = L <= 256 ? 8 : 16;
  *P = (L + *seg - 1) / *seg;
  *CW = *P <= 16 && ncol >= 256 * 32 ? 32 : 16;
}

bool dense_rows_ok(const Grid &g) {
  return g.nx <= 256 && (size_t)g.nx * g.ny * g.nz < (size_t(1) << 31) - 64;
}
bool dense_cols_ok(const Grid &g, int axis) {
  return (axis == 1 ? g.ny : g.nz) <= 512 &&
         (size_t)g.nx * g.ny * g.nz * sizeof(double) < (size_t(1) << 32);
}

bool dense_ry(const Grid &g) { return dense_rows_ok(g) && dense_cols_ok(g, 1); }

template <class V, int CPL, int G>
static hipError_t launch_drows_t(const Grid &g, const V &v, const double *Tn, double *Ts,
                                 const uint8_t *vmap, const double *vtab, const double *sfield,
                                 bool ry, hipStream_t s) {
  const long long nj = (g.ny + kWave / G - 1) / (kWave / G);
  // planes a wave walks: two share T and the z faces in registers, but halve
  // the waves; at 64x128x128 (4096 row groups) one takes 10.4 us and two 11.0,
  // in a batch of 48 thousand row groups 74.5 and 72.7 (four 75.2, eight 85.7)
  const int KC = nj * g.nz >= 8192 ? 2 : 1;
  const int units = (int)(nj * ((g.nz + KC - 1) / KC));
  const dim3 grid((unsigned)((units + 3) / 4)), block(256);
#define HS2_RUN(SRC, RY)                                                                     \
  hipLaunchKernelGGL((k_drows<V, CPL, G, SRC, RY>), grid, block, 0, s, g, v, Tn, Ts, vmap, vtab, \
                     sfield, KC, units)
  if (vmap || sfield) {
    if (ry) HS2_RUN(true, true);
    else HS2_RUN(true, false);
  } else {
    if (ry) HS2_RUN(false, true);
    else HS2_RUN(false, false);
  }
#undef HS2_RUN
  return hipGetLastError();
}

template <class V>
static hipError_t launch_drows(const Grid &g, const V &v, const double *Tn, double *Ts,
                               const uint8_t *vmap, const double *vtab, const double *sfield,
                               bool ry, hipStream_t s) {
  int cpl, G;
  drow_shape(g.nx, &cpl, &G);
#define HS2_ROW(C, GG) \
  if (cpl == C && G == GG) return launch_drows_t<V, C, GG>(g, v, Tn, Ts, vmap, vtab, sfield, ry, s);
  HS2_ROW(2, 16) HS2_ROW(3, 16) HS2_ROW(4, 16) HS2_ROW(3, 32) HS2_ROW(4, 32) HS2_ROW(3, 64)
  HS2_ROW(4, 64)
#undef HS2_ROW
  return hipErrorInvalidValue;
}

template <class V, int SEG>
static hipError_t launch_dcols_t(const Grid &g, const V &v, int axis, int P, int CW,
                                 const double *Tn, const double *Y, double *X, double *surf,
                                 double dz, bool ry, hipStream_t s) {
  const long long ncol = (long long)g.nx * (axis == 1 ? g.nz : g.ny);
  const dim3 grid((unsigned)((ncol + CW - 1) / CW)), block(P * CW);
  const size_t shm = sizeof(double) * 6 * P * CW;
#define HS2_RUN(AXIS, RY)                                                                        \
  hipLaunchKernelGGL((k_dcols<V, SEG, AXIS, RY>), grid, block, shm, s, g, v, P, CW, Tn, Y, X,    \
                     surf, dz)
  if (axis == 1 && ry) HS2_RUN(1, true);
  else if (axis == 1) HS2_RUN(1, false);
  else if (!ry) HS2_RUN(0, false);
  else return hipErrorInvalidValue;
#undef HS2_RUN
  return hipGetLastError();
}

template <class V>
static hipError_t launch_dcols(const Grid &g, const V &v, int axis, const double *Tn,
                               const double *Y, double *X, double *surf, double dz, bool ry,
                               hipStream_t s) {
  int seg, P, CW;
  dcol_shape(axis == 1 ? g.ny : g.nz, (long long)g.nx * (axis == 1 ? g.nz : g.ny), &seg, &P, &CW);
  return seg == 8 ? launch_dcols_t<V, 8>(g, v, axis, P, CW, Tn, Y, X, surf, dz, ry, s)
                  : launch_dcols_t<V, 16>(g, v, axis, P, CW, Tn, Y, X, surf, dz, ry, s);
}

hipError_t launch_dense_x(const Grid &g, const DenseView &v, const double *Tn, double *Ts,
                          const uint8_t *vmap, const double *vtab, const double *sfield, bool ry,
                          hipStream_t s) {
  return launch_drows(g, v, Tn, Ts, vmap, vtab, sfield, ry, s);
}
hipError_t launch_dense_x(const Grid &g, const AsymView &v, const double *Tn, double *Ts,
                          const uint8_t *vmap, const double *vtab, const double *sfield, bool ry,
                          hipStream_t s) {
  return launch_drows(g, v, Tn, Ts, vmap, vtab, sfield, ry, s);
}
hipError_t launch_dense_cols(const Grid &g, const DenseView &v, int axis, const double *Tn,
                             const double *Y, double *X, double *surf, double dz, bool ry,
                             hipStream_t s) {
  return launch_dcols(g, v, axis, Tn, Y, X, surf, dz, ry, s);
}
hipError_t launch_dense_cols(const Grid &g, const AsymView &v, int axis, const double *Tn,
                             const double *Y, double *X, double *surf, double dz, bool ry,
                             hipStream_t s) {
  return launch_dcols(g, v, axis, Tn, Y, X, surf, dz, ry, s);
}

hipError_t launch_dense_adj(const Grid &g, const DenseView &v, int axis, const double *R,
                            int scale_m, double *U, hipStream_t s) {
  if (axis == 2) {
    int cpl, G;
    drow_shape(g.nx, &cpl, &G);
    if (!G) return hipErrorInvalidValue;
    const long long rows = (long long)g.ny * g.nz;
    const int units = (int)((rows + kWave / G - 1) / (kWave / G));
    const dim3 grid((unsigned)((units + 3) / 4)), block(256);
#define HS2_ROW(C, GG)                                                                        \
  if (cpl == C && G == GG)                                                                    \
    hipLaunchKernelGGL((k_drows_adj<DenseView, C, GG>), grid, block, 0, s, g, v, R, scale_m, U, \
                       units);
    HS2_ROW(2, 16) HS2_ROW(3, 16) HS2_ROW(4, 16) HS2_ROW(3, 32) HS2_ROW(4, 32) HS2_ROW(3, 64)
    HS2_ROW(4, 64)
#undef HS2_ROW
    return hipGetLastError();
  }
  int seg, P, CW;
  const long long ncol = (long long)g.nx * g.nz;
  dcol_shape(g.ny, ncol, &seg, &P, &CW);
  const dim3 grid((unsigned)((ncol + CW - 1) / CW)), block(P * CW);
  const size_t shm = sizeof(double) * 6 * P * CW;
  if (seg == 8)
    hipLaunchKernelGGL((k_dcols_adj<DenseView, 8>), grid, block, shm, s, g, v, P, CW, R, scale_m, U);
  else
    hipLaunchKernelGGL((k_dcols_adj<DenseView, 16>), grid, block, shm, s, g, v, P, CW, R, scale_m,
                       U);
  return hipGetLastError();
}

hipError_t launch_dense_lambda(const Grid &g, const DenseView &v, const double *ux,
                               const double *uy, const double *uz, const double *gh, bool solve,
                               double *U, hipStream_t s) {
  int seg, P, CW;
  const long long ncol = (long long)g.nx * g.ny;
  dcol_shape(g.nz, ncol, &seg, &P, &CW);
  const dim3 grid((unsigned)((ncol + CW - 1) / CW)), block(P * CW);
  const size_t shm = sizeof(double) * 6 * P * CW;
#define HS2_RUN(SEG, SOLVE)                                                                   \
  if (seg == SEG && solve == SOLVE)                                                           \
    hipLaunchKernelGGL((k_dlambda<SEG, SOLVE>), grid, block, shm, s, g, v, P, CW, ux, uy, uz, gh, \
                       U);
  HS2_RUN(8, true) HS2_RUN(8, false) HS2_RUN(16, true) HS2_RUN(16, false)
#undef HS2_RUN
  return hipGetLastError();
}

hipError_t launch_dense_sens(const Grid &g, const DenseView &v, const AdjGroup &f, int cnt,
                             hipStream_t s) {
  const int nbp = (g.nx * g.ny + 255) / 256;
  const int KZ = std::clamp(nbp * 4 * g.nz / 2048, 1, 16);
  hipLaunchKernelGGL(k_dsens, dim3((unsigned)(nbp * ((g.nz + KZ - 1) / KZ))), dim3(256), 0, s, g,
                     v.w, f, cnt, KZ, nbp);
  return hipGetLastError();
}

// -------------------------------------------------------------- batches
// One launch covers every instance (axis lengths <= kBatchMaxLen); see
// hs2_batch.h for the block mapping.
template <bool RY>
__global__ __launch_bounds__(kBatchWaves *kWave) void kb_rows(BatchMap m, DenseView v,
                                                              const double *Tn, double *Ts,
                                                              const double *src, double *ck) {
  BatchInst I;
  int local, t;
  if (!batch_locate(m, I, local, t)) return;
  const int unit = local * kBatchWaves + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  if (unit >= I.units) return;
  double *c = nullptr;
  // T^t starts a checkpoint segment (aligned to the instance's end) or the run
  const int r = I.nsteps - t;
  if (ck && (r % m.K == 0 || t == 0))
    c = ck + I.ckoff + (long long)((r + m.K - 1) / m.K - 1) * ((long long)I.nz * I.ny * I.nx);
  const double *sf = (src && t == I.src_step) ? src + I.off : nullptr;
  const Grid g{I.nz, I.ny, I.nx};
  const DenseView vi = offset_view(v, I.off);
#define HS2_ROW(C, GG)                                                                         \
  row_sweep<DenseView, C, GG, true, RY>(g, vi, Tn + I.off, Ts + I.off, nullptr, nullptr, sf, c, \
                                        unit, kBatchPlanes)
  switch (I.row) {
    case 0: HS2_ROW(2, 16); break;
    case 1: HS2_ROW(4, 16); break;
    case 2: HS2_ROW(3, 32); break;
    default: HS2_ROW(4, 32); break;
  }
#undef HS2_ROW
}

template <int AXIS, bool RY>
__global__ __launch_bounds__(kBatchThreads) void kb_cols(BatchMap m, DenseView v, const double *Tn,
                                                         const double *Y, double *X,
                                                         double *hist) {
  BatchInst I;
  int local, t;
  if (!batch_locate(m, I, local, t)) return;
  double *surf = (AXIS == 0 && hist) ? hist + I.hoff + (long long)t * I.ny * I.nx : nullptr;
  col_sweep<DenseView, kBatchSeg, AXIS, RY>(
      Grid{I.nz, I.ny, I.nx}, offset_view(v, I.off), batch_line_segs(AXIS == 1 ? I.ny : I.nz),
      I.cw[AXIS], Tn + I.off, Y + I.off, X + I.off, surf, I.dz, local);
}

__global__ __launch_bounds__(kBatchWaves *kWave) void kb_rows_adj(BatchMap m, DenseView v,
                                                                  const double *R, int scale_m,
                                                                  double *U) {
  BatchInst I;
  int local, t;
  if (!batch_locate(m, I, local, t)) return;
  const int unit = local * kBatchWaves + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  if (unit >= I.rows) return;
  const Grid g{I.nz, I.ny, I.nx};
  const DenseView vi = offset_view(v, I.off);
#define HS2_ROW(C, GG) row_adjoint<DenseView, C, GG>(g, vi, R + I.off, scale_m, U + I.off, unit)
  switch (I.row) {
    case 0: HS2_ROW(2, 16); break;
    case 1: HS2_ROW(4, 16); break;
    case 2: HS2_ROW(3, 32); break;
    default: HS2_ROW(4, 32); break;
  }
#undef HS2_ROW
}

__global__ __launch_bounds__(kBatchThreads) void kb_cols_adj(BatchMap m, DenseView v,
                                                             const double *R, int scale_m,
                                                             double *U) {
  BatchInst I;
  int local, t;
  if (!batch_locate(m, I, local, t)) return;
  col_adjoint<DenseView, kBatchSeg>(Grid{I.nz, I.ny, I.nx}, offset_view(v, I.off),
                                    batch_line_segs(I.ny), I.cw[1], R + I.off, scale_m,
                                    U + I.off, local);
}

// u: the previous step's solves (uz, uy, ux, N apart); in the last step of an
// instance (segment 0, j = 0) lambda is the readout adjoint alone.
__global__ __launch_bounds__(kBatchThreads) void kb_lambda(BatchMap m, DenseView v,
                                                           const double *u, long long N,
                                                           const double *ghist, double *U) {
  BatchInst I;
  int local, t;
  if (!batch_locate(m, I, local, t)) return;
  const double *uz = u + I.off;
  const bool last = t + 1 == I.nsteps;
  col_lambda<kBatchSeg, true>(Grid{I.nz, I.ny, I.nx}, offset_view(v, I.off),
                              batch_line_segs(I.nz), I.cw[0], last ? nullptr : uz + 2 * N,
                              uz + N, uz, ghist + I.hoff + (long long)t * I.ny * I.nx,
                              U + I.off, local);
}

// f: base pointers of the concatenated fields; the group's steps are j = m.j to
// m.j + cnt - 1 of the segment
__global__ __launch_bounds__(256) void kb_sens(BatchMap m, const uint8_t *w, AdjGroup f, int cnt) {
  BatchInst I;
  int local, t;
  if (!batch_locate(m, I, local, t)) return;
  const int first = max(0, I.nsteps - (m.ctr[1] + 1) * m.K);  // the segment's first step
  const long long o = I.off;
  f.T += o; f.Tx += o; f.Ty += o; f.u += o;
  f.gM += o; f.gg[0] += o; f.gg[1] += o; f.gg[2] += o;
#pragma unroll
  for (int s = 0; s < kAdjGroup; s++)
    f.gsrc[s] = f.gsrc[s] && t - s == I.src_step ? f.gsrc[s] + o : nullptr;
  const int nbp = (I.nx * I.ny + 255) / 256, kc = local / nbp;
  add_sensitivities(Grid{I.nz, I.ny, I.nx}, w + o, f, min(cnt, t - first + 1),
                    (local - kc * nbp) * 256 + (int)threadIdx.x, kc * kBatchSensPlanes,
                    min((kc + 1) * kBatchSensPlanes, I.nz));
}

hipError_t launch_batch_lambda(const BatchMap &m, int nblocks, const DenseView &v, const double *u,
                               long long N, const double *ghist, double *U, hipStream_t s) {
  hipLaunchKernelGGL(kb_lambda, dim3(nblocks), dim3(kBatchThreads),
                     sizeof(double) * 6 * (size_t)kBatchThreads, s, m, v, u, N, ghist, U);
  return hipGetLastError();
}
hipError_t launch_batch_sens(const BatchMap &m, int nblocks, const DenseView &v, const AdjGroup &f,
                             int cnt, hipStream_t s) {
  hipLaunchKernelGGL(kb_sens, dim3(nblocks), dim3(256), 0, s, m, v.w, f, cnt);
  return hipGetLastError();
}

hipError_t launch_batch_rows(const BatchMap &m, int nblocks, const DenseView &v, const double *Tn,
                             double *Ts, const double *src, double *ck, bool ry, hipStream_t s) {
  if (ry)
    hipLaunchKernelGGL(kb_rows<true>, dim3(nblocks), dim3(kBatchWaves * kWave), 0, s, m, v, Tn,
                       Ts, src, ck);
  else
    hipLaunchKernelGGL(kb_rows<false>, dim3(nblocks), dim3(kBatchWaves * kWave), 0, s, m, v, Tn,
                       Ts, src, ck);
  return hipGetLastError();
}

hipError_t launch_batch_cols(const BatchMap &m, int nblocks, int axis, const DenseView &v,
                             const double *Tn, const double *Y, double *X, double *hist, bool ry,
                             hipStream_t s) {
  const size_t shm = sizeof(double) * 6 * (size_t)kBatchThreads;
  const dim3 grid(nblocks), block(kBatchThreads);
  if (axis == 1 && ry)
    hipLaunchKernelGGL((kb_cols<1, true>), grid, block, shm, s, m, v, Tn, Y, X, hist);
  else if (axis == 1)
    hipLaunchKernelGGL((kb_cols<1, false>), grid, block, shm, s, m, v, Tn, Y, X, hist);
  else
    hipLaunchKernelGGL((kb_cols<0, false>), grid, block, shm, s, m, v, Tn, Y, X, hist);
  return hipGetLastError();
}

hipError_t launch_batch_adj_line(const BatchMap &m, int nblocks, int axis, const DenseView &v,
                                 const double *R, int scale_m, double *U, hipStream_t s) {
  if (axis == 1)
    hipLaunchKernelGGL(kb_cols_adj, dim3(nblocks), dim3(kBatchThreads),
                       sizeof(double) * 6 * (size_t)kBatchThreads, s, m, v, R, scale_m, U);
  else
    hipLaunchKernelGGL(kb_rows_adj, dim3(nblocks), dim3(kBatchWaves * kWave), 0, s, m, v, R,
                       scale_m, U);
  return hipGetLastError();
}

}  // namespace hs2
