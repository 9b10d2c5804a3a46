// Row and column solves on per-voxel coefficients (device code shared by the
// forward sweeps and the adjoint's transposed solves; gfx950, FP64).
#pragma once
#include "hs2_device.h"

namespace hs2 {

// 16-byte accesses to cells whose row may start on any cell: 8-byte alignment
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));

// cells idx .. idx + CPL - 1 of an array of n (one by one at its end)
template <int CPL>
__device__ __forceinline__ void load_cells(const double *__restrict__ a, int idx, int n,
                                           double (&v)[CPL]) {
  if (idx + CPL <= n) {
#pragma unroll
    for (int q = 0; q + 1 < CPL; q += 2) {
      const d2u d = *reinterpret_cast<const d2u *>(a + idx + q);
      v[q] = d.x;
      v[q + 1] = d.y;
    }
    if (CPL & 1) v[CPL - 1] = a[idx + CPL - 1];
  } else {
#pragma unroll
    for (int q = 0; q < CPL; q++) v[q] = a[min(idx + q, n - 1)];
  }
}
// the bytes of up to eight cells, first one lowest
template <int CPL>
__device__ __forceinline__ uint64_t load_bytes(const uint8_t *__restrict__ a, int idx, int n) {
  typename std::conditional<(CPL > 4), uint64_t, uint32_t>::type w = 0;
  if (idx + (int)sizeof w <= n) {
    __builtin_memcpy(&w, a + idx, sizeof w);
    return w;
  }
  uint64_t v = 0;
#pragma unroll
  for (int q = 0; q < CPL; q++) v |= (uint64_t)a[min(idx + q, n - 1)] << (8 * q);
  return v;
}
template <int CPL>
__device__ __forceinline__ void store_cells(double *a, int o, int left, const double (&v)[CPL]) {
  if (left >= CPL) {
#pragma unroll
    for (int q = 0; q + 1 < CPL; q += 2) {
      d2u d;
      d.x = v[q];
      d.y = v[q + 1];
      *reinterpret_cast<d2u *>(a + o + q) = d;
    }
    if (CPL & 1) a[o + CPL - 1] = v[CPL - 1];
  } else {
#pragma unroll
    for (int q = 0; q < CPL; q++)
      if (q < left) a[o + q] = v[q];
  }
}

// lane l of the wave reads lane l-1 (up) or l+1 (down); 0 at the wave's ends
__device__ __forceinline__ double wave_up(double v) { return dpp_d<0x138>(v); }
__device__ __forceinline__ double wave_down(double v) { return dpp_d<0x130>(v); }

// Solve of one line spread over G lanes, CPL >= 2 consecutive rows per lane
// (fed to `s`), into x.  Each lane's rows are reduced to its two end rows; the
// lanes' last unknowns alone are then a tridiagonal system,
//   (1 - Ae Cs - Ce As') x_p - Ae As x_{p-1} - Ce Cs' x_{p+1} = Re - Ae Rs - Ce Rs'
// (primes: the next lane's first row), reduced by PCR across the lanes, and
// the first unknowns follow from them.
template <int CPL, int G>
__device__ __forceinline__ void row_solve(Seg<CPL> &s, double (&x)[CPL], int lig) {
  using X = LaneX<G>;
  double As, Cs, Rs, Ae, Ce, Re;
  s.finish(As, Cs, Rs, Ae, Ce, Re);
  double a = 0.0, c = 0.0, r = Re;
  if (__any(coupling(As, Cs, Ae, Ce) > kNegligible)) {
    const double An = X::down(As, 1, lig), Cn = X::down(Cs, 1, lig), Rn = X::down(Rs, 1, lig);
    const double k = rcp(1.0 - Ae * Cs - Ce * An);
    a = -Ae * As * k;
    c = -Ce * Cn * k;
    r = (Re - Ae * Rs - Ce * Rn) * k;
#pragma unroll
    for (int d = 1; d < G; d <<= 1) {
      // couplings shrink from level to level on a diagonally dominant line:
      // done once none in the wave can change a value
      if (!__any(fmax(fabs(a), fabs(c)) > kNegligible)) break;
      const double aL = X::up(a, d, lig), cL = X::up(c, d, lig), rL = X::up(r, d, lig);
      const double aR = X::down(a, d, lig), cR = X::down(c, d, lig), rR = X::down(r, d, lig);
      pcr_combine(a, c, r, aL, cL, rL, aR, cR, rR);
    }
  }
  const double xb = X::up(r, 1, lig);  // the lane before's last unknown
  x[CPL - 1] = r;
  x[0] = Rs - As * xb - Cs * r;
#pragma unroll
  for (int q = 1; q < CPL - 1; q++) x[q] = s.interior(q, x[0], r);
}

// The same across the threads of a block, one segment each: thread (p, cl) of
// P segments x CW lines holds a segment's end rows; xs, xe: its end values.
// LDS: 6 P CW doubles.  act as in lds_pcr_ends.  Contains barriers.
__device__ __forceinline__ void block_ends(double *lds, int p, int P, int CW, int cl, bool act,
                                           double As, double Cs, double Rs, double Ae, double Ce,
                                           double Re, double &xs, double &xe) {
  __shared__ int wave_more[2][kMaxWaves];
  const int n = P * CW, me = p * CW + cl;
  const int waves = (int)(blockDim.x + kWave - 1) / kWave, wave = threadIdx.x / kWave;
  double *cur = lds, *nxt = lds + 3 * n;
  if (act) {
    cur[me] = As;
    cur[n + me] = Cs;
    cur[2 * n + me] = Rs;
  }
  __syncthreads();
  double a = 0.0, c = 0.0, r = 0.0;
  if (act) {
    const bool last = p + 1 == P;
    const int o = last ? me : me + CW;
    const double An = last ? 0.0 : cur[o], Cn = last ? 0.0 : cur[n + o],
                 Rn = last ? 0.0 : cur[2 * n + o];
    const double k = rcp(1.0 - Ae * Cs - Ce * An);
    a = -Ae * As * k;
    c = -Ce * Cn * k;
    r = (Re - Ae * Rs - Ce * Rn) * k;
  }
  // each level goes to the other buffer, with one barrier; the decision to
  // go on rides on it (every wave posts whether it still has couplings)
  for (int d = 1, turn = 0;; d <<= 1, turn ^= 1) {
    if (act) {
      nxt[me] = a;
      nxt[n + me] = c;
      nxt[2 * n + me] = r;
    }
    const bool more = act && d < P && fmax(fabs(a), fabs(c)) > kNegligible;
    const unsigned long long bal = __ballot(more);
    if ((threadIdx.x & (kWave - 1)) == 0) wave_more[turn][wave] = bal != 0ull;
    __syncthreads();
    int any = 0;
    for (int w = 0; w < waves; w++) any |= wave_more[turn][w];
    if (!any) break;
    if (act) {
      const bool lo = p - d >= 0, hi = p + d < P;
      const int l = lo ? me - d * CW : me, h = hi ? me + d * CW : me;
      const double m0 = lo ? 1.0 : 0.0, m1 = hi ? 1.0 : 0.0;
      pcr_combine(a, c, r, m0 * nxt[l], m0 * nxt[n + l], m0 * nxt[2 * n + l], m1 * nxt[h],
                  m1 * nxt[n + h], m1 * nxt[2 * n + h]);
    }
    double *t = cur;
    cur = nxt;
    nxt = t;
  }
  if (act) {
    xe = r;
    xs = Rs - As * (p > 0 ? nxt[2 * n + me - CW] : 0.0) - Cs * r;
  }
}

}  // namespace hs2
