// Sweeps on line tables (gfx950, FP64); see hs2_lines.h.
#include <algorithm>
#include <cmath>
#include <functional>
#include <vector>

#include "hs2_dense.h"
#include "hs2_lines.h"

namespace hs2 {

// tables read through scalar loads (addresses the same for a whole wave)
typedef const __attribute__((address_space(4))) double *ScalarTab;
typedef const __attribute__((address_space(4))) uint32_t *ScalarIds;

// ------------------------------------------------------------ columns
// value of lane Q of each row of 16 lanes
extern "C" __device__ double hs2_update_dpp_f64(double, double, int, int, int,
                                                bool) __asm("llvm.amdgcn.update.dpp.f64");
template <int Q>
__device__ __forceinline__ double row_bcast(double v) {
  return hs2_update_dpp_f64(0.0, v, 0x150 + Q, 0xF, 0xF, true);
}

// Factors of one line's segment: lane l of a row of 16 lanes keeps cell l's
// (SEG < 16: cell l % SEG's), a cell's come by row broadcast.
template <int SEG>
struct RowCoef {
  double c[kColCoef];
  __device__ __forceinline__ void load(const double *t, int l) {
    const double2 *d = reinterpret_cast<const double2 *>(t + (l % SEG) * kColCoef);
#pragma unroll
    for (int h = 0; h < kColCoef / 2; h++) {
      const double2 v = d[h];
      c[2 * h] = v.x;
      c[2 * h + 1] = v.y;
    }
  }
  template <int Q>
  __device__ __forceinline__ double get(int which) const {
    return row_bcast<Q>(c[which]);
  }
};

template <int SEG, bool RY, int Q = 0>
__device__ __forceinline__ void col_down(const RowCoef<SEG> &c, const double (&d)[SEG + 1],
                                         double (&y)[SEG], double yp) {
  if constexpr (Q < SEG) {
    // what does not wait for y_{Q-1} first: one dependent FMA per cell
    const double l = c.template get<Q>(2);
    double v;
    if constexpr (RY)
      v = c.template get<Q>(1) * y[Q];
    else
      v = c.template get<Q>(0) * y[Q] - l * d[Q] + c.template get<Q>(3) * d[Q + 1];
    y[Q] = __builtin_fma(-l, yp, v);
    col_down<SEG, RY, Q + 1>(c, d, y, y[Q]);
  }
}
template <int SEG, int Q = SEG - 2>
__device__ __forceinline__ void col_up(const RowCoef<SEG> &c, double (&y)[SEG]) {
  if constexpr (Q >= 0) {
    y[Q] -= c.template get<Q>(3) * y[Q + 1];
    col_up<SEG, Q - 1>(c, y);
  }
}
template <int SEG, int Q = 0>
__device__ __forceinline__ void col_join(const RowCoef<SEG> &c, double xl, double xr,
                                         double (&y)[SEG]) {
  if constexpr (Q < SEG) {
    y[Q] -= c.template get<Q>(4) * xl + c.template get<Q>(5) * xr;
    col_join<SEG, Q + 1>(c, xl, xr, y);
  }
}

// xl and xr of every lane's segment from all P segments' end values: lane q
// of the row keeps segment Q0 + q's coefficients
template <int Q0, int Q = 0>
__device__ __forceinline__ void col_reduce(const double *rs, int P, const double *S,
                                           const double *E, int CW, double &xl, double &xr) {
  if constexpr (Q < 16) {
    if (Q0 + Q < P) {
      const double s = S[(Q0 + Q) * CW], e = E[(Q0 + Q) * CW];
      xl += row_bcast<Q>(rs[0]) * s + row_bcast<Q>(rs[1]) * e;
      xr += row_bcast<Q>(rs[2]) * s + row_bcast<Q>(rs[3]) * e;
      col_reduce<Q0, Q + 1>(rs, P, S, E, CW, xl, xr);
    }
  }
}

// y and z sweeps.  Bound by HBM: at 256^3 y 41 us and z 63 us (6.5 and 6.4
// TB/s of their 16 and 24 B per cell; the class kernel, which decodes a byte
// and divides three times per cell, 58 and 77), at 61 x 149 x 203 11.8 and
// 11.0 us (16.9 and 12.6).  The factors cost no memory traffic to speak of and
// no lookups: 12 registers per lane hold the segment's, and the segment keeps
// only its right-hand sides besides (4 waves per SIMD).  Segments of 16 cells
// beat 8 from 65 cells on (96 cells: 14.6 against 19.3 us), 8 beat 4 from 33
// (40^3: 3.6 against 3.9 us) and 16 at 61 cells (11.0 against 14.8).
//
// A block holds 1 << cs groups of 16 columns; a row of 16 lanes holds one
// segment of a group, whose columns are one line.  X may alias Y or T^n: a
// block owns whole columns, and all of its loads happen before its barrier
// and all of its stores after.
// PICK: the groups' columns are listed (t.base), else in memory order.
template <int SEG, int AXIS, bool RY, bool PICK>
__global__ __launch_bounds__(512) void k_cols(Grid g, ColTab t, int cs, const double *Tn,
                                              const double *Y, double *X, double *surf,
                                              double dz) {
  extern __shared__ double lds[];
  const int P = t.P, CW = 16 << cs;
  double *S = lds, *E = lds + P * CW;
  const int l = threadIdx.x & 15, r = threadIdx.x >> 4;
  const int p = r >> cs, cg = r & ((1 << cs) - 1), cl = (cg << 4) + l;
  const int nx = g.nx, ny = g.ny, nz = g.nz;
  const int L = AXIS == 1 ? ny : nz, stride = AXIS == 1 ? nx : nx * ny;
  const int group = (xcd_remap_chunks<64>(blockIdx.x, gridDim.x) << cs) + cg;
  const int gc = min(group, t.groups - 1);
  int base;
  bool valid;
  if constexpr (PICK) {
    const int id = t.base[gc * 16 + l];
    valid = id >= 0 && group < t.groups;
    base = id & 0x7fffffff;
  } else {
    const int ncol = nx * (AXIS == 1 ? nz : ny), col = group * 16 + l;
    valid = col < ncol;
    base = min(col, ncol - 1);
    if (AXIS == 1) {
      const int k = base / nx;
      base = k * ny * nx + (base - k * nx);
    }
  }
  const int line = t.pid[gc];
  const int t0 = p * SEG;
  const unsigned bytes = (unsigned)nx * (unsigned)ny * (unsigned)nz * 8u;  // below 4 GiB
  const BufRsrc bT = make_buf(Tn, bytes), bY = make_buf(Y, bytes), bX = make_buf(X, bytes);
  const unsigned so = (unsigned)stride * 8u, vo = (unsigned)base * 8u + (unsigned)t0 * so;
  // Rows past the line's end read what follows it in the array, or 0 past the
  // array's end (the buffer's bound, which holds for the lane's offset but not
  // for a scalar one: the row offset is added to the former); they are cleared
  // below.
  double d[SEG + 1], y[SEG];  // differences of T^n across the rows' faces
  if constexpr (!RY) {
    double T[SEG + 2];
    T[0] = buf_load_d(bT, t0 > 0 ? vo - so : vo);
#pragma unroll
    for (int q = 0; q <= SEG; q++) T[q + 1] = buf_load_d(bT, vo + q * so);
#pragma unroll
    for (int q = 0; q <= SEG; q++) d[q] = T[q + 1] - T[q];
  }
#pragma unroll
  for (int q = 0; q < SEG; q++) y[q] = buf_load_d(bY, vo + q * so);
  const bool whole = t0 + SEG <= L;
  if (t0 + SEG >= L) {
    if constexpr (!RY) {
#pragma unroll
      for (int q = 0; q <= SEG; q++) d[q] = t0 + q < L ? d[q] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < SEG; q++) y[q] = t0 + q < L ? y[q] : 0.0;
  }
  RowCoef<SEG> rc;
  rc.load(t.coef + ((size_t)line * P + p) * SEG * kColCoef, l);
  // the coefficients of xl and xr: the neighbouring segments' where no others
  // matter, else lane q segment q's (and 16 + q's)
  const double *red = t.red + ((size_t)line * P + p) * P * 4;
  const bool near = t.band <= 1;
  double rd[12];
  if (near) {
#pragma unroll
    for (int o = 0; o < 3; o++) {
      const double2 *c = reinterpret_cast<const double2 *>(red + min(max(p + o - 1, 0), P - 1) * 4);
      const double2 a = c[0], b = c[1];
      rd[4 * o] = a.x;
      rd[4 * o + 1] = a.y;
      rd[4 * o + 2] = b.x;
      rd[4 * o + 3] = b.y;
    }
  } else {
#pragma unroll
    for (int o = 0; o < 2; o++) {
      const double2 *c = reinterpret_cast<const double2 *>(red + min(l + 16 * o, P - 1) * 4);
      const double2 a = c[0], b = c[1];
      rd[4 * o] = a.x;
      rd[4 * o + 1] = a.y;
      rd[4 * o + 2] = b.x;
      rd[4 * o + 3] = b.y;
    }
  }
  col_down<SEG, RY>(rc, d, y, 0.0);
  col_up<SEG>(rc, y);
  S[p * CW + cl] = y[0];
  E[p * CW + cl] = y[SEG - 1];
  __syncthreads();
  double xl = 0.0, xr = 0.0;
  if (near) {
#pragma unroll
    for (int o = 0; o < 3; o++) {
      const int j = p + o - 1, jc = min(max(j, 0), P - 1);
      const double s = j == jc ? S[jc * CW + cl] : 0.0, e = j == jc ? E[jc * CW + cl] : 0.0;
      xl += rd[4 * o] * s + rd[4 * o + 1] * e;
      xr += rd[4 * o + 2] * s + rd[4 * o + 3] * e;
    }
  } else {
    col_reduce<0>(rd, P, S + cl, E + cl, CW, xl, xr);
    col_reduce<16>(rd + 4, P, S + cl, E + cl, CW, xl, xr);
  }
  col_join<SEG>(rc, xl, xr, y);
  if (!valid) return;
  if (whole) {
#pragma unroll
    for (int q = 0; q < SEG; q++) buf_store_ds(y[q], bX, vo, q * so);
  } else {
#pragma unroll
    for (int q = 0; q < SEG; q++)
      if (t0 + q < L) buf_store_ds(y[q], bX, vo, q * so);
  }
  if (AXIS == 0 && surf && p == 0 && L >= 2) surf[base] = surface_readout(y[0], y[1], dz);
}

// --------------------------------------------------------------- rows
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_rows(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffLL), CTRL, ROWS, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xF, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ double read_lane(double v, int l) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), l);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Inclusive scan of y_p += f y_{p-1} over the lanes of each group of G: inside
// rows of 16 lanes by doubling (the factors double along), then from the
// rows' last lanes, with the products up to this lane from the start of its
// row (f[1]) and from lane 32 (f[2]).  `on`: the steps whose factors matter.
template <int G>
__device__ __forceinline__ double scan_up(double v, const double *f, unsigned on) {
  if (on & 1u) v += f[0] * dpp_d<0x111>(v);
  if (on & 2u) {
    const double f2 = f[0] * dpp_d<0x111>(f[0]);
    v += f2 * dpp_d<0x112>(v);
    if (on & 4u) {
      const double f4 = f2 * dpp_d<0x112>(f2);
      v += f4 * dpp_d<0x114>(v);
      if (on & 8u) v += f4 * dpp_d<0x114>(f4) * dpp_d<0x118>(v);
    }
  }
  if (G >= 32 && (on & 16u)) v += f[1] * dpp_rows<0x142, 0xA>(v);  // row_bcast:15
  if (G >= 64 && (on & 32u)) v += f[2] * dpp_rows<0x143, 0xC>(v);  // row_bcast:31
  return v;
}
// the same from above: x_p += b x_{p+1}
template <int G>
__device__ __forceinline__ double scan_down(double v, const double *b, unsigned on, int lane) {
  if (on & 1u) v += b[0] * dpp_d<0x101>(v);
  if (on & 2u) {
    const double b2 = b[0] * dpp_d<0x101>(b[0]);
    v += b2 * dpp_d<0x102>(v);
    if (on & 4u) {
      const double b4 = b2 * dpp_d<0x102>(b2);
      v += b4 * dpp_d<0x104>(v);
      if (on & 8u) v += b4 * dpp_d<0x104>(b4) * dpp_d<0x108>(v);
    }
  }
  if (G >= 32 && (on & 16u)) {
    const double lo = read_lane(v, 16), hi = read_lane(v, 48);
    const double in = (lane & 32) ? hi : lo;
    v += b[1] * ((lane & 16) ? 0.0 : in);
  }
  if (G >= 64 && (on & 32u)) {
    const double in = read_lane(v, 32);
    v += b[2] * ((lane & 32) ? 0.0 : in);
  }
  return v;
}

// x sweep: a wave holds 64/G neighbouring rows, G lanes x CPL consecutive
// cells each, or W waves hold one row (G = 64), in registers, and walks KC
// planes: a row's own cells and the plane's before it are carried, so a row
// costs three row loads (y-1, y+1 and the next plane) and one store.  No
// right-hand side is staged and no class byte is read.  Bound by the row
// loads through L1 and L2 at large sizes (256^3: 56 us, 4.8 TB/s of 16 B per
// cell, against 72 for the staged class kernel; 128 x 512 x 512: 137 us
// against 198), by latency at small ones (61 x 149 x 203: 12.1 against 25
// us, 40^3: 3.8 against 5.6).  The factors are read from LDS for every row: in
// registers they cost a wave per SIMD (61 us at 256^3).  Lanes of more than 6
// cells do worse than two waves per row (512 cells: 178 us against 145 then): their
// loads are 64 bytes apart, and too few waves fit; rows put in lane order
// through LDS made whole-line loads and stores of it (170 us there, but 60 at
// 256^3).  Waves in flight weigh most: two rows to a wave (a third of the row
// loads saved, 160 registers) take 69 us at 256^3 and 170 at 512 cells; the next
// plane's rows loaded during the solve 55 and 151; five waves per SIMD in 96
// registers 58 and 156.
template <int CPL, int G, int W, bool SRC, bool RY>
__global__ __launch_bounds__(256) void k_rows(Grid g, RowTab t, const double *__restrict__ Tn,
                                              double *__restrict__ Ts,
                                              const uint8_t *__restrict__ vmap,
                                              const double *__restrict__ vtab_g,
                                              const double *__restrict__ sfield, int KC) {
  static_assert(CPL <= 6 && (W == 1 || G == kWave), "");
  constexpr int LPW = kWave / G, RPB = 4 / W;  // rows per wave; row groups per block
  constexpr int GL = G * W;                    // lanes of a row
  constexpr int NP = row_pairs(CPL);
  // the first `nlds` lines' factors, then the source table
  extern __shared__ double lds[];
  __shared__ double2 carry[W > 1 ? 2 : 1][4];  // W > 1: the waves' carries, up and down
  double *vtab = lds + (size_t)t.nlds * NP * GL * 2;
  const int nx = g.nx, ny = g.ny, nz = g.nz;
  const int n = nx * ny * nz;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), wr = wave % W;
  const int lig = lane % G + wr * kWave;  // lane of the row
  const int nj = (ny + LPW - 1) / LPW, units = nj * ((nz + KC - 1) / KC);
  const int unit = xcd_remap(blockIdx.x, gridDim.x) * RPB + wave / W;
  const int uc = min(unit, units - 1);
  const int kc = uc / nj, jg = uc - kc * nj;
  const int jr = jg * LPW + lane / G;
  const bool jv = jr < ny && unit < units;
  const int j = min(jr, ny - 1);
  const int i0 = lig * CPL;
  // where a lane reads: one partly past the row's end reads on into what
  // follows it (masked below), one wholly past it the row's last cells again
  const int ir = i0 < nx ? i0 : max(0, nx - CPL);
  const int ym = j > 0 ? j - 1 : j, yp = min(j + 1, ny - 1);
  // every wave of a block walks KC planes, the last ones past the grid's end
  // stay on its last plane (W > 1) and store nothing
  const int k0 = kc * KC, k1 = min(k0 + KC, nz), ke = W > 1 ? k0 + KC : k1;
  auto load = [&](int k, int jj, double(&v)[CPL]) {
    load_cells<CPL>(Tn, (k * ny + jj) * nx + ir, n, v);
  };
  auto row_id = [&](int k) -> uint32_t {
    if constexpr (G == kWave) return ((ScalarIds)(uintptr_t)t.pid)[k * ny + j];
    else return t.pid[k * ny + j];
  };
  double Tm[CPL], T[CPL], Tp[CPL];
  load(k0 > 0 ? k0 - 1 : k0, j, Tm);
  load(k0, j, T);
  // (behind the wave's own first loads: the two wait together)
  for (int e = threadIdx.x; e < t.nlds * NP * GL; e += 256)
    reinterpret_cast<double2 *>(lds)[e] = reinterpret_cast<const double2 *>(t.lane)[e];
  if (SRC && vmap)
    for (int e = threadIdx.x; e < kMaxVtab; e += 256) vtab[e] = vtab_g[e];
  __syncthreads();
  if (W == 1 && unit >= units) return;  // W > 1: the block's waves meet at barriers
  uint32_t erow = ~0u;
  double ex[kRowExpl];
  for (int kk = k0; kk < ke; kk++) {
    const int k = min(kk, nz - 1);
    const int o = (k * ny + j) * nx + i0;
    double Tym[CPL], Typ[CPL];
    load(k, ym, Tym);
    load(k, yp, Typ);
    load(min(k + 1, nz - 1), j, Tp);
    [[maybe_unused]] uint64_t cls = 0;
    [[maybe_unused]] double S[CPL] = {};
    if constexpr (SRC) {
      if (vmap) cls = load_bytes<CPL>(vmap, (k * ny + j) * nx + ir, n);
      if (sfield) load_cells<CPL>(sfield, (k * ny + j) * nx + ir, n, S);
    }
    double TL = wave_up(T[CPL - 1]), TR = wave_down(T[0]);
    if constexpr (W > 1) {  // the neighbouring waves' cells
      if (lane == 0 && wr > 0 && i0 < nx) TL = Tn[o - 1];
      if (lane == kWave - 1 && i0 + CPL < nx) TR = Tn[o + CPL];
    }
    const uint32_t id = row_id(k);
    const bool vary = __any((id >> 16) & kRowVaries);
    if (G == kWave) {
      erow = id >> 16;
      const ScalarTab c = (ScalarTab)(uintptr_t)(t.row + (size_t)(vary ? 0 : erow) * kRowExpl);
#pragma unroll
      for (int q = 0; q < kRowExpl; q++) ex[q] = c[q];
    } else if (__any((id >> 16) != erow)) {
      erow = id >> 16;
      const double *c = t.row + (size_t)((erow & kRowVaries) ? 0 : erow) * kRowExpl;
#pragma unroll
      for (int q = 0; q < kRowExpl; q++) ex[q] = c[q];
    }
    double r[CPL], ly[CPL];
    // a varying row's own numbers, cell by cell
    const double *cell = t.cell + ((size_t)(erow & ~kRowVaries) * (GL * CPL) + i0) * kRowExpl;
    const bool mine = erow & kRowVaries;
    if (!vary) {
#pragma unroll
      for (int q = 0; q < CPL; q++) {
        ly[q] = ex[1] * (Tym[q] - T[q]) + ex[2] * (Typ[q] - T[q]);
        r[q] = ex[0] * T[q] + ly[q] + (ex[3] * (Tm[q] - T[q]) + ex[4] * (Tp[q] - T[q]));
      }
    } else {
#pragma unroll
      for (int q = 0; q < CPL; q++) {
        const double *c = mine ? cell + q * kRowExpl : t.row + (size_t)erow * kRowExpl;
        ly[q] = c[1] * (Tym[q] - T[q]) + c[2] * (Typ[q] - T[q]);
        r[q] = c[0] * T[q] + ly[q] + (c[3] * (Tm[q] - T[q]) + c[4] * (Tp[q] - T[q]));
        asm volatile("" ::: "memory");  // the next cell's loads stay after this one's
      }
    }
    if constexpr (SRC) {
#pragma unroll
      for (int q = 0; q < CPL; q++) {
        const double s = vmap ? S[q] + vtab[(cls >> (8 * q)) & 0xffu] : S[q];
        r[q] += (mine ? cell[q * kRowExpl + 5] : ex[5]) * s;
      }
    }
    // the line's factors: inv, l, u per cell, then the scans'
    double c[2 * NP];
    const uint32_t line = id & 0xffffu;
    if (!__any(line >= (uint32_t)t.nlds)) {
      const double2 *d = reinterpret_cast<const double2 *>(lds) + (size_t)line * NP * GL + lig;
#pragma unroll
      for (int h = 0; h < NP; h++) {
        const double2 v = d[h * GL];
        c[2 * h] = v.x;
        c[2 * h + 1] = v.y;
      }
    } else {
      const double2 *d = reinterpret_cast<const double2 *>(t.lane) + (size_t)line * NP * GL + lig;
#pragma unroll
      for (int h = 0; h < NP; h++) {
        const double2 v = d[h * GL];
        c[2 * h] = v.x;
        c[2 * h + 1] = v.y;
      }
    }
    const double *inv = c, *l = c + CPL, *u = c + 2 * CPL, *f = c + 3 * CPL, *b = f + kRowScan;
    // y_i = r_i/piv_i - l_i y_{i-1}, the x faces' explicit half folded in
    double Y = 0.0;
#pragma unroll
    for (int q = 0; q < CPL; q++) {
      const bool in = i0 + q < nx;
      const double dm = q > 0 ? T[q - 1] - T[q] : lig > 0 ? TL - T[q] : 0.0;
      const double tr = q < CPL - 1 ? T[q + 1] : TR;
      const double dp = i0 + q + 1 < nx ? tr - T[q] : 0.0;
      r[q] = in ? inv[q] * r[q] - l[q] * dm - u[q] * dp : 0.0;
      Y = r[q] - l[q] * Y;
    }
    Y = scan_up<G>(Y, f, t.scan);
    double in = wave_up(Y);
    if (lane % G == 0) in = 0.0;
    if constexpr (W > 1) {
      // f[3]: the product from the wave's first lane.  A wave's carry in is
      // the waves' before it, each shrunk by those between
      if (lane == kWave - 1) carry[0][wave] = make_double2(Y, f[3]);
      __syncthreads();
      double c0 = 0.0;
#pragma unroll
      for (int w = 0; w < W - 1; w++)
        if (w < wr) {
          const double2 v = carry[0][wave - wr + w];
          c0 = v.x + v.y * c0;
        }
      const double up = wave_up(f[3]);
      in += (lane == 0 ? 1.0 : up) * c0;
    }
#pragma unroll
    for (int q = 0; q < CPL; q++) {
      r[q] -= l[q] * in;
      in = r[q];
    }
    double Xs = r[CPL - 1];
#pragma unroll
    for (int q = CPL - 2; q >= 0; q--) Xs = r[q] - u[q] * Xs;
    Xs = scan_down<G>(Xs, b, t.scan >> 8, lane);
    in = wave_down(Xs);
    if (lane % G == G - 1) in = 0.0;
    if constexpr (W > 1) {
      if (lane == 0) carry[1][wave] = make_double2(Xs, b[3]);
      __syncthreads();
      double c0 = 0.0;
#pragma unroll
      for (int w = W - 1; w > 0; w--)
        if (w > wr) {
          const double2 v = carry[1][wave - wr + w];
          c0 = v.x + v.y * c0;
        }
      const double dn = wave_down(b[3]);
      in += (lane == kWave - 1 ? 1.0 : dn) * c0;
    }
#pragma unroll
    for (int q = CPL - 1; q >= 0; q--) {
      r[q] -= u[q] * in;
      in = r[q];
    }
    if constexpr (RY) {
      if (!vary) {
#pragma unroll
        for (int q = 0; q < CPL; q++) r[q] = ex[0] * r[q] - 0.5 * ly[q];
      } else {
#pragma unroll
        for (int q = 0; q < CPL; q++)
          r[q] = (mine ? cell[q * kRowExpl] : ex[0]) * r[q] - 0.5 * ly[q];
      }
    }
    if (jv && kk < k1) {
      if (i0 + CPL <= nx) {
#pragma unroll
        for (int q = 0; q + 1 < CPL; q += 2) {
          d2u d;
          d.x = r[q];
          d.y = r[q + 1];
          *reinterpret_cast<d2u *>(Ts + o + q) = d;
        }
        if (CPL & 1) Ts[o + CPL - 1] = r[CPL - 1];
      } else {
#pragma unroll
        for (int q = 0; q < CPL; q++)
          if (i0 + q < nx) Ts[o + q] = r[q];
      }
    }
#pragma unroll
    for (int q = 0; q < CPL; q++) {
      Tm[q] = T[q];
      T[q] = Tp[q];
    }
  }
}

// ------------------------------------------------- telling lines apart
// the finaliser of SplitMix64 (Steele, Lea, Flood 2014)
__device__ __forceinline__ unsigned long long mix64(unsigned long long x) {
  x ^= x >> 30;
  x *= 0xbf58476d1ce4e5b9ull;
  x ^= x >> 27;
  x *= 0x94d049bb133111ebull;
  return x ^ (x >> 31);
}

// byte t of line `ln` (which as in launch_line_hash); for which == 3, t runs
// over five sequences of nx bytes
__device__ __forceinline__ int line_byte(const Grid &g, const uint8_t *cz, const uint8_t *cy,
                                         const uint8_t *cx, int which, int ln, int t) {
  const int nx = g.nx, ny = g.ny, nz = g.nz, sxy = nx * ny;
  if (which == 0) return cz[ln + t * sxy];
  if (which == 1) {
    const int k = ln / nx;
    return cy[k * sxy + (ln - k * nx) + t * nx];
  }
  if (which == 2) return cx[ln * nx + t];
  const int k = ln / ny, j = ln - k * ny;
  const int s = t / nx, c = ln * nx + (t - s * nx);
  switch (s) {
    case 0: return cx[c];
    case 1: return cy[c];
    case 2: return j < ny - 1 ? cy[c + nx] : 256;
    case 3: return cz[c];
    default: return k < nz - 1 ? cz[c + sxy] : 256;
  }
}

__device__ __forceinline__ int line_len(const Grid &g, int which) {
  return which == 0 ? g.nz : which == 1 ? g.ny : which == 2 ? g.nx : 5 * g.nx;
}
static int line_count(const Grid &g, int which) {
  return which == 0 ? g.ny * g.nx : which == 1 ? g.nz * g.nx : g.nz * g.ny;
}

// columns: a thread each (coalesced across them); rows: a wave each
__global__ __launch_bounds__(256) void k_line_hash(Grid g, const uint8_t *cz, const uint8_t *cy,
                                                   const uint8_t *cx, int which, int count,
                                                   unsigned long long *out) {
  const int tid = blockIdx.x * blockDim.x + threadIdx.x;
  const bool rows = which >= 2;
  const int ln = rows ? tid / kWave : tid;
  if (ln >= count) return;
  const int L = line_len(g, which);
  unsigned long long h0 = 0, h1 = 0;
  for (int t = rows ? tid % kWave : 0; t < L; t += rows ? kWave : 1) {
    const unsigned long long v =
        ((unsigned long long)(t + 1) << 9) | (unsigned)line_byte(g, cz, cy, cx, which, ln, t);
    h0 += mix64(v);
    h1 += mix64(v ^ 0x9e3779b97f4a7c15ull);
  }
  if (rows) {
    for (int d = kWave / 2; d > 0; d >>= 1) {
      h0 += __shfl_down(h0, d, kWave);
      h1 += __shfl_down(h1, d, kWave);
    }
    if (tid % kWave) return;
  }
  out[2 * (size_t)ln] = h0;
  out[2 * (size_t)ln + 1] = h1;
}

__global__ __launch_bounds__(256) void k_line_check(Grid g, const uint8_t *cz, const uint8_t *cy,
                                                    const uint8_t *cx, int which, int count,
                                                    const int *rep, int *flag) {
  const int tid = blockIdx.x * blockDim.x + threadIdx.x;
  const bool rows = which >= 2;
  const int ln = rows ? tid / kWave : tid;
  if (ln >= count) return;
  const int L = line_len(g, which), other = rep[ln];
  if (other == ln) return;
  bool bad = false;
  for (int t = rows ? tid % kWave : 0; t < L; t += rows ? kWave : 1)
    bad |= line_byte(g, cz, cy, cx, which, ln, t) != line_byte(g, cz, cy, cx, which, other, t);
  if (bad) *flag = 1;
}

__global__ __launch_bounds__(256) void k_line_gather(Grid g, const uint8_t *cz, const uint8_t *cy,
                                                     const uint8_t *cx, int which, const int *line,
                                                     int count, uint8_t *out) {
  const int L = line_len(g, which);
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < count * L;
       e += gridDim.x * blockDim.x) {
    const int q = e / L;
    out[e] = (uint8_t)line_byte(g, cz, cy, cx, which, line[q], e - q * L);
  }
}

hipError_t launch_line_hash(const Grid &g, const uint8_t *cz, const uint8_t *cy,
                            const uint8_t *cx, int which, unsigned long long *out, hipStream_t s) {
  const int count = line_count(g, which);
  const long long threads = (long long)count * (which >= 2 ? kWave : 1);
  hipLaunchKernelGGL(k_line_hash, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, g, cz,
                     cy, cx, which, count, out);
  return hipGetLastError();
}
hipError_t launch_line_check(const Grid &g, const uint8_t *cz, const uint8_t *cy,
                             const uint8_t *cx, int which, const int *rep, int *flag,
                             hipStream_t s) {
  const int count = line_count(g, which);
  const long long threads = (long long)count * (which >= 2 ? kWave : 1);
  hipLaunchKernelGGL(k_line_check, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, g, cz,
                     cy, cx, which, count, rep, flag);
  return hipGetLastError();
}
hipError_t launch_line_gather(const Grid &g, const uint8_t *cz, const uint8_t *cy,
                              const uint8_t *cx, int which, const int *line, int count,
                              uint8_t *out, hipStream_t s) {
  hipLaunchKernelGGL(k_line_gather, dim3(256), dim3(256), 0, s, g, cz, cy, cx, which, line, count,
                     out);
  return hipGetLastError();
}

// ---------------------------------------------------------- factors
// in extended precision on the host, rounded once: the same factors act on
// every step, so their errors would add up
typedef long double Wide;

// rows of one line: a = -w g-/2, c = -w g+/2, b = M - a - c
static void line_rows(int L, const double *M, const double *w, const double *g,
                      std::vector<Wide> &a, std::vector<Wide> &b, std::vector<Wide> &c) {
  a.resize(L);
  b.resize(L);
  c.resize(L);
  for (int t = 0; t < L; t++) {
    a[t] = t > 0 ? -0.5 * w[t] * g[t] : 0.0;
    c[t] = t + 1 < L ? -0.5 * w[t] * g[t + 1] : 0.0;
    b[t] = M[t] - a[t] - c[t];
  }
}

void factor_column(int L, int seg, int P, const double *M, const double *w, const double *g,
                   double *coef, double *red, int *band) {
  std::vector<Wide> a, b, c, u(seg), v(seg), piv(seg);
  line_rows(L, M, w, g, a, b, c);
  std::fill(coef, coef + (size_t)P * seg * kColCoef, 0.0);
  std::vector<Wide> ends((size_t)P * 4, 0.0);  // V, W of each segment's first and last cell
  for (int p = 0; p < P; p++) {
    const int t0 = p * seg, m = std::min(seg, L - t0);
    double *k = coef + (size_t)p * seg * kColCoef;
    for (int q = 0; q < m; q++) {
      const int t = t0 + q;
      piv[q] = q > 0 ? b[t] - a[t] * u[q - 1] : b[t];
      u[q] = c[t] / piv[q];
      k[q * kColCoef] = M[t] / piv[q];
      k[q * kColCoef + 1] = 1.0L / piv[q];
      k[q * kColCoef + 2] = a[t] / piv[q];
      k[q * kColCoef + 3] = u[q];
    }
    // responses of the segment to its neighbours: A V = a_0 e_0, A W = c_last e_last
    for (int side = 0; side < 2; side++) {
      for (int q = 0; q < m; q++) {
        const Wide r = side == 0 ? (q == 0 ? a[t0] : 0.0) : (q == m - 1 ? c[t0 + q] : 0.0);
        v[q] = (r - (q > 0 ? a[t0 + q] * v[q - 1] : 0.0L)) / piv[q];
      }
      for (int q = m - 2; q >= 0; q--) v[q] -= u[q] * v[q + 1];
      for (int q = 0; q < m; q++) k[q * kColCoef + 4 + side] = v[q];
      ends[p * 4 + side] = v[0];
      ends[p * 4 + 2 + side] = v[m - 1];
    }
    if (m < seg) {
      // the kernel's end value is cell seg-1's, an identity row's zero, in
      // the line's last, short segment: nothing lies after it
      ends[p * 4 + 2] = ends[p * 4 + 3] = 0.0;
    }
  }
  // first and last cell of every segment from the segments' own end values:
  //   f_p + V_first g_{p-1} + W_first f_{p+1} = s_p
  //   g_p + V_last  g_{p-1} + W_last  f_{p+1} = e_p     (2P x 2P, dense)
  const int n = 2 * P;
  std::vector<Wide> A((size_t)n * 2 * n, 0.0);
  for (int p = 0; p < P; p++)
    for (int h = 0; h < 2; h++) {
      Wide *row = &A[(size_t)(2 * p + h) * 2 * n];
      row[2 * p + h] = 1.0;
      if (p > 0) row[2 * (p - 1) + 1] += ends[p * 4 + 2 * h];
      if (p + 1 < P) row[2 * (p + 1)] += ends[p * 4 + 2 * h + 1];
      row[n + 2 * p + h] = 1.0;
    }
  for (int i = 0; i < n; i++) {
    int best = i;
    for (int r = i + 1; r < n; r++)
      if (std::fabs(A[(size_t)r * 2 * n + i]) > std::fabs(A[(size_t)best * 2 * n + i])) best = r;
    if (best != i)
      for (int j = 0; j < 2 * n; j++) std::swap(A[(size_t)i * 2 * n + j], A[(size_t)best * 2 * n + j]);
    const Wide d = 1.0L / A[(size_t)i * 2 * n + i];
    for (int j = 0; j < 2 * n; j++) A[(size_t)i * 2 * n + j] *= d;
    for (int r = 0; r < n; r++) {
      const Wide m = A[(size_t)r * 2 * n + i];
      if (r == i || m == 0.0) continue;
      for (int j = i; j < 2 * n; j++) A[(size_t)r * 2 * n + j] -= m * A[(size_t)i * 2 * n + j];
    }
  }
  for (int p = 0; p < P; p++)
    for (int j = 0; j < P; j++) {
      double *r = red + ((size_t)p * P + j) * 4;
      for (int h = 0; h < 2; h++) {
        r[h] = p > 0 ? A[(size_t)(2 * (p - 1) + 1) * 2 * n + n + 2 * j + h] : 0.0;
        r[2 + h] = p + 1 < P ? A[(size_t)(2 * (p + 1)) * 2 * n + n + 2 * j + h] : 0.0;
      }
      for (int h = 0; h < 4; h++)
        if (std::fabs(r[h]) >= kNegligible) *band = std::max(*band, std::abs(j - p));
    }
}

void factor_row(int nx, int cpl, int G, const double *M, const double *w, const double *g,
                double *lane, unsigned *scan) {
  std::vector<Wide> a, b, c, l(nx), u(nx);
  line_rows(nx, M, w, g, a, b, c);
  const int np = row_pairs(cpl);
  std::fill(lane, lane + (size_t)G * np * 2, 0.0);
  // number c of lane p (pairs of numbers side by side over the lanes)
  auto at = [&](int p, int c) -> double & { return lane[((size_t)(c / 2) * G + p) * 2 + c % 2]; };
  std::vector<Wide> lf(G, 1.0), lb(G, 1.0);  // transfer factors of each lane
  for (int i = 0; i < nx; i++) {
    const Wide piv = i > 0 ? b[i] - a[i] * u[i - 1] : b[i];
    l[i] = a[i] / piv;
    u[i] = c[i] / piv;
    at(i / cpl, i % cpl) = 1.0L / piv;
    at(i / cpl, cpl + i % cpl) = l[i];
    at(i / cpl, 2 * cpl + i % cpl) = u[i];
  }
  for (int p = 0; p < G; p++)
    for (int q = 0; q < cpl; q++) {
      const int i = p * cpl + q;
      lf[p] *= i < nx ? -l[i] : 0.0;
      lb[p] *= i < nx ? -u[i] : 0.0;
    }
  for (int p = 0; p < G; p++) {
    double f[kRowScan] = {(double)lf[p]}, r[kRowScan] = {(double)lb[p]};
    const int row = p / 16 * 16, w0 = p / 64 * 64;  // first lane of this lane's 16, of its wave
    auto up = [&](int from, int to) {
      Wide v = 1.0L;
      for (int e = from; e <= to; e++) v *= lf[e];
      return (double)v;
    };
    auto down = [&](int from, int to) {
      Wide v = 1.0L;
      for (int e = from; e <= std::min(to, G - 1); e++) v *= lb[e];
      return (double)v;
    };
    for (int s = 0; s < 4; s++) {  // the steps inside rows of 16 lanes
      const int d = 1 << s;
      if (p - d >= row && std::fabs(up(p - d + 1, p)) >= kNegligible) *scan |= 1u << s;
      if (p + d < row + 16 && std::fabs(down(p, p + d - 1)) >= kNegligible) *scan |= 256u << s;
    }
    // rows 1 and 3 of a wave take the last lane of rows 0 and 2; rows 2 and 3
    // lane 31; rows 0 and 2 the first lane of rows 1 and 3; rows 0 and 1 lane
    // 32; and the whole wave what the waves beside it carry
    if ((row / 16) & 1) f[1] = up(row, p);
    else if (G > 16) r[1] = down(p, row + 15);
    if (p - w0 >= 32) f[2] = up(w0 + 32, p);
    else if (G > 32) r[2] = down(p, w0 + 31);
    f[3] = up(w0, p);
    r[3] = down(p, w0 + 63);
    for (int h = 1; h < 3; h++) {
      if (std::fabs(f[h]) >= kNegligible) *scan |= 8u << h;
      if (std::fabs(r[h]) >= kNegligible) *scan |= 2048u << h;
    }
    for (int h = 0; h < kRowScan; h++) {
      at(p, 3 * cpl + h) = f[h];
      at(p, 3 * cpl + kRowScan + h) = r[h];
    }
  }
}

int group_columns(int ncol, const std::vector<int> &id, const std::function<int(int)> &base,
                  std::vector<int> *idx, std::vector<uint16_t> *line) {
  idx->clear();
  line->clear();
  for (int w = 0; w < ncol; w += kColWindow) {
    const int e = std::min(ncol, w + kColWindow);
    bool taken[kColWindow] = {};
    for (int c = w; c < e; c++) {
      if (taken[c - w]) continue;
      int in = 0;  // columns of line id[c] left in the window, 16 to a group
      for (int o = c; o < e; o++) {
        if (taken[o - w] || id[o] != id[c]) continue;
        taken[o - w] = true;
        if (in++ % 16 == 0) line->push_back((uint16_t)id[c]);
        idx->push_back(base(o));
      }
      const int last = idx->back();
      for (; in % 16; in++) idx->push_back((int)(0x80000000u | (unsigned)last));
    }
  }
  return (int)line->size();
}

// ---------------------------------------------------------- launchers
void row_shape(int nx, int *cpl, int *g) {
  *g = nx <= 64 ? 16 : nx <= 128 ? 32 : nx <= 384 ? 64 : nx <= 512 ? 128 : 256;
  *cpl = (nx + *g - 1) / *g;
  if (nx > 1024) *g = *cpl = 0;
}

void col_shape(int L, int *seg, int *P) {  // see k_cols
  *seg = L <= 32 ? 4 : L <= 64 ? 8 : 16;
  *P = (L + *seg - 1) / *seg;
  if (*P > kColMaxSegs) *seg = *P = 0;
}

template <int CPL, int GL>
static hipError_t launch_rows_t(const Grid &g, const RowTab &t, const double *Tn, double *Ts,
                                const uint8_t *vmap, const double *vtab, const double *sfield,
                                bool ry, hipStream_t s) {
  constexpr int G = GL < kWave ? GL : kWave, W = GL / G;
  constexpr int LPW = kWave / G, RPB = 4 / W;
  const long long nj = (g.ny + LPW - 1) / LPW;
  // planes per wave: as many as still leave each CU about 16 waves (160 x 224
  // cells x 96 planes: 4 planes 16.8 us, 2 18.8, 7 20.6)
  const int KC = (int)std::min<long long>(16, (nj * W * g.nz + 4095) / 4096);
  const long long units = nj * ((g.nz + KC - 1) / KC);
  const dim3 grid((unsigned)((units + RPB - 1) / RPB)), block(256);
  const bool src = vmap || sfield;
  const size_t shm = sizeof(double) * ((size_t)t.nlds * row_pairs(CPL) * GL * 2 + (vmap ? kMaxVtab : 0));
#define HS2_RUN(SRC, RY)                                                                        \
  hipLaunchKernelGGL((k_rows<CPL, G, W, SRC, RY>), grid, block, shm, s, g, t, Tn, Ts, vmap, vtab, \
                     sfield, KC)
  if (src && ry) HS2_RUN(true, true);
  else if (src) HS2_RUN(true, false);
  else if (ry) HS2_RUN(false, true);
  else HS2_RUN(false, false);
#undef HS2_RUN
  return hipGetLastError();
}

hipError_t launch_rows(const Grid &g, const RowTab &t, const double *Tn, double *Ts,
                       const uint8_t *vmap, const double *vtab, const double *sfield, bool ry,
                       hipStream_t s) {
#define HS2_ROW(C, GG)           \
  if (t.cpl == C && t.g == GG)   \
    return launch_rows_t<C, GG>(g, t, Tn, Ts, vmap, vtab, sfield, ry, s);
  HS2_ROW(1, 16) HS2_ROW(2, 16) HS2_ROW(3, 16) HS2_ROW(4, 16) HS2_ROW(3, 32) HS2_ROW(4, 32)
  HS2_ROW(3, 64) HS2_ROW(4, 64) HS2_ROW(5, 64) HS2_ROW(6, 64) HS2_ROW(4, 128) HS2_ROW(3, 256) HS2_ROW(4, 256)
#undef HS2_ROW
  return hipErrorInvalidValue;
}

template <int SEG>
static hipError_t launch_cols_t(const Grid &g, const ColTab &t, int axis, const double *Tn,
                                const double *Y, double *X, double *surf, double dz, bool ry,
                                hipStream_t s) {
  // z: 32 columns to a block (256^3: 66 us against 71 with 16, 71 with 64); y:
  // 16 where that makes two waves or more (43 against 46)
  const int cs = (axis == 0 || t.P < 8) && t.P * 32 <= 512 ? 1 : 0;
  const int CW = 16 << cs;
  const dim3 grid((unsigned)((t.groups + (1 << cs) - 1) >> cs)), block(t.P * CW);
  const size_t shm = sizeof(double) * 2 * t.P * CW;
  if (ry && axis != 1) return hipErrorInvalidValue;
#define HS2_RUN(AXIS, RY, PICK)                                                             \
  hipLaunchKernelGGL((k_cols<SEG, AXIS, RY, PICK>), grid, block, shm, s, g, t, cs, Tn, Y, X, \
                     surf, dz)
  if (t.base) {
    if (ry) HS2_RUN(1, true, true);
    else if (axis == 1) HS2_RUN(1, false, true);
    else HS2_RUN(0, false, true);
  } else {
    if (ry) HS2_RUN(1, true, false);
    else if (axis == 1) HS2_RUN(1, false, false);
    else HS2_RUN(0, false, false);
  }
#undef HS2_RUN
  return hipGetLastError();
}

hipError_t launch_cols(const Grid &g, const ColTab &t, int axis, const double *Tn,
                       const double *Y, double *X, double *surf, double dz, bool ry,
                       hipStream_t s) {
  switch (t.seg) {
    case 4: return launch_cols_t<4>(g, t, axis, Tn, Y, X, surf, dz, ry, s);
    case 8: return launch_cols_t<8>(g, t, axis, Tn, Y, X, surf, dz, ry, s);
    case 16: return launch_cols_t<16>(g, t, axis, Tn, Y, X, surf, dz, ry, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace hs2
