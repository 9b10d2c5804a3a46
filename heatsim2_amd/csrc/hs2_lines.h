// Line tables: a class-map plan's lines, told apart by their class bytes and
// factored once.
//
// On a class-map plan the matrix of a line depends only on the class bytes
// along it, and few different sequences occur (a plate has one per axis, a
// laminate one per overlap of delaminations).  The plan numbers the distinct
// lines of each axis, eliminates each once on the host, and the sweeps read
// the finished factors: no division, no class byte and no table lookup per
// cell, and only the right-hand side in registers.
//
// y, z (ColTab): a column of L cells in P segments of SEG cells.  Row t of
// its segment's own elimination (rows a x[t-1] + b x[t] + c x[t+1] = r, no
// coupling into the segment) keeps
//   m = M/piv, inv = 1/piv, l = a/piv, u = c/piv     (y_t = r/piv - l y_{t-1},
//                                                     x_t = y_t - u x_{t+1})
// and V, W, the segment's response to its outer neighbours xl and xr:
//   x_t = (segment's own solution)_t - V_t xl - W_t xr.
// xl and xr of every segment are a fixed linear function of all segments' own
// end values; `red` holds its coefficients, `band` how many segments away
// they matter (entries below 2^-64 are left out).
//
// x (RowTab): a row of nx cells over G lanes x CPL cells, factored over the
// whole line; the two recurrences are scanned across lanes with the lanes'
// transfer factors.  A row's explicit part needs M, w, g_y and g_z of its
// cells: six numbers per row where they do not vary along it, per cell
// where they do.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <functional>
#include <vector>

#include "hs2_device.h"

namespace hs2 {

constexpr int kColCoef = 6;     // m, inv, l, u, V, W per cell
constexpr int kColMaxSegs = 32;
constexpr int kColWindow = 64;  // columns a group is picked from
constexpr int kRowScan = 4;     // scan factors per lane and direction
constexpr int kRowExpl = 6;     // M, w gy-, w gy+, w gz-, w gz+, w

struct ColTab {
  const double *coef;   // [line][P][SEG][kColCoef]
  const double *red;    // [line][P][P][4]: xl from s_j, e_j; xr from s_j, e_j
  const int *base;      // [group][16]: a column's first cell; top bit: no
                        // column.  Null: the columns in memory order
  const uint16_t *pid;  // distinct line of each group's columns
  int groups;
  int seg, P, band;
};

struct RowTab {
  const double *lane;   // [line][row_pairs][G][2]: inv, l, u per cell; scan factors
  const double *row;    // [explicit row][kRowExpl]
  const double *cell;   // [varying explicit row][G CPL][kRowExpl]
  const uint32_t *pid;  // per row (k, j): line | explicit row << 16 (kRowVaries: varying)
  int cpl, g;
  int nlds;             // lines whose factors the blocks keep in LDS
  unsigned scan;        // bits 0..5: forward scan steps that matter; 8..13: backward
};
constexpr uint32_t kRowVaries = 0x8000u;
// pairs of numbers per lane and line
__host__ __device__ constexpr int row_pairs(int cpl) { return (3 * cpl + 2 * kRowScan + 1) / 2; }

// which rows of lanes x cells serve nx cells per row (g = 0: none)
void row_shape(int nx, int *cpl, int *g);
// segment length and count for columns of L cells (0: none)
void col_shape(int L, int *seg, int *P);

// host: factors of one distinct line.  M, w, g: L cells (g: minus faces)
void factor_column(int L, int seg, int P, const double *M, const double *w, const double *g,
                   double *coef, double *red, int *band);
void factor_row(int nx, int cpl, int G, const double *M, const double *w, const double *g,
                double *lane, unsigned *scan);

// Puts columns of one line together, 16 to a group, out of windows of
// kColWindow neighbouring columns (id: each column's line; base: its first
// cell); a group's places without a column repeat its last one with the top
// bit set.  Returns the number of groups.
int group_columns(int ncol, const std::vector<int> &id, const std::function<int(int)> &base,
                  std::vector<int> *idx, std::vector<uint16_t> *line);

// 128-bit position-dependent sums over each line's bytes: axis 0, 1: the
// class bytes of z, y columns; axis 2: of x rows; axis 3: of x rows' explicit
// part (the y, z classes of the row, the next row and the next plane)
hipError_t launch_line_hash(const Grid &g, const uint8_t *cz, const uint8_t *cy,
                            const uint8_t *cx, int which, unsigned long long *out, hipStream_t s);
// *flag = 1 where a line differs from the line that stands for it
hipError_t launch_line_check(const Grid &g, const uint8_t *cz, const uint8_t *cy,
                             const uint8_t *cx, int which, const int *rep, int *flag,
                             hipStream_t s);
// the class bytes of `count` lines, one after another (which == 3: five
// sequences per row: M's class, y, y+1, z, z+1)
hipError_t launch_line_gather(const Grid &g, const uint8_t *cz, const uint8_t *cy,
                              const uint8_t *cx, int which, const int *line, int count,
                              uint8_t *out, hipStream_t s);

hipError_t launch_rows(const Grid &g, const RowTab &t, const double *Tn, double *Ts,
                       const uint8_t *vmap, const double *vtab, const double *sfield, bool ry,
                       hipStream_t s);
hipError_t launch_cols(const Grid &g, const ColTab &t, int axis, const double *Tn,
                       const double *Y, double *X, double *surf, double dz, bool ry,
                       hipStream_t s);

}  // namespace hs2
