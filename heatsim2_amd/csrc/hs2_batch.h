// Batched execution of many independent ADI problems of different sizes and
// step counts: one launch per sweep covers every instance of a group (groups
// run two at a time; see kBatchGroupCells).  Each launch kind
// has a block -> instance table; a block finds its instance, its local block
// index and its instance's current step, and works on that instance's slice
// of the concatenated fields (per-voxel coefficients, DenseView).
//
// Time is driven by counters in device memory (ctr[0]: the forward step a
// chunk of steps begins with, ctr[1]: backward segment), so a captured graph
// of a chunk can be replayed without changing any kernel argument.  Checkpoints are aligned
// to each instance's end: with K steps per segment, backward segment s of
// instance i covers steps [max(0, e-K), e), e = nsteps_i - s*K, so every
// instance is at the same position inside its segment and the recomputation
// runs in lockstep.  Segment slot q (0..K) holds T^{e-K+q}; T* and T** of
// step e-K+q are kept in slot q of their own stores.
#pragma once
#include <hip/hip_runtime.h>

#include "hs2_device.h"

namespace hs2 {

constexpr int kBatchMaxLen = 128;  // axis length limit of the batched kernels
constexpr int kBatchThreads = 256; // threads per block of the y and z kernels
constexpr int kBatchWaves = 4;     // waves (units of rows) per block of the x kernels
constexpr int kBatchSeg = 8;       // cells per thread segment of the line kernels
constexpr int kBatchPlanes = 2;    // planes a wave of the x sweep walks (1, 4: 2% slower, 8: 18%)
constexpr int kBatchSensPlanes = 8;  // planes per block of the sensitivity pass
// Cells of a group, about: two groups run side by side (kBatchLanes), and a
// step's fields of both (T, T*, M, three conductances, w: 49 bytes a cell) fit the
// 256 MB Infinity Cache.  ns per cell and step by the cells run together on one
// stream, forward | with gradient: 12.7 million 0.0265 | 0.1023, 8.7 0.0259 |
// 0.1013, 4.2 to 4.8 0.0241 | 0.0953, 2.0 to 2.6 0.0305 | 0.1029.  24 instances of
// 32..128^3 and 40 to 160 steps, ms for histories | gradients: all together 29.7 |
// 118.1, groups of 4.5 million one by one 28.0 | 113.1, on two lanes of 4.5 million
// 26.6 | 109.7, of 3 million 25.4 | 106.9, of 2.25 million 24.9 | 107.4, of 1.5
// million 26.6 | 110.6; three lanes of 1.5 million 25.3 | 108.5, four of 1.2 31.4 |
// 116.7.
constexpr long long kBatchGroupCells = 2250000;
constexpr int kBatchAlign = 32;    // instance offsets are multiples of this many cells

// Segments of kBatchSeg cells per line of L cells in the y and z line
// kernels (the fewest that cover L), and the lines a 256-thread block holds
// side by side, cw = floor(256 / P): consecutive columns in memory order.
__host__ __device__ inline int batch_line_segs(int L) { return (L + kBatchSeg - 1) / kBatchSeg; }
__host__ __device__ inline int batch_flat_cw(int L) { return kBatchThreads / batch_line_segs(L); }
// The x kernels' row shape by nx: 16 lanes x 2 or 4 cells, 32 x 3 or 4; and the
// rows a wave holds.
__host__ __device__ inline int batch_row(int nx) {
  return nx <= 32 ? 0 : nx <= 64 ? 1 : nx <= 96 ? 2 : 3;
}
__host__ __device__ inline int batch_row_group(int nx) { return nx <= 64 ? 4 : 2; }

struct BatchInst {
  int nz, ny, nx, nsteps;
  long long off;    // first cell in the concatenated fields
  long long hoff;   // first value of the surface history (nsteps x ny x nx)
  long long ckoff;  // first value of the checkpoints (ceil(nsteps/K) fields)
  int src_step;     // step whose source field applies (-1: none)
  int row;          // batch_row(nx)
  int units;        // waves of the x sweep: row groups x chunks of kBatchPlanes planes
  int rows;         // waves of the adjoint x solve: row groups
  int cw[2];        // lines per block: batch_flat_cw of the z and y line lengths
  double dz;
};

enum BatchRule { RULE_FWD, RULE_RECOMP, RULE_BWD, RULE_SEG };

struct BatchMap {
  const BatchInst *inst;
  const int *blk_inst;  // instance of each block of this launch kind
  const int *blk0;      // first block of each instance
  const int *ctr;       // device counters
  int rule, j, K;
  int off;              // first block of the launch's group in the tables
};

// Logical block of hardware block b among nb.  Hardware hands block b to XCD
// b % 8, each with its own L2; consecutive logical blocks touch neighbouring
// rows (and share cache lines of rows that do not start on a line), so they
// go to one XCD in chunks of kBatchChunk (32: measured best among 1 to
// 1024), and the chunks go round the XCDs so
// that every XCD keeps a share of every instance (instances finish at
// different steps).  Blocks past the last whole round of chunks keep their
// index.
constexpr int kBatchChunk = 32;
__device__ __forceinline__ int batch_block(int b, int nb) {
  return xcd_remap_chunks<kBatchChunk>(b, nb);
}

// Instance, local block and step of this block; false if the instance has
// nothing to do under the launch's rule (the whole block returns).
__device__ __forceinline__ bool batch_locate(const BatchMap &m, BatchInst &I, int &local, int &t) {
  const int gb = m.off + batch_block(blockIdx.x, gridDim.x);
  const int i = m.blk_inst[gb];
  local = gb - m.blk0[i];
  I = m.inst[i];
  if (m.rule == RULE_FWD) {
    t = m.ctr[0] + m.j;
    return t < I.nsteps;
  }
  const int e = I.nsteps - m.ctr[1] * m.K;
  if (e <= 0) return false;
  const int s = e - m.K > 0 ? e - m.K : 0;
  if (m.rule == RULE_SEG) {
    t = s;
    return true;
  }
  if (m.rule == RULE_RECOMP) {  // step t: T^t (slot j) -> T^{t+1} (slot j+1)
    t = e - m.K + m.j;
    return t >= s;
  }
  t = e - 1 - m.j;  // RULE_BWD
  return t >= s;
}

__device__ __forceinline__ DenseView offset_view(DenseView v, long long off) {
  v.M += off;
  v.w += off;
  v.g[0] += off;
  v.g[1] += off;
  v.g[2] += off;
  return v;
}

}  // namespace hs2

namespace hs2 {
struct AdjGroup;
// launchers (hs2_dense.hip, hs2_adjoint.hip); nblocks = this kind's block total
// the x sweep; with ck != nullptr (forward) T^t is copied into the instance's
// checkpoint slot on a checkpoint step; ry as for a plan's sweeps
hipError_t launch_batch_rows(const BatchMap &m, int nblocks, const DenseView &v, const double *Tn,
                             double *Ts, const double *src, double *ck, bool ry, hipStream_t s);
hipError_t launch_batch_cols(const BatchMap &m, int nblocks, int axis, const DenseView &v,
                             const double *Tn, const double *Y, double *X, double *hist, bool ry,
                             hipStream_t s);
// transposed y or x solves (axis 1, 2)
hipError_t launch_batch_adj_line(const BatchMap &m, int nblocks, int axis, const DenseView &v,
                                 const double *R, int scale_m, double *U, hipStream_t s);
hipError_t launch_batch_lambda(const BatchMap &m, int nblocks, const DenseView &v, const double *u,
                               long long N, const double *ghist, double *U, hipStream_t s);
hipError_t launch_batch_sens(const BatchMap &m, int nblocks, const DenseView &v, const AdjGroup &f,
                             int cnt, hipStream_t s);
hipError_t launch_batch_ckpt_load(const BatchMap &m, int nblocks, const double *ck, double *seg,
                                  long long N, hipStream_t s);
hipError_t launch_batch_counter(int *ctr, int which, int value, int add, hipStream_t s);
}  // namespace hs2
