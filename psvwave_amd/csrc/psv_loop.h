// psv_loop.h -- resident time loops: a whole forward or adjoint time loop in
// one launch, the state of every tile kept in the registers and LDS of the
// compute unit that owns it (psv_loop.hip), and the gate that keeps all
// blocks of such launches resident at once.
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "psv_kernels.h"

namespace psv {

// The loop kernels: rows per wave and waves per block.  A tile owns at most
// 60 columns (64 lanes less the two-column stress ring on either side) and
// rows * waves - 4 rows.
struct LoopKind {
  int rows, waves;
};
constexpr LoopKind kLoopKinds[] = {{1, 8}, {2, 8}, {3, 8}, {4, 8}, {4, 16}};
constexpr int kNumLoopKinds = 5;
constexpr int kLoopTileX = 60;
// Loop kernels and blocks per compute unit in the order of their time per step
// (3.1, 3.9, 3.7, 4.8 to 5.1, 5.3, 5.9, 6.2, 7.6 and 7.8 to 8.1 us, a forward
// with 19 receivers on a grid that each of them holds and the one before does
// not): launches take the first whose tiles all fit.  Fewer rows a wave make a
// step shorter, and so does a block alone on its unit, up to a wave of rows
// less: compared in one run each, 960 x 448 points took 6.0 us on 256 tiles of
// 28 rows and 6.5 on 368 of 20, 800 x 700 points 6.5 on 490 of 20 rows and 7.7
// on 350 of 28.  (The third,
// two blocks of 4 rows, comes up only where a tile of 12 rows has too many
// receivers.)
struct LoopFit {
  int kind, per_unit;
};
constexpr LoopFit kLoopFits[] = {{0, 1}, {1, 1}, {0, 2}, {2, 1}, {1, 2},
                                 {3, 1}, {2, 2}, {3, 2}, {4, 1}};
constexpr int loop_tile_rows(int kind) {
  return kLoopKinds[kind].rows * kLoopKinds[kind].waves - 4;
}
// receivers a tile can record, one per thread
constexpr int loop_max_receivers(int kind) { return 64 * kLoopKinds[kind].waves; }

// Entries of a loop's tables are InjEntry with, for the injection terms of a
// wave's strip, local = row in the strip * 64 + lane and pad = 1 where more
// terms of the same target follow, and for the receivers of a tile local =
// LDS index of the point's velocity (loop_velocity_index).
struct LoopArgs {
  int nx, nz, pitch, ntx, ntz;
  long long origin;
  const double *lm, *mu, *b, *taper_x, *taper_z;
  double dts, dt, dx, dz, rdx, rdz, zhx, zlx, zhz, zlz, dxdz, d4x, d4z;
  int nt, k0, k1;  // loop indices; time step it = k forward, nt - 1 - k adjoint
  // state at loop index k0 (null: zero) and where to leave the state at k1
  // (null: nowhere): vx, vz, txx, tzz, txz
  const double *in[5];
  int in_pitch;
  long long in_origin;
  double *out[5];  // padded layout (pitch, origin)
  // snapshots of every si-th step (null: none): slot s = it / si, kept when
  // slot_every divides it, at snap + (s / slot_every - slot0) * slot_stride
  double *snap[5];
  long long slot_stride;
  int si, slot0, slot_every;
  // correlation (adjoint): kernels, or with defer_stride > 0 fresh terms of
  // slot s at the pointers + s * defer_stride
  double *rho_k, *lam_k, *mu_k;
  long long defer_stride;
  int kx0, kx1, kz0, kz1;
  double wcorr;
  // injection targets (one component of one point) by tile * waves + wave:
  // targets inj_off[i] .. inj_off[i + 1], the terms of target t being
  // inj[inj_first[t]] .. inj[inj_first[t + 1]] in list order, inj_head[t] the
  // first of them
  const int *inj_off, *inj_first;
  const InjEntry *inj, *inj_head;
  const double *stf, *adj_x, *adj_z;
  // receivers, CSR by tile (null: none recorded)
  const int *rec_off;
  const InjEntry *rec;
  double *rtf_x, *rtf_z;
  // exchange cells, 16 bytes each: [tile][step parity][vx, vz][rim cell]
  void *cells;
  unsigned cells_bytes;
};

// LDS index of the velocity of a tile's own point (row r, column c).
inline int loop_velocity_index(int r, int c) { return (r + 4) * 67 + c + 4; }

// One launch: blocks[i] = (loop, tile column, tile row, 0).
struct LoopLaunch {
  const LoopArgs *loops;
  const int4 *blocks;
  int nblocks;
  unsigned tag0;      // exchange tag of the first step
  unsigned *sync;     // two words, zero before the launch: arrivals, state
  unsigned *poison;   // nonzero: do nothing; set when the blocks were not
                      // resident together in time
  unsigned *status;   // host memory: 1 once the loop runs, 2 after a stall
};
enum { kLoopNotRun = 0, kLoopRan = 1, kLoopStalled = 2 };

hipError_t launch_loop(int kind, bool adjoint, const LoopLaunch &l, hipStream_t s);
// *dst = a and the two meeting words zeroed, in stream order.
hipError_t launch_loop_prepare(LoopArgs *dst, const LoopArgs &a, unsigned *sync, hipStream_t s);

// Tiles of a grid for a loop kernel, which split the columns and the rows
// evenly.
inline int loop_tiles_x(int nx) { return (nx + kLoopTileX - 1) / kLoopTileX; }
inline int loop_tiles_z(int nz, int kind) {
  return (nz + loop_tile_rows(kind) - 1) / loop_tile_rows(kind);
}

// Rim cells kept for a tile (the points at most three from its edge), and
// bytes of the exchange cells of one loop.
constexpr int loop_rim_cells(int kind) { return kLoopKinds[kind].waves == 16 ? 1024 : 512; }
inline size_t loop_cells_bytes(int kind, int ntiles) {
  return (size_t)ntiles * 4 * loop_rim_cells(kind) * 16;
}

// Blocks of a loop kernel that the current device holds at once, at most
// per_unit of them on a compute unit (0: it cannot run them).
int loop_capacity(int kind, int per_unit = 2);

// Launches through the gate of the current device: the blocks of all loop
// launches that may run at the same time fit the device together.
void gated_launch_loop(int kind, bool adjoint, const LoopLaunch &l, hipStream_t s);
// Before a synchronised stream is destroyed: the gate drops its events.
void loop_gate_forget(hipStream_t s);

}  // namespace psv
