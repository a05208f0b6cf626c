// Work-tile descriptors shared by the temporal-blocked tile kernels and their
// host-side planner.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

namespace npbx {

enum GridKind : int32_t { kJacobi2D = 0, kHeat3D = 1 };

// One grid in one round: `depth` sweeps from level L0 (interior in X) to
// level L0+depth (interior written to Y).  Global-boundary values of level L
// are A's when L is even and B's when L is odd (the reference's ping-pong
// leaves each array's boundary untouched).
struct GridRound {
  void* A;
  void* B;
  const void* X;
  void* Y;
  int32_t n;        // side length
  int32_t kind;     // GridKind
  int32_t parity0;  // L0 & 1
  int32_t depth;    // 1 .. T
  // tiling (fixed per grid for a given T)
  int32_t tiles_k;  // tiles along the contiguous axis
  int32_t tiles_j;  // tiles along the row axis
  int32_t seg;      // heat: output planes per tile along i
  int32_t rows;     // heat: rows per wave (a tile is 4*rows rows)
  // FP32 heat: packed boundary columns of A and B (npbx_pack_cols layout
  // [array][plane][row][2]), or null to read them from A and B directly
  const void* cols;
};

// Up to kMaxBatch grid rounds passed by value as one launch's kernel
// argument (< 4 KB); cum[g] is the number of tiles of rounds 0..g-1, so tile
// t of the launch belongs to the round g with cum[g] <= t < cum[g+1].
constexpr int kMaxBatch = 48;
struct RoundBatch {
  int32_t count;
  int32_t cum[kMaxBatch + 1];
  GridRound round[kMaxBatch];
};

// A grid of a plan that runs outside the tile kernels: sweeps [first,
// first + nsweeps) between A and B.
struct SweepGrid {
  void* A;
  void* B;
  int n;
  int64_t first, nsweeps;
};

// One 2-D grid in one launch of register blocks (jacobi2d_deep.hip), as
// GridRound without the tiles.
struct BlockRound {
  const void* A;
  const void* B;
  const void* X;
  void* Y;
  int32_t n, parity0, depth, tiles_j, tiles_i;
};
struct BlockBatch {
  int32_t count;
  int32_t cum[kMaxBatch + 1];
  BlockRound round[kMaxBatch];
};
// A batch's launches and the shape they share: columns per lane, rows per wave.
struct BlockPlan {
  int v = 0, rows = 0;
  std::vector<BlockBatch> launches;
};
int jacobi_batch_plan(int dtype, const std::vector<SweepGrid>& grids, BlockPlan& plan);
int jacobi_batch_launch(int dtype, const BlockPlan& plan, hipStream_t stream);

// The plain sweeps of several heat grids, one launch per sweep of all of them
// (heat3d.hip); with `enqueue` false only counts launches and workgroups.
int heat_batch_sweeps(int dtype, const std::vector<SweepGrid>& grids, bool enqueue,
                      hipStream_t stream, int64_t* launches, int64_t* tiles);

// Rounds of FP32 heat grids on wave-stacked tiles (heatmarch.hip): depths up
// to kHeatMarchDepth, sides of at least kHeatMarchRows.  A batch's cum counts
// planes of tile columns: (columns of a round) * (n - 2) each.
constexpr int kHeatMarchDepth = 4;
constexpr int kHeatMarchRows = 33;
int heat_march_columns(int n, int depth, int* tiles_k, int* tiles_j);
int heat_march_launch(const RoundBatch& b, int blocks, hipStream_t stream);

// Per-launch queue state, self-resetting: `next` hands out tile indices and
// `done` counts workgroups that found the queue empty; the last one resets
// both to zero for the next launch.
struct QueueState {
  int32_t next;
  int32_t done;
  int32_t pad[62];  // one 256-byte line per queue
};

}  // namespace npbx
