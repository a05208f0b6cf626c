// 2-D Jacobi sweeps (jacobi_2d_numpy.py:4-10), temporal-blocked in registers:
// a launch advances every grid point by up to kMaxDepth sweeps.
//
// A workgroup of 16 waves stacked along i holds a region of 16 R rows x 64 V
// columns, each wave R rows and each lane V adjacent columns of them, and
// sweeps it `depth` times in place.  Next to other blocks the outer `depth`
// cells of the region are halo, recomputed by both and one cell less valid
// per sweep; at the grid's edges the region ends with the interior.  West and
// east neighbours are the adjacent lanes (full-wave DPP shifts, two per row
// and sweep whatever V is), north and south the wave's own registers; a
// wave's two edge rows go to its neighbours through LDS, one barrier per
// sweep, written as soon as they are computed and read while the rows between
// them are.
//
// The grid's boundary holds, at every level, what the level's array holds in
// the reference (A's at even levels, B's at odd: the ping-pong never writes
// boundaries): the outer lanes carry the two values of their row, which the
// shifts hand in where the region ends (elsewhere they only reach the halo),
// and the boundary rows lie in LDS.  NARROW: grids smaller than a region,
// where the boundary falls inside it and is put back per point after each
// sweep.  Each level is rounded through the storage type, as the plain
// sweep's stores round it, and each point is jacobi_point -- the reference's
// ((((c + W) + E) + S) + N) * 0.2 -- so results are bitwise the plain sweeps'
// (FP64: the NumPy reference's).
//
// Rounds follow sweep_rounds (tiles.hip): depths <= T covering all but the
// last sweep, their count of the parity that leaves the last two levels in A
// and B as the reference does, then a depth-1 round.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <type_traits>
#include <vector>

#include "common.h"
#include "lanes.h"
#include "points.h"
#include "tiles.h"
#include "vecio.h"

namespace npbx {
namespace {

constexpr int kDeep = 8;       // "jacobi.deep": 8, the default, lets the shape choose
constexpr int kMaxDepth = 28;  // most sweeps per launch
constexpr int kWaves = 16;

std::atomic<int> g_jacobi_deep{kDeep};    // 0 or 1 = plain sweeps
std::atomic<int> g_jacobi_deep_waves{0};  // accepted; the kernel has 16 waves

// A wave's rows of one level.
template <class C, int V, int R>
struct Rows {
  C v[R][V];
};

// Rows [r0, r1) of the next level y from x; above and below are the rows
// outside the wave's, ring its rows' values west of lane 0 and east of lane 63.
template <class S, int V, int R, class C = typename Storage<S>::C>
__device__ __forceinline__ void sweep_rows(const Rows<C, V, R>& x, Rows<C, V, R>& y, int r0,
                                           int r1, const C (&above)[V], const C (&below)[V],
                                           const C (&ring)[R]) {
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (r < r0 || r >= r1) continue;
    const C west = lane_from_left_or(ring[r], x.v[r][V - 1]);
    const C east = lane_from_right_or(ring[r], x.v[r][0]);
#pragma unroll
    for (int c = 0; c < V; ++c)
      y.v[r][c] = Storage<S>::load(Storage<S>::store(jacobi_point<C>(
          x.v[r][c], c == 0 ? west : x.v[r][c - 1], c == V - 1 ? east : x.v[r][c + 1],
          r == R - 1 ? below[c] : x.v[r + 1][c], r == 0 ? above[c] : x.v[r - 1][c])));
  }
}

// LDS of a workgroup.
template <class C, int V>
struct BlockLds {
  struct alignas(sizeof(C) * V) Cols {
    C v[V];
  };
  Cols edge[2][kWaves][2][64];  // per level parity: each wave's first and last row
  Cols outer[2][2][64];         // per level parity: the rows above and below the region
};

template <class S, int V, int R, bool NARROW>
__device__ __forceinline__ void block_sweeps(const S* __restrict__ X, S* __restrict__ Y,
                                             const S* __restrict__ A, const S* __restrict__ B,
                                             int n, int parity0, int depth, int tiles_j,
                                             int tiles_i, int tile,
                                             BlockLds<typename Storage<S>::C, V>& lds) {
  using St = Storage<S>;
  using C = typename St::C;
  using Cols = typename BlockLds<C, V>::Cols;
  auto& edge = lds.edge;
  auto& outer = lds.outer;
  const int lane = threadIdx.x % 64;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const Span sj = span_of(tile % tiles_j, tiles_j, n - 2, 64 * V, depth);
  const Span si = span_of(tile / tiles_j, tiles_i, n - 2, R * kWaves, depth);
  const int gj = sj.origin + lane * V, gi0 = si.origin + w * R;
  const S* const bnd[2] = {parity0 ? B : A, parity0 ? A : B};

  // Level 0, clamped into the grid in a NARROW one (where what lies past its
  // edge is replaced below), the two boundary values of each row (lanes 0 and
  // 63) and the rows outside the region.
  auto at = [&](int i, int j) {
    return static_cast<int64_t>(min(i, n - 1)) * n + (NARROW ? min(j, n - 1) : j);
  };
  Rows<C, V, R> x, y;
  C ring[2][R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
#pragma unroll
    for (int c = 0; c < V; ++c) x.v[r][c] = St::load(X[at(gi0 + r, gj + c)]);
  }
  // (lanes 0 and 63 use them; two addresses for the wave)
  const int gr = lane < 32 ? sj.origin - 1 : min(sj.origin + 64 * V, n - 1);
#pragma unroll
  for (int p = 0; p < 2; ++p) {
#pragma unroll
    for (int r = 0; r < R; ++r)
      ring[p][r] = St::load(bnd[p][static_cast<int64_t>(min(gi0 + r, n - 1)) * n + gr]);
  }
  if (w < 4) {  // (parity, side) = (w / 2, w % 2)
    Cols o;
    const int i = w % 2 ? min(si.origin + R * kWaves, n - 1) : si.origin - 1;
#pragma unroll
    for (int c = 0; c < V; ++c) o.v[c] = St::load(bnd[w / 2][at(i, gj + c)]);
    outer[w / 2][w % 2][lane] = o;
  }
  // NARROW: the boundary's values at the region's points that lie on it
  C fixed[2][NARROW ? R : 1][V];
  if constexpr (NARROW) {
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < V; ++c) fixed[p][r][c] = St::load(bnd[p][at(gi0 + r, gj + c)]);
  }
  auto put_boundary = [&](Rows<C, V, R>& z, int p) {
    if constexpr (NARROW) {
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < V; ++c)
          if (gi0 + r >= n - 1 || gj + c >= n - 1) z.v[r][c] = fixed[p][r][c];
    }
  };
  auto publish = [&](const Rows<C, V, R>& z, int p) {
    Cols first, last;
#pragma unroll
    for (int c = 0; c < V; ++c) first.v[c] = z.v[0][c], last.v[c] = z.v[R - 1][c];
    edge[p][w][0][lane] = first;
    edge[p][w][1][lane] = last;
  };
  put_boundary(x, 0);
  publish(x, 0);
  __syncthreads();

  const int useful = si.useful(w * R, w * R + R);
  // One sweep from z (level parity p) into q.  The neighbours' edge rows are
  // asked for first; rows that need none of them are computed meanwhile, half
  // before and half after this wave's own edge rows are published.
  auto sweep = [&](const Rows<C, V, R>& z, Rows<C, V, R>& q, int p, int s) {
    if (s + 1 >= useful) {  // only halo rows that nothing valid reads any more
      __syncthreads();
      return;
    }
    const Cols a = w == 0 ? outer[p][0][lane] : edge[p][w - 1][1][lane];
    const Cols b = w == kWaves - 1 ? outer[p][1][lane] : edge[p][w + 1][0][lane];
    constexpr int kMid = (R + 1) / 2;
    sweep_rows<S, V, R>(z, q, 1, R > 2 ? kMid : 1, a.v, b.v, ring[p]);
    __builtin_amdgcn_sched_barrier(0);
    sweep_rows<S, V, R>(z, q, 0, 1, a.v, b.v, ring[p]);
    if (R > 1) sweep_rows<S, V, R>(z, q, R - 1, R, a.v, b.v, ring[p]);
    if constexpr (!NARROW) publish(q, p ^ 1);
    __builtin_amdgcn_sched_barrier(0);
    sweep_rows<S, V, R>(z, q, R > 2 ? kMid : 1, R - 1, a.v, b.v, ring[p]);
    if constexpr (NARROW) {
      put_boundary(q, p ^ 1);
      publish(q, p ^ 1);
    }
    __syncthreads();
  };
  int s = 0;
  for (; s + 2 <= depth; s += 2) {
    sweep(x, y, 0, s);
    sweep(y, x, 1, s + 1);
  }
  if (s < depth) {
    sweep(x, y, 0, s);
    x = y;
  }

  // the block's points of level `depth`
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int gi = gi0 + r, k = w * R + r;
    if (k < si.lo || k >= si.hi || gi > n - 2) continue;
    S* to = Y + static_cast<int64_t>(gi) * n + gj;
#pragma unroll
    for (int c = 0; c < V; ++c) {
      const int l = lane * V + c;
      if (l >= sj.lo && l < sj.hi && gj + c <= n - 2) to[c] = St::store(x.v[r][c]);
    }
  }
}

template <class S, int V, int R, bool NARROW>
__global__ __launch_bounds__(64 * kWaves) void jacobi2d_block(const S* __restrict__ X,
                                                              S* __restrict__ Y,
                                                              const S* __restrict__ A,
                                                              const S* __restrict__ B, int n,
                                                              int parity0, int depth, int tiles_j,
                                                              int tiles_i) {
  __shared__ BlockLds<typename Storage<S>::C, V> lds;
  block_sweeps<S, V, R, NARROW>(X, Y, A, B, n, parity0, depth, tiles_j, tiles_i,
                                xcd_tile(blockIdx.x, gridDim.x), lds);
}

// Whether a side's grid is smaller than a region.
__host__ __device__ constexpr bool narrow(int n, int v, int rows) {
  return n - 2 < 64 * v || n - 2 < rows * kWaves;
}

// The rounds of several grids: block t belongs to the round g with cum[g] <= t
// < cum[g+1].
template <class S, int V, int R>
__global__ __launch_bounds__(64 * kWaves) void jacobi2d_blocks(const BlockBatch b) {
  __shared__ BlockLds<typename Storage<S>::C, V> lds;
  const int t = xcd_tile(blockIdx.x, gridDim.x);
  int lo = 0, hi = b.count - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (b.cum[mid] <= t) lo = mid; else hi = mid - 1;
  }
  const BlockRound& g = b.round[lo];
  auto run = [&](auto is_narrow) {
    block_sweeps<S, V, R, decltype(is_narrow)::value>(
        static_cast<const S*>(g.X), static_cast<S*>(g.Y), static_cast<const S*>(g.A),
        static_cast<const S*>(g.B), g.n, g.parity0, g.depth, g.tiles_j, g.tiles_i,
        t - b.cum[lo], lds);
  };
  if (narrow(g.n, V, R))
    run(std::true_type{});
  else
    run(std::false_type{});
}

// Launch shape: columns per lane, rows per wave and sweeps per launch.
struct Shape {
  int v, rows, depth;
};

constexpr Shape kShapes[] = {{1, 3, 0}, {1, 4, 0}, {2, 3, 0}, {2, 4, 0},
                             {2, 5, 0}, {2, 6, 0}, {2, 8, 0}};

// The shape and depth with the smallest modelled time: 5.4 us a launch; per
// sweep 0.06 us plus 9 ns per instruction of a wave's rows that is not idle
// halo, times the workgroups a CU runs; and where a CU holds one workgroup at
// a time (more than 64 VGPRs: over 8 FP64 points a lane), its loads, about
// 10 us, for each further one.  The constants are fitted to 200 measured
// (shape, size, type) times, 10 % off on average; the shapes of the fastest:
// FP64 150^2 1 x 3 rows, depth 20 (52 us for 98 sweeps, 2 x 8: 167); 1000^2
// 2 x 5, 19 (204 us for 200; 1 x 3: 626); 2800^2 2 x 4, 12 (513 us for 100;
// 2 x 8: 717).
// Several grids advance by a round each per launch: as many launches as the
// grid with the most rounds has, and their mean number of workgroups.
Shape pick_shape(int dtype, const std::vector<SweepGrid>& grids, int cap, int max_points = 16) {
  Shape best{2, 4, 2};
  double best_us = INFINITY;
  const bool fp64 = dtype == NPBX_F64;
  // depths past all but a grid's last sweep give the rounds that this one does
  int64_t most = 0;
  for (const SweepGrid& g : grids) most = std::max(most, g.nsweeps - 1);
  for (const Shape& sh : kShapes) {
    if (sh.v * sh.rows > max_points) continue;
    const int wj = 64 * sh.v, wi = kWaves * sh.rows;
    const double issue =
        sh.rows * (5.0 * sh.v + (fp64 ? 4 : 2) + (dtype == NPBX_BF16 ? 2.0 * sh.v : 0));
    const int resident = fp64 && sh.rows * sh.v > 8 ? 1 : 2;
    for (int depth = std::min(cap, 4); depth <= std::min(cap, kMaxDepth); depth += 2) {
      if (wj - 2 * depth < 8 || wi - 2 * depth < 8) break;
      double launches = 0, blocks = 0, d = 1;
      for (const SweepGrid& g : grids) {
        // sweep_rounds: that many rounds and a last one of depth 1
        int64_t rounds = cdiv(g.nsweeps - 1, depth);
        rounds += (rounds ^ (g.nsweeps - 1)) & 1;
        const int dg = static_cast<int>(cdiv(g.nsweeps - 1, std::max<int64_t>(rounds, 1)));
        blocks += static_cast<double>(rounds) * span_count(g.n - 2, wj, dg) *
                  span_count(g.n - 2, wi, dg);
        if (static_cast<double>(rounds) > launches) {
          launches = static_cast<double>(rounds);
          d = dg;
        }
      }
      const double tiles = blocks / std::max(launches, 1.0) / 256;
      const double shared = std::max(1.0, std::min<double>(resident, std::ceil(tiles)));
      const double turns = std::max(1.0, (tiles / shared + std::ceil(tiles / shared)) / 2);
      const double sweep = 0.06 + 0.0091 * issue * (1.0 - d / wi) * shared;
      const double us =
          launches * (5.4 + turns * d * sweep + (turns - 1) * (resident == 1 ? 10 : 2.5));
      if (us < best_us) {
        best_us = us;
        best = {sh.v, sh.rows, depth};
      }
      if (depth >= most) break;
    }
  }
  return best;
}

template <class S, int V, int R>
void launch_shape(const S* X, S* Y, const S* A, const S* B, int n, int parity, int depth,
                  hipStream_t stream) {
  const int tj = span_count(n - 2, 64 * V, depth), ti = span_count(n - 2, R * kWaves, depth);
  const dim3 grid(static_cast<unsigned>(int64_t(tj) * ti)), block(64 * kWaves);
  if (narrow(n, V, R))
    hipLaunchKernelGGL((jacobi2d_block<S, V, R, true>), grid, block, 0, stream, X, Y, A, B, n,
                       parity, depth, tj, ti);
  else
    hipLaunchKernelGGL((jacobi2d_block<S, V, R, false>), grid, block, 0, stream, X, Y, A, B, n,
                       parity, depth, tj, ti);
}

// Calls f.template operator()<V, R>() for a shape of kShapes.
template <class F>
int with_shape(int v, int rows, F&& f) {
  switch (v * 10 + rows) {
    case 13: return f.template operator()<1, 3>();
    case 14: return f.template operator()<1, 4>();
    case 23: return f.template operator()<2, 3>();
    case 24: return f.template operator()<2, 4>();
    case 25: return f.template operator()<2, 5>();
    case 26: return f.template operator()<2, 6>();
    default: return f.template operator()<2, 8>();
  }
}

}  // namespace

int jacobi_deep_depth() { return g_jacobi_deep.load(); }
void set_jacobi_deep_depth(int d) { g_jacobi_deep.store(d); }
int jacobi_deep_waves() { return g_jacobi_deep_waves.load(); }
void set_jacobi_deep_waves(int w) { g_jacobi_deep_waves.store(w); }
int jacobi_deep_max() { return kDeep; }

// Sweeps [first, first + nsweeps) of one grid in blocks, T the "jacobi.deep"
// setting (2 .. 7: at most that many sweeps per launch; 8: by shape).
int jacobi_deep_sweeps(int dtype, void* A, void* B, int n, int64_t first, int64_t nsweeps, int T,
                       hipStream_t stream) {
  NPBX_REQUIRE(T >= 2 && T <= kDeep, "jacobi.deep=%d outside [2, %d]", T, kDeep);
  const Shape shape =
      pick_shape(dtype, {{A, B, n, first, nsweeps}}, T == kDeep ? kMaxDepth : T);
  return dispatch_dtype(dtype, [&](auto tag) -> int {
    using S = decltype(tag);
    S* a = static_cast<S*>(A);
    S* b = static_cast<S*>(B);
    int64_t level = first;
    // the first round reads the array that holds level `first`; each round
    // writes the other array and the next reads it
    S* X = (first & 1) ? b : a;
    for (int depth : sweep_rounds(nsweeps, shape.depth)) {
      S* Y = X == a ? b : a;
      const int parity = static_cast<int>(level & 1);
      with_shape(shape.v, shape.rows, [&]<int V, int R>() {
        launch_shape<S, V, R>(X, Y, a, b, n, parity, depth, stream);
        return NPBX_OK;
      });
      NPBX_LAUNCHED("jacobi2d_block");
      X = Y;
      level += depth;
    }
    return NPBX_OK;
  });
}

// Launch r runs round r of every grid that has one.
int jacobi_batch_plan(int dtype, const std::vector<SweepGrid>& grids, BlockPlan& plan) {
  // more than 10 FP64 points a lane spill beside the NARROW form
  const Shape shape = pick_shape(dtype, grids, kMaxDepth, dtype == NPBX_F64 ? 10 : 16);
  plan.v = shape.v;
  plan.rows = shape.rows;
  std::vector<std::vector<int>> depths;
  size_t nrounds = 0;
  for (const SweepGrid& g : grids) {
    depths.push_back(sweep_rounds(g.nsweeps, shape.depth));
    nrounds = std::max(nrounds, depths.back().size());
  }
  std::vector<int64_t> level;
  for (const SweepGrid& g : grids) level.push_back(g.first);
  // round r reads the array that holds its first level: A or B by the parity
  // of `first`, then in turn
  for (size_t r = 0; r < nrounds; ++r) {
    bool open = false;
    for (size_t i = 0; i < grids.size(); ++i) {
      if (r >= depths[i].size()) continue;
      if (!open || plan.launches.back().count == kMaxBatch) {
        plan.launches.emplace_back();
        plan.launches.back().count = 0;
        plan.launches.back().cum[0] = 0;
        open = true;
      }
      const SweepGrid& g = grids[i];
      BlockBatch& b = plan.launches.back();
      const bool from_a = ((g.first + static_cast<int64_t>(r)) & 1) == 0;
      const int depth = depths[i][r];
      const int tj = span_count(g.n - 2, 64 * shape.v, depth);
      const int ti = span_count(g.n - 2, shape.rows * kWaves, depth);
      const int64_t end = b.cum[b.count] + int64_t(tj) * ti;
      NPBX_REQUIRE(end < (int64_t(1) << 31), "jacobi batch: too many blocks");
      b.round[b.count] = {g.A, g.B, from_a ? g.A : g.B, from_a ? g.B : g.A, g.n,
                          static_cast<int32_t>(level[i] & 1), depth, tj, ti};
      b.cum[++b.count] = static_cast<int32_t>(end);
      level[i] += depth;
    }
  }
  return NPBX_OK;
}

int jacobi_batch_launch(int dtype, const BlockPlan& plan, hipStream_t stream) {
  return dispatch_dtype(dtype, [&](auto tag) -> int {
    using S = decltype(tag);
    for (const BlockBatch& b : plan.launches)
      NPBX_TRY(with_shape(plan.v, plan.rows, [&]<int V, int R>() -> int {
        hipLaunchKernelGGL((jacobi2d_blocks<S, V, R>),
                           dim3(static_cast<unsigned>(b.cum[b.count])), dim3(64 * kWaves), 0,
                           stream, b);
        NPBX_LAUNCHED("jacobi2d_blocks");
        return NPBX_OK;
      }));
    return NPBX_OK;
  });
}

}  // namespace npbx
