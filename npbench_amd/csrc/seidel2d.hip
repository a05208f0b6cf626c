// 2-D Gauss-Seidel of polybench's seidel_2d
// (npbench/benchmarks/polybench/seidel_2d/seidel_2d_numpy.py:4-13), FP64,
// bitwise the NumPy reference.
//
// A sweep updates rows 1..N-2 in order: row i adds the sum of its seven
// neighbours -- row i-1 already swept, its own right neighbour and row i+1
// not yet -- and then runs x_j = (x_j + x_{j-1}) / 9 along j.  Point (t, i, j)
// (t the sweep) needs (t, i, j-1), (t, i-1, j-1..j+1), (t-1, i, j+1) and
// (t-1, i+1, j-1..j+1), so all points of one 4 t + 2 i + j may be computed
// together: the serial chain is 4 sweeps + 2 N + N points long, not
// sweeps x N x N.
//
// A wave runs 64 consecutive rows of one sweep, lane l two columns behind
// lane l-1: at step s lane l computes column s - 2 l.  Everything a step needs
// is then one step old or older -- the row above's next value is what lane
// l-1 has just computed (a DPP shift), the row below's old value is a stream
// of one new value per step, and the row's own old value is lane l-1's stream
// two steps ago (another shift).  A workgroup runs kW consecutive sweeps over
// the same 64 rows, wave w shifted up by w rows: its stream is what wave w-1
// computed, handed over through LDS kG steps (a chunk) at a time with one
// barrier per chunk.  As many helper waves keep memory off the chains: they
// bring wave 0's stream and every wave's lane-0 neighbours from A into LDS and
// write the last wave's rows and the other waves' last row to A.
// A itself thus carries everything between tiles.
//
// Tiles (group g of kW sweeps, band b of 64 rows) need (g, b-1), (g-1, b) and
// (g-1, b+1), each only a bounded number of steps ahead.  seidel2d_tiles<true>
// runs a whole range of groups in one launch: workgroups take tiles from a
// ticket counter in an order in which a tile needs only earlier ones -- those
// have been taken by workgroups that are running, so every wait ends,
// whatever the device holds at once -- and each tile publishes how far its
// rows in A have come.  seidel2d_tiles<false> runs one slot b + 2 g of
// independent tiles per launch with no counters: for stream capture, where a
// replay must not share state with other calls.
//
// Bound by the chunks' chain, 1.4 us each (some 420 at N = 400): sixteen steps
// of a shift and ten dependent FP64 operations, about 90 cycles (14 and 7.5 each,
// timed on one wave) or 0.6 us at 2.40 GHz, then the chunk's exchange through
// LDS, the helpers' loads and the barrier; and about 12 chunks from one tile's
// start to the next one's in either direction (8 of them the bands' skew).
// N = 400, 99 sweeps on the MI355X: 0.59 ms (slot by slot 2.5 ms; the former
// kernel, one workgroup running row recurrences back to back, 39.6 ms).
// Chunks of 8 steps measured 0.63 ms; helpers at the default priority 0.62;
// one memory wave for loads and one for stores instead of four of both 0.77;
// and without helpers -- each wave loading and storing for itself -- 1.5 ms.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <climits>
#include <mutex>

#include "common.h"
#include "division.h"
#include "lanes.h"

namespace npbx {
namespace {

constexpr int kW = 4;    // sweeps (computing waves) per tile: one wave per SIMD
constexpr int kG = 16;   // steps per chunk
constexpr int kRows = 64 / kG;  // rows one loader or storer access covers, kG columns each
constexpr int kPitch = 65;      // LDS doubles per step: kG lanes of one row on different banks
constexpr int kThreads = 64 * 2 * kW;
static_assert(64 % (kG * kW) == 0);
constexpr int kMaxN = 1 << 14;
constexpr int kMaxTiles = 4096;      // tiles per launch
constexpr int kLine = 16;            // ints per counter

// Tiles per launch ("seidel.blocks").
std::atomic<int> g_seidel_blocks{2048};
// Polls after which a wait gives up ("seidel.polls"): some seconds.
std::atomic<int> g_seidel_polls{1 << 22};

// What the workgroups of one launch share; all zero between launches.
struct SeidelSync {
  int ticket, done, failed, pad[kLine - 3];
  // per tile, a cache line apart so that waits do not queue on one: intervals
  // whose outputs are in A
  int stored[kMaxTiles * kLine];
};

struct SeidelArgs {
  double* A;
  int n, sweeps;      // sweeps of this launch's groups in all
  int bands, groups;  // tiles per group, groups of this launch
  int polls;          // after which a wait gives up
  int* gave_up;       // host memory: set where one did
};

// Tiles read each other's rows within a launch.  Every access to A is an
// atomic of device scope, performed where all XCDs see it (no L1 or L2 holds
// a copy), so a store that has completed (vmcnt 0) is what later loads
// return, and the counters need no cache flush or invalidation around them.
__device__ __forceinline__ double get(const double* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void put(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int peek(const int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void poke(int* p, int v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The recurrence's state of one lane at column j: the newest value (column
// j-1), the row above at j-1 and j, the row's own old value at j, the row
// below's old values at j-1 and j.
struct LaneState {
  double x, um, u0, oc, dm, d0;
};

// How a chunk divides by 9.  The short division is the operator's result
// where nothing in the IEEE sequence rescales; it is written so that n = +-0
// keeps its sign.
enum class Div {
  kPositive,  // short; every input is in [2^-800, 2^800], so every value a
              // sum of such: an average of nine stays in range
  kChecked,   // short; reports an n that is neither zero nor in 2^-899 .. 2^900
  kOperator
};

// One chunk of steps from column j0 on: dn the row below's old values from
// column j0+1 on, edge (lane 0's) the row above, swept, and the row's own old
// value, from column j0+1 on; results go to out[step][lane].  MASKED: points
// off the interior keep their old value.  False where kChecked left its range.
template <bool MASKED, Div DIV>
__device__ __forceinline__ bool run_chunk(LaneState& s, const double (&dn)[kG],
                                          const double2 (&edge)[kG], double (*out)[kPitch],
                                          int lane, int j0, int n, double ninth) {
  int emin = 0;
  bool ok = true;
#pragma unroll
  for (int k = 0; k < kG; ++k) {
    const double u1 = lane_from_left_or(edge[k].x, s.x);
    const double o1 = lane_from_left_or(edge[k].y, s.dm);
    const double d1 = dn[k];
    double sum = s.um + s.u0;
    sum = sum + u1;
    sum = sum + o1;
    sum = sum + s.dm;
    sum = sum + s.d0;
    sum = sum + d1;
    const double num = (s.oc + sum) + s.x;
    double x;
    if constexpr (DIV == Div::kOperator) {
      x = num / 9.0;
    } else {
      if constexpr (DIV == Div::kChecked) {
        emin = min(emin, __builtin_amdgcn_frexp_exp(num));
        ok = ok && fabs(num) < 0x1p900;
      }
      const double m = num * ninth;
      const double r = __builtin_fma(9.0, m, -num);
      x = __builtin_fma(-r, ninth, m);
    }
    if constexpr (MASKED) {
      asm("" : "+v"(x));  // a select, not a branch around the quotient
      x = static_cast<unsigned>(j0 + k - 1) < static_cast<unsigned>(n - 2) ? x : s.oc;
    }
    s.um = s.u0;
    s.u0 = u1;
    s.oc = o1;
    s.dm = s.d0;
    s.d0 = d1;
    s.x = x;
    out[k][lane] = x;
  }
  return ok && emin >= -898;
}

// A workgroup's view of its tile.  Interval tau runs chunk tau - w of every
// computing wave w < waves; chunk c of wave w is the steps
// s = kG c - w - 1 + (0 .. kG-1).
struct Tile {
  int grp, band, waves, chunks;
};

struct SeidelLds {
  double ring[kW + 1][2][kG][kPitch];  // [0] from the loader, [w + 1] from wave w
  double2 edges[2][kW][kG];
  double spoil;  // added to all that comes from A: -0.0, which changes no bit, or NaN
  int signs;     // nonzero once a value outside [2^-800, 2^800] came from A
  int taken;
};

// A computing wave.
__device__ __forceinline__ void compute_wave(const SeidelArgs& g, const Tile& t, SeidelLds& lds,
                                             int w, int lane) {
  const int n = g.n;
  const int row = 1 + 64 * t.band - w + lane;
  const bool rows_inside = t.band > 0 && 64 * t.band + 64 <= n - 2;
  const double ninth = division_reciprocal(9.0);
  LaneState st{};
  for (int tau = 0; tau <= t.chunks + t.waves - 1; ++tau) {
    const int c = tau - w;
    if (c >= 0 && c < t.chunks && w < t.waves) {
      const int s0 = c * kG - w - 1;
      // rows off the interior: no column is
      const int j0 = row >= 1 && row <= n - 2 ? s0 - 2 * lane : INT_MIN / 2;
      double dn[kG];
      double2 edge[kG];
#pragma unroll
      for (int k = 0; k < kG; ++k) dn[k] = lds.ring[w][(tau + 1) & 1][k][lane];
      if (lane == 0) {  // the other lanes' copies would only load the LDS
#pragma unroll
        for (int k = 0; k < kG; ++k) edge[k] = lds.edges[(tau + 1) & 1][w][k];
      }
      double(*out)[kPitch] = lds.ring[w + 1][tau & 1];
      const bool inside = rows_inside && s0 - 126 >= 1 && s0 + kG - 1 <= n - 2;
      if (__builtin_amdgcn_readfirstlane(lds.signs) == 0) {
        if (inside)
          run_chunk<false, Div::kPositive>(st, dn, edge, out, lane, j0, n, ninth);
        else
          run_chunk<true, Div::kPositive>(st, dn, edge, out, lane, j0, n, ninth);
      } else {
        const LaneState before = st;
        if (!__all(run_chunk<true, Div::kChecked>(st, dn, edge, out, lane, j0, n, ninth))) {
          st = before;
          run_chunk<true, Div::kOperator>(st, dn, edge, out, lane, j0, n, ninth);
        }
      }
    }
    __syncthreads();
  }
}

// A helper wave; helper h shares its SIMD with computing wave h and does a
// quarter of the tile's memory work.  In interval tau the helpers write what
// interval tau - 1 computed to A, and bring into LDS what interval tau + 1
// takes from A: wave 0's stream, the rows below its 64, and the two rows lane
// 0 of wave h needs.  Lane 0 of wave w at step s reads column s + 1 of rows
// 64 band - w and 64 band - w + 1, which waves w and w - 1 of tile (g, b-1)
// compute at step s + 127; wave 0's lanes read rows that the last wave of the
// group before computes kW sweeps on and as many rows up, at step
// s + 1 + 2 kW of tile (g-1, b) and 128 steps earlier of tile (g-1, b+1).
template <bool WAIT>
__device__ __forceinline__ void helper_wave(const SeidelArgs& g, const Tile& t, SeidelLds& lds,
                                            SeidelSync* sync, int h, int lane) {
  __builtin_amdgcn_s_setprio(2);  // few instructions, all of them waited for
  constexpr int kPart = 64 / kRows / kW;  // accesses per helper for 64 rows
  const int n = g.n;
  const int k = lane % kG, q = lane / kG;
  const int end = t.chunks + t.waves - 1;  // intervals that compute
  const int lw = t.waves - 1;              // the wave whose rows all go to A
  int* mine = nullptr;
  const int* watched = nullptr;
  int ahead = INT_MIN / 2, seen = 0;  // lanes that watch nothing need nothing
  if constexpr (WAIT) {
    auto counter = [&](int gg, int bb) { return sync->stored + (gg * g.bands + bb) * kLine; };
    constexpr int kBelow = (kG - 1 + 3 * kW) / kG;  // chunks
    watched = mine = counter(t.grp, t.band);
    auto watch = [&](int gg, int bb, int need) {
      if (gg < 0 || bb < 0 || bb >= g.bands) return;
      watched = counter(gg, bb);
      ahead = need;
    };
    if (lane == 0) watch(t.grp, t.band - 1, (kG + 126) / kG + 1);
    if (lane == 1) watch(t.grp - 1, t.band, kBelow + kW);
    if (lane == 2) watch(t.grp - 1, t.band + 1, kBelow - 128 / kG + kW);
  }
  // Helper 0 waits for all.  Every wait ends, because the tiles waited for run
  // already; the bound only keeps a broken launch from hanging the device.
  // Where it is reached, all that the tile takes from A from then on is NaN,
  // so the grid is from there on, and the host is told.
  bool failed = false;
  auto wait_for = [&](int tau) {
    if (!WAIT || h != 0) return;
    for (int polls = 0; !failed && !__all(seen >= tau + ahead); ++polls) {
      seen = peek(watched);
      if (polls < g.polls && !(polls % 64 == 63 && peek(&sync->failed))) continue;
      if (__all(seen >= tau + ahead)) break;
      failed = true;
      poke(&sync->failed, 1);
      if (lane == 0) {
        lds.spoil = NAN;  // the helpers read it behind the next barrier
        __hip_atomic_store(g.gave_up, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      }
    }
    asm volatile("" ::: "memory");
  };
  int from[kPart];  // rows below wave 0's: element of column -2 l
#pragma unroll
  for (int m = 0; m < kPart; ++m) {
    const int l = (h * kPart + m) * kRows + q;
    from[m] = min(2 + 64 * t.band + l, n - 1) * n;
  }
  const int erow = min(max(64 * t.band - h + (q & 1), 0), n - 1) * n;
  double v[kPart], e = 1.0, spoil = -0.0;
  auto load = [&](int tau) {
    const int c0 = tau * kG + k;  // the column lane row 0 of wave 0 needs, s + 1
#pragma unroll
    for (int m = 0; m < kPart; ++m) {
      const int l = (h * kPart + m) * kRows + q;
      v[m] = get(g.A + from[m] + min(max(c0 - 2 * l, 0), n - 1));
    }
    if (q < 2) e = get(g.A + erow + min(max(c0 - h * (kG + 1), 0), n - 1));
    if constexpr (WAIT) spoil = lds.spoil;
  };
  auto commit = [&](int tau) {
    auto plain = [](double a) { return a >= 0x1p-800 && a <= 0x1p800; };
    bool all = q >= 2 || plain(e);
#pragma unroll
    for (int m = 0; m < kPart; ++m) {
      lds.ring[0][(tau + 1) & 1][k][(h * kPart + m) * kRows + q] = v[m] + spoil;
      all = all && plain(v[m]);
    }
    if (!__all(all)) lds.signs = 1;
    double2* to = &lds.edges[(tau + 1) & 1][h][k];
    if (q < 2) (q ? to->y : to->x) = e + spoil;
  };
  auto store = [&](int tau) {  // what interval tau computed
    const int par = tau & 1, c = tau - lw, s0 = c * kG - lw - 1 + k;
    if (c >= 0) {
#pragma unroll
      for (int m = 0; m < kPart; ++m) {
        const int l = (h * kPart + m) * kRows + q, row = 1 + 64 * t.band - lw + l, j = s0 - 2 * l;
        const double x = lds.ring[lw + 1][par][k][l];
        if (row >= 1 && row <= n - 2 && static_cast<unsigned>(j - 1) < static_cast<unsigned>(n - 2))
          put(g.A + row * n + j, x);
      }
    }
    // lane 63 of the waves before the last
    const int cw = tau - h;
    if (h < lw && cw >= 0 && cw < t.chunks && q == 0) {
      const int row = 64 + 64 * t.band - h, j = cw * kG - h - 1 + k - 126;
      if (row <= n - 2 && static_cast<unsigned>(j - 1) < static_cast<unsigned>(n - 2))
        put(g.A + row * n + j, lds.ring[h + 1][par][k][63]);
    }
  };
  wait_for(0);
  __syncthreads();
  load(0);
  commit(0);
  wait_for(1);
  __syncthreads();
  for (int tau = 0; tau <= end; ++tau) {
    // every helper's stores of the interval before have completed
    if (WAIT && h == 0 && lane == 0 && tau > 1) poke(mine, tau - 1);
    if (tau + 1 < end) load(tau + 1);
    if (tau > 0) store(tau - 1);
    if (tau + 2 < end) wait_for(tau + 2);  // for all helpers' next loads
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (tau + 1 < end) commit(tau + 1);
    __syncthreads();
  }
  if (WAIT && h == 0 && lane == 0) poke(mine, INT_MAX / 2);
}

template <bool WAIT>
__global__ __launch_bounds__(kThreads) void seidel2d_tiles(SeidelArgs g, int slot,
                                                           SeidelSync* sync) {
  __shared__ SeidelLds lds;
  const int tid = threadIdx.x, lane = tid % 64;
  if (tid == 0) lds.signs = 0, lds.spoil = -0.0;
  const int w = __builtin_amdgcn_readfirstlane(tid / 64);
  Tile t;
  if constexpr (WAIT) {
    if (tid == 0)
      lds.taken =
          __hip_atomic_fetch_add(&sync->ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const int taken = __builtin_amdgcn_readfirstlane(lds.taken);
    t.grp = taken / g.bands;
    t.band = taken % g.bands;
  } else {
    t.grp = max(0, (slot - g.bands + 2) / 2) + blockIdx.x;
    t.band = slot - 2 * t.grp;
    __syncthreads();
  }
  t.waves = min(kW, g.sweeps - t.grp * kW);  // sweeps of this group
  // the last lane any wave needs (row n-1 passes its values on)
  const int last = min(63, g.n + kW - 3 - 64 * t.band);
  t.chunks = (g.n + 2 * last + kW + kG - 1) / kG;

  if (w >= kW) {
    helper_wave<WAIT>(g, t, lds, sync, w - kW, lane);
  } else {
    __syncthreads();  // the helpers' first wait
    __syncthreads();  // and chunk
    compute_wave(g, t, lds, w, lane);
  }

  if constexpr (WAIT) {
    // the last workgroup to finish leaves the counters zero for the next launch
    // (its helper 0 after its last word in them)
    if (w == kW) {
      const int tiles = g.bands * g.groups;
      int before = 0;
      if (lane == 0)
        before =
            __hip_atomic_fetch_add(&sync->done, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
      if (__builtin_amdgcn_readfirstlane(before) == tiles - 1) {
        for (int i = lane; i < tiles; i += 64) poke(sync->stored + i * kLine, 0);
        if (lane == 0) {
          poke(&sync->ticket, 0);
          poke(&sync->done, 0);
          poke(&sync->failed, 0);
        }
      }
    }
  }
}

// Grids of up to kSmallN: one wave, the grid in LDS, a step for each 4 t + 2 i + j.
// Lane 8 (t mod 8) + i - 1 has row i of sweep t; at most seven sweeps have a point
// in one step, and none of a step's points reads another.  A step is nine LDS reads
// and some twenty dependent operations; the tiles above spend twelve chunks of
// mostly masked steps on such a grid.  us, 69 sweeps, tiles | here: 3 x 3 114 | 29,
// 10 x 10 154 | 63; one sweep of 3 x 3 9.8 | 8.1.
constexpr int kSmallN = 10;
constexpr int64_t kSmallSweeps = 1 << 16;  // per launch: some 40 ms

__global__ __launch_bounds__(64) void seidel2d_small(double* __restrict__ A, int n, int sweeps) {
  __shared__ double g[kSmallN * kSmallN];
  const int lane = threadIdx.x, i = lane % 8 + 1, phase = lane / 8;
  for (int e = lane; e < n * n; e += 64) g[e] = A[e];
  __syncthreads();
  const int last = 4 * (sweeps - 1) + 3 * (n - 2);
  for (int tau = 3; tau <= last; ++tau) {
    const int newest = (tau - 2 * i - 1) >> 2;  // the sweep whose column is 1 .. 4
    const int t = newest - ((newest - phase) & 7), j = tau - 4 * t - 2 * i;
    if (i <= n - 2 && t >= 0 && t < sweeps && j <= n - 2) {
      double* p = g + i * n + j;
      double sum = p[-n - 1] + p[-n];
      sum = sum + p[-n + 1];
      sum = sum + p[1];
      sum = sum + p[n - 1];
      sum = sum + p[n];
      sum = sum + p[n + 1];
      p[0] = ((p[0] + sum) + p[-1]) / 9.0;
    }
    __syncthreads();
  }
  for (int e = lane; e < n * n; e += 64) A[e] = g[e];
}

// Counter sets for kSyncSlots launches in flight per device: fixed device
// arrays, one copy per GPU, zero at load.  A launch takes the next slot in
// turn after the event of the slot's previous user, whatever streams and
// threads the two are on.
constexpr int kSyncSlots = 8;
constexpr int kMaxDevices = 64;
static __device__ __align__(256) SeidelSync seidel_sync[kSyncSlots];

struct SyncPool {
  SeidelSync* base = nullptr;  // null until seidel_setup ran on the device
  hipEvent_t last[kSyncSlots] = {};
  int next = 0;
  std::atomic<int*> gave_up{nullptr};  // host memory the device writes
};
std::mutex g_pool_mu;
SyncPool g_pool[kMaxDevices];

bool capturing(hipStream_t stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &status) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return status != hipStreamCaptureStatusNone;
}

// One launch for all groups of g, or `launched` false where the device has no
// counters.
int launch_chained(SeidelArgs g, hipStream_t stream, bool& launched) {
  int dev = 0;
  NPBX_HIP(hipGetDevice(&dev));
  launched = false;
  if (dev < 0 || dev >= kMaxDevices) return NPBX_OK;
  std::lock_guard<std::mutex> lock(g_pool_mu);
  SyncPool& pool = g_pool[dev];
  if (!pool.base) return NPBX_OK;
  g.polls = g_seidel_polls.load();
  g.gave_up = pool.gave_up.load();
  const int k = pool.next;
  NPBX_HIP(hipStreamWaitEvent(stream, pool.last[k], 0));
  hipLaunchKernelGGL(seidel2d_tiles<true>, dim3(g.bands * g.groups), dim3(kThreads), 0, stream, g,
                     0, pool.base + k);
  NPBX_LAUNCHED("seidel2d_tiles");
  NPBX_HIP(hipEventRecord(pool.last[k], stream));
  pool.next = (k + 1) % kSyncSlots;
  launched = true;
  return NPBX_OK;
}

// The same groups as one launch per slot of independent tiles.
int launch_slots(const SeidelArgs& g, hipStream_t stream) {
  for (int slot = 0; slot < g.bands + 2 * (g.groups - 1); ++slot) {
    const int lo = std::max(0, (slot - g.bands + 2) / 2), hi = std::min(g.groups - 1, slot / 2);
    if (hi < lo) continue;  // odd slots of a single band
    hipLaunchKernelGGL(seidel2d_tiles<false>, dim3(hi - lo + 1), dim3(kThreads), 0, stream, g, slot,
                       static_cast<SeidelSync*>(nullptr));
    NPBX_LAUNCHED("seidel2d_tiles");
  }
  return NPBX_OK;
}

}  // namespace

int seidel_blocks() { return g_seidel_blocks.load(); }
void set_seidel_blocks(int blocks) { g_seidel_blocks.store(blocks); }
int seidel_polls() { return g_seidel_polls.load(); }
void set_seidel_polls(int polls) { g_seidel_polls.store(polls); }

// EHIP, once, where a wait of an earlier call on the current device gave up.
int seidel_failure() {
  int dev = 0;
  NPBX_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return NPBX_OK;
  int* gave_up = g_pool[dev].gave_up.load();
  if (!gave_up || !__atomic_load_n(gave_up, __ATOMIC_RELAXED) ||
      !__atomic_exchange_n(gave_up, 0, __ATOMIC_RELAXED))
    return NPBX_OK;
  return fail(NPBX_EHIP, "seidel2d: a tile of an earlier call gave up waiting for another; "
              "that call's grid holds NaN");
}

// The current device's counters and their events, once per device.
int seidel_setup() {
  int dev = 0;
  NPBX_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return NPBX_OK;
  std::lock_guard<std::mutex> lock(g_pool_mu);
  SyncPool& pool = g_pool[dev];
  if (pool.base) return NPBX_OK;
  void* p = nullptr;
  NPBX_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(seidel_sync)));
  for (hipEvent_t& e : pool.last)
    if (!e) NPBX_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  void* word = nullptr;
  NPBX_HIP(hipHostMalloc(&word, kLine * sizeof(int), hipHostMallocMapped | hipHostMallocCoherent));
  *static_cast<int*>(word) = 0;
  pool.gave_up.store(static_cast<int*>(word));
  pool.base = static_cast<SeidelSync*>(p);
  return NPBX_OK;
}

}  // namespace npbx

extern "C" int npbx_seidel2d(int dtype, void* A, int64_t N, int64_t tsteps, void* stream) {
  using namespace npbx;
  NPBX_REQUIRE(dtype == NPBX_F64, "seidel2d: dtype %s not supported (f64)", dtype_name(dtype));
  NPBX_REQUIRE(N >= 0 && N <= kMaxN, "seidel2d: N=%lld out of range (0 .. %d)",
               static_cast<long long>(N), kMaxN);
  NPBX_REQUIRE(tsteps <= (int64_t(1) << 30), "seidel2d: TSTEPS out of range");
  const int64_t sweeps = tsteps - 1;  // range(0, TSTEPS - 1)
  if (N < 3 || sweeps <= 0) return NPBX_OK;
  NPBX_REQUIRE(A != nullptr, "seidel2d: null array");
  NPBX_TRY(seidel_failure());
  const hipStream_t s = as_stream(stream);
  if (N <= kSmallN) {
    for (int64_t done = 0; done < sweeps; done += kSmallSweeps) {
      hipLaunchKernelGGL(seidel2d_small, dim3(1), dim3(64), 0, s, static_cast<double*>(A),
                         static_cast<int>(N),
                         static_cast<int>(std::min(kSmallSweeps, sweeps - done)));
      NPBX_LAUNCHED("seidel2d_small");
    }
    return NPBX_OK;
  }
  SeidelArgs g{};
  g.A = static_cast<double*>(A);
  g.n = static_cast<int>(N);
  g.bands = static_cast<int>(cdiv(N - 2 + kW - 1, 64));
  const int tiles = std::min(kMaxTiles, std::max(1, g_seidel_blocks.load()));
  const int64_t per_launch = int64_t(std::max(1, tiles / g.bands)) * kW;
  const bool chained = !capturing(s);
  for (int64_t done = 0; done < sweeps; done += per_launch) {
    g.sweeps = static_cast<int>(std::min(per_launch, sweeps - done));
    g.groups = static_cast<int>(cdiv(g.sweeps, kW));
    bool launched = false;
    if (chained) NPBX_TRY(launch_chained(g, s, launched));
    if (!launched) NPBX_TRY(launch_slots(g, s));
  }
  return NPBX_OK;
}
