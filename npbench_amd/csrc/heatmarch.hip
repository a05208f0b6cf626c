// Heat sweeps of many FP32 grids, temporal-blocked: the rounds of a batch
// plan's grids on one wave-stacked tile form.
//
// A workgroup of 8 waves holds a tile of 32 rows (j) x 256 columns (k), each
// wave 4 rows and each lane 4 adjacent columns of them, and marches along i.
// Level l keeps per row a[l], its values at its newest plane q, and part[l],
// the five-term partial sums (heat_partial) of level l+1 at plane q.  A step
// takes one level-0 plane: it finishes plane P-1 of level 1 (heat_finish),
// that one plane P-2 of level 2, and so on to the output plane P-D -- nothing
// of which needs a neighbour -- and then, after one barrier, forms the new
// partial sums, for which each wave's edge rows were passed through LDS and
// columns cross lanes by full-wave DPP shifts.  So depth costs no barriers, and
// a wave's state, 2 D planes of 4 rows and three level-0 planes (the newest, the
// one before and one in flight, which the three-fold unrolled loop rotates
// through by name), stays under 256 VGPRs: two waves per SIMD cover each
// other's waits.  The wave-private tile (tiles.hip) keeps all rows of a tile in
// one wave, past 256 VGPRs, and spends half its instructions moving them.
//
// A tile ends with the grid where it can (no halo rows beyond a boundary: the
// first tile starts at row 0, the last ends at row n-1), so a boundary row is
// the first row of the first wave or the last of the last.  Global-boundary
// points of level L hold A's (L even) or B's (L odd) values.  EQ: A's and B's
// boundaries are equal (the packed columns' flag), so a produced plane's
// boundary points are the previous level's at the same plane.  Otherwise
// both arrays' boundary columns (from the packed copy) and rows of the last
// planes are kept in LDS.
//
// Work: the planes of all columns of tiles in one list, an equal contiguous
// part for each workgroup, one workgroup per CU.  A part that spans two columns
// pays the 2 D filling planes twice; whole tiles would leave a third of the
// chip idle in the last turn (8 grids of 256^3: 88 columns).
//
// 8 grids of 256^3, B = A.copy(), depth 4: 246 us a launch, 64 us a sweep
// (2100 G updates/s; wave-private tiles of depth 3: 90 us).  What bounds it: a
// step is about 600 instructions of each of two waves a SIMD, 448 of them the
// update's, 104 steps a part -- 200 us of issue -- and the launch moves some 1.3
// GB (halo rows of neighbouring columns meet in L2 only in part), near a copy's
// rate.  Depth 3 takes 82 us a sweep; stores past the caches 90.  With A's and
// B's boundaries different 92 us (wave-private tiles: 133).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "common.h"
#include "lanes.h"
#include "points.h"
#include "tiles.h"
#include "vecio.h"

namespace npbx {
namespace {

constexpr int V = 4;                // columns per lane
constexpr int R = 4;                // rows per wave
constexpr int W = 8;                // waves
constexpr int kRows = R * W;        // rows of a tile
constexpr int kCols = 64 * V;       // columns of a tile
constexpr int kMaxDepth = kHeatMarchDepth;

struct alignas(16) Quad {
  float v[V];
};
// LDS of a workgroup: by step parity and level each wave's first and last row;
// by plane (mod 8) and array, where A's and B's boundaries differ, the tile's
// rows' columns 0 and n-1 and its boundary row.
constexpr int kRing = 8;
struct MarchLds {
  Quad edge[2][kMaxDepth][W][2][64];
  Quad cols[kRing][2][2][W];  // a wave's 4 rows
  Quad row[kRing][2][64];
};

template <int D, bool EQ>
__device__ __forceinline__ void march(const GridRound& g, int column, int i0, int i1,
                                      MarchLds& lds) {
  auto& edge = lds.edge;
  const int n = g.n;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tk = column % g.tiles_k, tj = column / g.tiles_k;
  const bool last_j = tj == g.tiles_j - 1;
  const int nominal = tj * (kRows - 2 * D);
  const int tile_row = last_j ? n - kRows : nominal;
  const int row0 = tile_row + w * R;  // the wave's first row
  const int jlo = tj == 0 ? 1 : nominal + D, jhi = last_j ? n - 1 : nominal + kRows - D;
  const bool top = tj == 0 && w == 0, bottom = last_j && w == W - 1;
  int kl = 0, klo = 1, khi = n - 1;
  if (g.tiles_k > 1) {
    kl = tk * (kCols - 2 * V) - V;
    klo = max(kl + V, 1);
    khi = min(kl + kCols - V, n - 1);
  }
  const int k0 = kl + lane * V;
  const bool live = k0 >= 0 && k0 + V <= n;
  const uint32_t lob = live ? static_cast<uint32_t>(k0) * 4u : 0u;
  const bool store_any = live && k0 + V > klo && k0 < khi;
  const bool is_k0 = live && k0 == 0, is_kn = live && k0 + V == n;
  const int64_t plane = static_cast<int64_t>(n) * n;
  const float* X = static_cast<const float*>(g.X);
  float* Y = static_cast<float*>(g.Y);
  const float* gA = static_cast<const float*>(g.A);
  const float* gB = static_cast<const float*>(g.B);
  auto parity = [&](int level) { return (g.parity0 + level) & 1; };
  auto bsrc = [&](int level) { return parity(level) ? gB : gA; };
  auto clamped = [&](int q) { return min(max(q, 0), n - 1); };
  auto plane_of = [&](const float* base, int q) {
    return plane_rsrc(base + clamped(q) * plane, plane);
  };
  const uint32_t row_bytes = static_cast<uint32_t>(n) * 4u;
  auto rowoff = [&](int r) { return static_cast<uint32_t>(row0 + r) * row_bytes; };

  // The boundary values of plane P of both arrays (not EQ), loaded to LDS two
  // steps ahead of level 0: threads 0 .. 127 one column value each, the wave
  // that has the boundary row both arrays' rows.  Level m's come from the array
  // of its parity, by the plane.
  struct Bnd {
    float col;
    float row[2][V];
  };
  const int t = threadIdx.x;
  const int carr = (t >> 6) & 1, cside = (t >> 5) & 1, crow = t & 31;
  auto fetch_bnd = [&](int P, Bnd& x) {
    if (w < 2)
      x.col = static_cast<const float*>(
          g.cols)[((carr * static_cast<int64_t>(n) + clamped(P)) * n + tile_row + crow) * 2 +
                  cside];
    if (top || bottom) {
      buf_load16(plane_of(gA, P), lob, rowoff(top ? 0 : R - 1), x.row[0]);
      buf_load16(plane_of(gB, P), lob, rowoff(top ? 0 : R - 1), x.row[1]);
    }
  };
  auto keep_bnd = [&](int P, const Bnd& x) {
    if (w < 2) lds.cols[P & (kRing - 1)][carr][cside][crow / R].v[crow % R] = x.col;
    if (top || bottom) {
#pragma unroll
      for (int arr = 0; arr < 2; ++arr) {
        Quad y;
#pragma unroll
        for (int v = 0; v < V; ++v) y.v[v] = x.row[arr][v];
        lds.row[P & (kRing - 1)][arr][lane] = y;
      }
    }
  };
  auto patch_cols = [&](float (&x)[R][V], int m, int q) {
    const Quad c = lds.cols[q & (kRing - 1)][parity(m)][is_kn ? 1 : 0][w];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      x[r][0] = is_k0 ? c.v[r] : x[r][0];
      x[r][V - 1] = is_kn ? c.v[r] : x[r][V - 1];
    }
  };
  auto load_plane = [&](int P, float (&x)[R][V]) {
    if constexpr (EQ) {
      const Rsrc rx = plane_of(X, P);
#pragma unroll
      for (int r = 0; r < R; ++r) buf_load16(rx, lob, rowoff(r), x[r]);
    } else {
      const float* b = bsrc(0);
      const Rsrc rx = plane_of(P <= 0 || P >= n - 1 ? b : X, P), rb = plane_of(b, P);
#pragma unroll
      for (int r = 0; r < R; ++r)
        buf_load16((r == 0 && top) || (r == R - 1 && bottom) ? rb : rx, lob, rowoff(r), x[r]);
    }
  };

  float f[3][R][V];      // level-0 planes
  float a[D][R][V];      // levels 1 .. D-1 at their newest plane
  float part[D][R][V];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int v = 0; v < V; ++v) {
      f[2][r][v] = 0.0f;
#pragma unroll
      for (int l = 0; l < D; ++l) a[l][r][v] = part[l][r][v] = 0.0f;
    }

  auto step = [&](int P, float (&in0)[R][V], float (&a0)[R][V]) {
    const int par = P & 1;
    float lv[D][R][V];  // the arriving plane of each level
    if constexpr (!EQ) patch_cols(in0, 0, P);
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int v = 0; v < V; ++v) lv[0][r][v] = in0[r][v];
#pragma unroll
    for (int l = 0; l < D; ++l) {
      const float(&al)[R][V] = l == 0 ? a0 : a[l];
      Quad e0, e1;
#pragma unroll
      for (int v = 0; v < V; ++v) e0.v[v] = lv[l][0][v], e1.v[v] = lv[l][R - 1][v];
      edge[par][l][w][0][lane] = e0;
      edge[par][l][w][1][lane] = e1;
      const int m = l + 1, q = P - m;
      float o[R][V];
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int v = 0; v < V; ++v) {
          o[r][v] = heat_finish(part[l][r][v], lv[l][r][v], al[r][v]);
          // computed here: sunk into the branches below it leaves copies of al
          asm volatile("" : "+v"(o[r][v]));
        }
      if (m == D) {
        if constexpr (EQ) {
#pragma unroll
          for (int r = 0; r < R; ++r) {
            o[r][0] = is_k0 ? al[r][0] : o[r][0];
            o[r][V - 1] = is_kn ? al[r][V - 1] : o[r][V - 1];
          }
        }
        if (q >= i0 && q < i1) {
          char* yq = reinterpret_cast<char*>(Y + static_cast<int64_t>(q) * plane);
#pragma unroll
          for (int r = 0; r < R; ++r) {
            if (row0 + r < jlo || row0 + r >= jhi) continue;
            float* to = reinterpret_cast<float*>(yq + rowoff(r) + lob);
            if constexpr (EQ) {
              if (store_any) store16(to, o[r]);
            } else {
              // Y's own boundary columns stay
              if (store_any && !is_k0 && !is_kn) store16(to, o[r]);
              if (is_k0 || is_kn) {
                const int from = is_k0 ? 1 : 0;
#pragma unroll
                for (int v = 0; v < V - 1; ++v) to[from + v] = is_k0 ? o[r][v + 1] : o[r][v];
              }
            }
          }
        }
      } else {
        // a boundary plane, or one before or past the grid that feeds none
        const bool outside = q <= 0 || q >= n - 1;
        if constexpr (EQ) {
#pragma unroll
          for (int r = 0; r < R; ++r) {
            o[r][0] = is_k0 ? al[r][0] : o[r][0];
            o[r][V - 1] = is_kn ? al[r][V - 1] : o[r][V - 1];
          }
        } else {
          patch_cols(o, m, q);
        }
        // the rest in one branch: the common path has no copies to merge
        if (outside || top || bottom) {
          asm volatile("");
          if (!outside) {
            if constexpr (EQ) {
#pragma unroll
              for (int v = 0; v < V; ++v) (top ? o[0][v] : o[R - 1][v]) = (top ? al[0] : al[R - 1])[v];
            } else {
              const Quad c = lds.row[q & (kRing - 1)][parity(m)][lane];
#pragma unroll
              for (int v = 0; v < V; ++v) (top ? o[0][v] : o[R - 1][v]) = c.v[v];
            }
          } else if constexpr (EQ) {
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
              for (int v = 0; v < V; ++v) o[r][v] = al[r][v];
          } else {
            const Rsrc rb = plane_of(bsrc(m), q);
#pragma unroll
            for (int r = 0; r < R; ++r) buf_load16(rb, lob, rowoff(r), o[r]);
            // the wait here keeps the compiler from waiting on the common path
            __builtin_amdgcn_s_waitcnt(0);
          }
        }
        if constexpr (D > 1) {
          constexpr int kLast = D - 1;
          const int nxt = m < kLast ? m : kLast;
#pragma unroll
          for (int r = 0; r < R; ++r)
#pragma unroll
            for (int v = 0; v < V; ++v) lv[nxt][r][v] = o[r][v];
        }
      }
    }
    lds_barrier();
    Bnd bnd;
    if constexpr (!EQ) fetch_bnd(P + 2, bnd);
    const int wu = max(w - 1, 0), wd = min(w + 1, W - 1);  // a tile's outer rows feed only halo
    // a level's edges are asked for a level ahead, and rows that need none go first
    Quad up[2], dn[2];
    auto read_edges = [&](int l) {
      up[l & 1] = edge[par][l][wu][1][lane];
      dn[l & 1] = edge[par][l][wd][0][lane];
    };
    read_edges(0);
#pragma unroll
    for (int l = 0; l < D; ++l) {
      float(&al)[R][V] = l == 0 ? a0 : a[l];
      if (l + 1 < D) read_edges(l + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int rr = 0; rr < R; ++rr) {
        const int r = rr + 1 < R ? rr + 1 : 0;
        if (rr == R - 2) __builtin_amdgcn_sched_barrier(0);
        const float left = lane_from_left(lv[l][r][V - 1]);
        const float right = lane_from_right(lv[l][r][0]);
#pragma unroll
        for (int v = 0; v < V; ++v)
          part[l][r][v] = heat_partial(al[r][v], r == 0 ? up[l & 1].v[v] : lv[l][r - 1][v],
                                       r == R - 1 ? dn[l & 1].v[v] : lv[l][r + 1][v],
                                       v == 0 ? left : lv[l][r][v - 1],
                                       v == V - 1 ? right : lv[l][r][v + 1]);
      }
      if (l > 0) {
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int v = 0; v < V; ++v) al[r][v] = lv[l][r][v];
      }
    }
    if constexpr (!EQ) keep_bnd(P + 2, bnd);
    load_plane(P + 2, a0);
  };

  const int begin = max(i0 - D, 0), end = i1 - 1 + D;
  load_plane(begin, f[0]);
  load_plane(begin + 1, f[1]);
  if constexpr (!EQ) {
    for (int P = begin; P < begin + 2; ++P) {
      Bnd bnd;
      fetch_bnd(P, bnd);
      keep_bnd(P, bnd);
    }
    __syncthreads();
  }
  // whole turns of three: a break between the steps would cost copies of the
  // planes and a wait for those in flight; steps past the end store nothing
  for (int P = begin; P <= end; P += 3) {
    step(P, f[0], f[2]);
    step(P + 1, f[1], f[0]);
    step(P + 2, f[2], f[1]);
  }
}

// cum counts planes of tile columns; `part` of them for each workgroup.
__global__ __launch_bounds__(64 * W, 2) void heat_march(const RoundBatch b, int part) {
  __shared__ MarchLds lds;
  const int total = b.cum[b.count];
  int at = xcd_tile(blockIdx.x, gridDim.x) * part;
  const int end = min(at + part, total);
  while (at < end) {
    int lo = 0, hi = b.count - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (b.cum[mid] <= at) lo = mid; else hi = mid - 1;
    }
    const GridRound& g = b.round[lo];
    const int planes = g.n - 2, local = at - b.cum[lo];
    const int column = local / planes, first = local % planes;
    const int count = min(end - at, planes - first);
    const bool eq = *reinterpret_cast<const int*>(static_cast<const float*>(g.cols) +
                                                  4 * static_cast<int64_t>(g.n) * g.n) != 0;
    auto run = [&](auto depth) {
      constexpr int D = decltype(depth)::value;
      if (eq)
        march<D, true>(g, column, 1 + first, 1 + first + count, lds);
      else
        march<D, false>(g, column, 1 + first, 1 + first + count, lds);
    };
    switch (g.depth) {
      case 1: run(std::integral_constant<int, 1>{}); break;
      case 2: run(std::integral_constant<int, 2>{}); break;
      case 3: run(std::integral_constant<int, 3>{}); break;
      default: run(std::integral_constant<int, 4>{}); break;
    }
    at += count;
    __syncthreads();  // the next part writes the edges this one read
  }
}

}  // namespace

int heat_march_columns(int n, int depth, int* tiles_k, int* tiles_j) {
  *tiles_k = n <= kCols ? 1 : static_cast<int>(cdiv(n, kCols - 2 * V));
  *tiles_j = static_cast<int>(
      std::max<int64_t>(1, cdiv(n - 2 * depth, kRows - 2 * depth)));
  return *tiles_k * *tiles_j;
}

int heat_march_launch(const RoundBatch& b, int blocks, hipStream_t stream) {
  const int total = b.cum[b.count];
  const int part = static_cast<int>(cdiv(total, blocks));
  hipLaunchKernelGGL(heat_march, dim3(static_cast<unsigned>(cdiv(total, part))),
                     dim3(64 * W), 0, stream, b, part);
  NPBX_LAUNCHED("heat_march");
  return NPBX_OK;
}

}  // namespace npbx
