// 3-D 7-point explicit heat sweeps (heat_3d_numpy.py:4-20).
//
// Layout: N x N x N, C order (i slowest, k contiguous).  A sweep writes the
// interior [1, N-2]^3 of dst from src; boundary faces are never written.
//
// Plain sweep (2.5-D): each lane owns V consecutive k, a wave spans 64*V k, a
// 256-thread workgroup is one wave-row x 4 j-rows, and each thread marches
// along i over kPlanes planes carrying the i-1 / i / i+1 vectors in registers.
// Loads for kUnroll planes (i+1, j+-1 vectors and the two k-edge scalars) are
// issued before any of them is used.  The j+-1 rows and k edges are L1/L2
// hits.  Tiles are numbered XCD by XCD (xcd_tile) so neighbours share an L2.
// Each src element crosses HBM about once per sweep.  Accesses ask only for
// the elements' own alignment, so any side and any base take this form.
//
// Arithmetic (points.h): the FP64 drop-in follows the reference order, per
// axis 0.125*((x[+1] - 2*c) + x[-1]), the axis terms summed i, j, k left to
// right, then + c; FP32 arithmetic uses the 7-operation form of the same map.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "points.h"
#include "tiles.h"
#include "vecio.h"

namespace npbx {
namespace {

constexpr int kLanes = 64;
constexpr int kCols = 4;
constexpr int kRows = 16;

// One point a lane, 16 planes, the grid's own block order: BF16 sides of 129 to
// 194 and sides whose rows leave much of the last vectors empty (run_sweeps).
template <class S>
__global__ __launch_bounds__(kLanes* kCols) void heat3d_sweep(const S* __restrict__ src,
                                                             S* __restrict__ dst, int n) {
  using T = Storage<S>;
  using C = typename T::C;
  const int k = 1 + blockIdx.x * kLanes + threadIdx.x;
  const int j = 1 + blockIdx.y * kCols + threadIdx.y;
  const int i0 = 1 + blockIdx.z * kRows;
  if (k > n - 2 || j > n - 2) return;
  const int i_end = min(i0 + kRows, n - 1);
  const int64_t plane = static_cast<int64_t>(n) * n;
  int64_t p = static_cast<int64_t>(i0) * plane + static_cast<int64_t>(j) * n + k;
  C below = T::load(src[p - plane]);  // i - 1
  C centre = T::load(src[p]);
  for (int i = i0; i < i_end; ++i, p += plane) {
    const C above = T::load(src[p + plane]);  // i + 1
    const C jp = T::load(src[p + n]);
    const C jm = T::load(src[p - n]);
    const C kp = T::load(src[p + 1]);
    const C km = T::load(src[p - 1]);
    dst[p] = T::store(heat_point<C>(centre, above, below, jp, jm, kp, km));
    below = centre;
    centre = above;
  }
}

// The first column a wave takes: vectors start with the row, single points
// with its interior, so that 64 m + 2 points take m waves.
__host__ __device__ constexpr int first_column(int v) { return v == 1 ? 1 : 0; }
int k_tiles(int n, int v) {
  return static_cast<int>(cdiv(n - 2 * first_column(v), kLanes * v));
}

// kPlanes = planes per workgroup (i segment); kUnroll = planes whose loads
// are issued together (run_sweeps below).  A row's last vector is shifted
// back to end with it where vectors do not divide the row; it shares points,
// with the same values, with the one before.
template <class S, int V, int kPlanes, int kUnroll>
__device__ __forceinline__ void sweep_tile(const S* __restrict__ src, S* __restrict__ dst, int n,
                                           int tiles_k, int tiles_j, int t) {
  using T = Storage<S>;
  using C = typename T::C;
  const int tk = t % tiles_k;
  const int tj = (t / tiles_k) % tiles_j;
  const int ti = t / (tiles_k * tiles_j);
  const int kv = (tk * kLanes + threadIdx.x) * V + first_column(V);
  const int j = 1 + tj * kCols + threadIdx.y;
  const int i0 = 1 + ti * kPlanes;
  if (kv >= n - first_column(V) || j > n - 2) return;
  const int k0 = min(kv, n - V);
  const int i_end = min(i0 + kPlanes, n - 1);
  const int64_t plane = static_cast<int64_t>(n) * n;
  const int64_t col = static_cast<int64_t>(j) * n + k0;
  const bool has_km = k0 > 0, has_kp = k0 + V < n;
  const bool full = k0 >= 1 && k0 + V <= n - 1;  // all V points interior in k
  auto load = [&](const S* p, C(&x)[V]) {
    S raw[V];
    __builtin_memcpy(raw, p, sizeof(raw));
#pragma unroll
    for (int v = 0; v < V; ++v) x[v] = T::load(raw[v]);
  };

  C below[V], centre[V];
  load(src + col + (i0 - 1) * plane, below);
  load(src + col + i0 * plane, centre);
  for (int i = i0; i < i_end; i += kUnroll) {
    C above[kUnroll][V], jp[kUnroll][V], jm[kUnroll][V], km[kUnroll], kp[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      // clamp so the loads of planes past the segment end stay in bounds
      const int64_t q = col + min(i + u, n - 2) * plane;
      load(src + q + plane, above[u]);
      load(src + q + n, jp[u]);
      load(src + q - n, jm[u]);
      km[u] = has_km ? T::load(src[q - 1]) : C(0);
      kp[u] = has_kp ? T::load(src[q + V]) : C(0);
    }
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      if (i + u >= i_end) break;
      C out[V];
#pragma unroll
      for (int v = 0; v < V; ++v) {
        const C left = v == 0 ? km[u] : centre[v - 1];
        const C right = v == V - 1 ? kp[u] : centre[v + 1];
        out[v] = heat_point<C>(centre[v], above[u][v], below[v], jp[u][v], jm[u][v], right, left);
      }
      S* o = dst + col + static_cast<int64_t>(i + u) * plane;
      if (full) {
        if constexpr (V == 1)
          *o = T::store(out[0]);
        else  // (BF16: two conversions an instruction; 512^3 204 -> 177 us a sweep)
          storev_any<S, V>(o, out);
      } else {
#pragma unroll
        for (int v = 0; v < V; ++v)
          if (k0 + v >= 1 && k0 + v <= n - 2) o[v] = T::store(out[v]);
      }
#pragma unroll
      for (int v = 0; v < V; ++v) {
        below[v] = centre[v];
        centre[v] = above[u][v];
      }
    }
  }
}

template <class S, int V, int kPlanes, int kUnroll>
__global__ __launch_bounds__(kLanes* kCols) void heat3d_sweep_vec(const S* __restrict__ src,
                                                                 S* __restrict__ dst, int n,
                                                                 int tiles_k, int tiles_j) {
  sweep_tile<S, V, kPlanes, kUnroll>(src, dst, n, tiles_k, tiles_j,
                                     xcd_tile(blockIdx.x, gridDim.x));
}

// One sweep of up to kMaxBatch grids: tile t of the launch belongs to the grid
// g with cum[g] <= t < cum[g+1].  `form` is the grid's kernel form (batch_form).
struct HeatBatch {
  int32_t count;
  int32_t cum[kMaxBatch + 1];
  struct {
    const void* src;
    void* dst;
    int32_t n, tiles_k, tiles_j, form;
  } grid[kMaxBatch];
};

// The forms of a batch's grids by type: points a lane, planes, planes ahead.
struct Form {
  int v, planes;
};
template <class S>
struct BatchForms;
template <>
struct BatchForms<double> {
  static constexpr Form form[3] = {{2, 2}, {2, 4}, {2, 8}};
  static constexpr int ahead[3] = {2, 4, 4};
};
template <>
struct BatchForms<float> {
  static constexpr Form form[3] = {{1, 1}, {1, 4}, {1, 8}};
  static constexpr int ahead[3] = {1, 4, 4};
};
template <>
struct BatchForms<bf16> {
  static constexpr Form form[3] = {{2, 2}, {4, 2}, {8, 4}};
  static constexpr int ahead[3] = {2, 2, 2};
};

template <class S>
__global__ __launch_bounds__(kLanes* kCols) void heat3d_sweep_batch(const HeatBatch b) {
  using F = BatchForms<S>;
  const int t = xcd_tile(blockIdx.x, gridDim.x);
  int lo = 0, hi = b.count - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (b.cum[mid] <= t) lo = mid; else hi = mid - 1;
  }
  const auto& g = b.grid[lo];
  const S* src = static_cast<const S*>(g.src);
  S* dst = static_cast<S*>(g.dst);
  const int tile = t - b.cum[lo];
  if (g.form == 0)
    sweep_tile<S, F::form[0].v, F::form[0].planes, F::ahead[0]>(src, dst, g.n, g.tiles_k,
                                                                g.tiles_j, tile);
  else if (g.form == 1)
    sweep_tile<S, F::form[1].v, F::form[1].planes, F::ahead[1]>(src, dst, g.n, g.tiles_k,
                                                                g.tiles_j, tile);
  else
    sweep_tile<S, F::form[2].v, F::form[2].planes, F::ahead[2]>(src, dst, g.n, g.tiles_k,
                                                                g.tiles_j, tile);
}

// A batch's grids take the forms that a single grid of as many points takes
// (run_sweeps); BF16's follow the row length, which its vectors have to fill.
int batch_form(int dtype, int n, int64_t points) {
  if (dtype == NPBX_BF16) return n <= 128 ? 0 : n <= 256 ? 1 : 2;
  const int64_t lo = dtype == NPBX_F64 ? 112 : 56, hi = dtype == NPBX_F64 ? 176 : 112;
  return points <= lo * lo * lo ? 0 : points <= hi * hi * hi ? 1 : 2;
}

// Grids are swept in groups that fit the Infinity Cache with both arrays, one
// group after the other: a sweep of more runs at HBM's rate (FP32, 256^3 grids:
// 8 in one launch 303 us a sweep, 1 at a time 25).
constexpr int64_t kGroupBytes = int64_t(256) << 20;

template <class S>
int group_sweeps(int dtype, const SweepGrid* grids, size_t count, bool enqueue,
                 hipStream_t stream, int64_t* launches, int64_t* tiles) {
  int64_t sweeps = 0;
  for (size_t i = 0; i < count; ++i) sweeps = std::max(sweeps, grids[i].nsweeps);
  for (int64_t s = 0; s < sweeps; ++s) {
    int64_t points = 0;
    for (size_t i = 0; i < count; ++i)
      if (s < grids[i].nsweeps) points += int64_t(grids[i].n) * grids[i].n * grids[i].n;
    HeatBatch b;
    b.count = 0;
    b.cum[0] = 0;
    for (size_t i = 0; i <= count; ++i) {
      if (b.count == kMaxBatch || (i == count && b.count > 0)) {
        const int blocks = b.cum[b.count];
        *launches += 1;
        *tiles += blocks;
        if (enqueue) {
          hipLaunchKernelGGL(heat3d_sweep_batch<S>, dim3(static_cast<unsigned>(blocks)),
                             dim3(kLanes, kCols), 0, stream, b);
          NPBX_LAUNCHED("heat3d_sweep_batch");
        }
        b.count = 0;
      }
      if (i == count || s >= grids[i].nsweeps) continue;
      const SweepGrid& g = grids[i];
      const int form = batch_form(dtype, g.n, points);
      const Form f = BatchForms<S>::form[form];
      const bool even = ((g.first + s) & 1) == 0;
      auto& d = b.grid[b.count];
      d.src = even ? g.A : g.B;
      d.dst = even ? g.B : g.A;
      d.n = g.n;
      d.form = form;
      d.tiles_k = k_tiles(g.n, f.v);
      d.tiles_j = static_cast<int32_t>(cdiv(g.n - 2, kCols));
      const int64_t nt = int64_t(d.tiles_k) * d.tiles_j * cdiv(g.n - 2, f.planes);
      NPBX_REQUIRE(b.cum[b.count] + nt < (int64_t(1) << 31), "heat batch: too many tiles");
      b.cum[b.count + 1] = b.cum[b.count] + static_cast<int32_t>(nt);
      ++b.count;
    }
  }
  return NPBX_OK;
}

template <class S>
int batch_sweeps(int dtype, const std::vector<SweepGrid>& grids, bool enqueue,
                 hipStream_t stream, int64_t* launches, int64_t* tiles) {
  auto bytes = [](const SweepGrid& g) {
    return 2 * int64_t(sizeof(S)) * g.n * g.n * g.n;
  };
  for (size_t i = 0; i < grids.size();) {
    int64_t total = bytes(grids[i]);
    size_t end = i + 1;
    while (end < grids.size() && total + bytes(grids[end]) <= kGroupBytes)
      total += bytes(grids[end++]);
    NPBX_TRY(group_sweeps<S>(dtype, &grids[i], end - i, enqueue, stream, launches, tiles));
    i = end;
  }
  return NPBX_OK;
}

template <class S, int V, int kPlanes, int kUnroll>
int run_vec(S* A, S* B, int n, int64_t first, int64_t nsweeps, hipStream_t stream) {
  const dim3 block(kLanes, kCols);
  const int tiles_k = k_tiles(n, V);
  const int tiles_j = static_cast<int>(cdiv(n - 2, kCols));
  const int tiles_i = static_cast<int>(cdiv(n - 2, kPlanes));
  const int64_t nblocks = int64_t(tiles_k) * tiles_j * tiles_i;
  NPBX_REQUIRE(nblocks < (int64_t(1) << 31), "heat3d: grid too large");
  for (int64_t s = first; s < first + nsweeps; ++s) {
    const bool even = (s % 2) == 0;
    hipLaunchKernelGGL((heat3d_sweep_vec<S, V, kPlanes, kUnroll>),
                       dim3(static_cast<unsigned>(nblocks)), block, 0, stream, even ? A : B,
                       even ? B : A, n, tiles_k, tiles_j);
    NPBX_LAUNCHED("heat3d_sweep_vec");
  }
  return NPBX_OK;
}

template <class S>
int run_points(S* A, S* B, int n, int64_t first, int64_t nsweeps, hipStream_t stream) {
  const dim3 block(kLanes, kCols);
  const dim3 grid(static_cast<unsigned>(cdiv(n - 2, kLanes)),
                  static_cast<unsigned>(cdiv(n - 2, kCols)),
                  static_cast<unsigned>(cdiv(n - 2, kRows)));
  for (int64_t s = first; s < first + nsweeps; ++s) {
    const bool even = (s % 2) == 0;
    hipLaunchKernelGGL(heat3d_sweep<S>, grid, block, 0, stream, even ? A : B, even ? B : A, n);
    NPBX_LAUNCHED("heat3d_sweep");
  }
  return NPBX_OK;
}

// The sweeps in the launch shape of the setting "sweep.shape" where that is
// not 0, else by size.  A march over planes is a chain of load latencies, so
// it is as short as leaves the chip some waves to switch between; from about
// 128^3 on it saves loads of planes i-1 and i.  Narrow vectors fill a wave's
// lanes on short rows, and FP32 keeps them: with one point a lane a row's
// accesses are whole lines and the k-edge scalars hit the same ones.
// Past the Infinity Cache a sweep's time goes with the waves a row takes, whether
// or not points fill them, so there the count decides between vectors and single
// points: FP64 385^3 takes four waves of vectors or six of points, 348 | 283 us;
// FP32 keeps points but where rows are whole multiples of 256, whose planes then
// fall on few channels (512^3 350 | 4x8/4 314).
// Measured, us per sweep, V points a lane x planes / ahead (1x16: heat3d_sweep):
//   FP64       2x1/1  2x2/2  2x4/4  2x8/4  2x16/4   1x16
//     64^3       3.7    3.7    3.7    4.9    7.6
//     101^3      6.3    6.1    6.3    7.1    8.4
//     160^3     18.3   17.4   16.8   17.5   19.6    19.8
//     201^3     29.1   27.6   25.8   25.7   29.8
//     385^3             372    349    346    351     283
//     400^3             385    358    356    361     344
//     512^3      723    678    626    612    626     665
//   FP32       2x1/1  1x4/4  1x8/4  4x4/4   4x8/4  4x16/4   1x16
//     64^3       3.5    3.2    3.8    3.9             8.5
//     101^3      5.2    4.7    5.1    5.5             8.5
//     201^3     20.9   18.4   14.8   15.6            18.2
//     256^3     32.0   27.1   23.0   25.1    25.6    26.3     39
//     384^3             125    123    167     166     165    144
//     512^3             322    353    316     315     320    378
//   BF16       2x2/2  4x2/2  8x4/2  8x8/4   4x8/4   1x16
//     100^3      5.0    5.9    7.8   11.0     9.2    7.6
//     176^3     13.8   11.3   13.6   13.7    12.4   10.9
//     200^3     16.7   13.0   15.5   15.9    14.2   16.7
//     258^3     36.7   34.8   23.1   25.9    31.6   26.6
//     400^3      114     79     54     58      69     88
//     512^3      272    201    176    176     185    237
//     513^3      332    276    328    323     247    199
//     700^3      755    549    615    596     500    562
//     1024^3    2217   1625   1382   1289    1454   2122
template <class S>
int run_sweeps(S* A, S* B, int n, int64_t first, int64_t nsweeps, hipStream_t stream) {
  constexpr int N = Vec16<S>::N;
  if (n >= N) {
    switch (sweep_shape()) {
      case 1: return run_vec<S, N, 16, 8>(A, B, n, first, nsweeps, stream);
      case 2: return run_vec<S, N, 32, 8>(A, B, n, first, nsweeps, stream);
      case 3: return run_vec<S, N, 8, 4>(A, B, n, first, nsweeps, stream);
      default: break;
    }
  }
  const auto waves = [n](int v) { return k_tiles(n, v); };  // a row's
  if (n <= 88) return run_vec<S, 2, 1, 1>(A, B, n, first, nsweeps, stream);
  if constexpr (std::is_same_v<S, double>) {
    if (n <= 112) return run_vec<S, 2, 2, 2>(A, B, n, first, nsweeps, stream);
    // rows of 129 to 194 points fill two or three waves of single points:
    // 129^3 9.7 us (vectors of two 11.4, 16 planes a thread 10.6), 177^3 20.3 | 20.7
    if (n <= 128) return run_vec<S, 2, 4, 4>(A, B, n, first, nsweeps, stream);
    if (n <= 194) return run_vec<S, 1, 4, 4>(A, B, n, first, nsweeps, stream);
    if (n >= 330 && 3.2 * waves(1) < 5.7 * waves(2))
      return run_points<S>(A, B, n, first, nsweeps, stream);
    return run_vec<S, 2, 8, 4>(A, B, n, first, nsweeps, stream);
  } else if constexpr (std::is_same_v<S, float>) {
    if (n <= 112) return run_vec<S, 1, 4, 4>(A, B, n, first, nsweeps, stream);
    if (n >= 512 && n % 256 == 0) return run_vec<S, 4, 8, 4>(A, B, n, first, nsweeps, stream);
    return run_vec<S, 1, 8, 4>(A, B, n, first, nsweeps, stream);
  } else {
    if (n <= 128) return run_vec<S, 2, 2, 2>(A, B, n, first, nsweeps, stream);
    if (n <= 194) return run_points<S>(A, B, n, first, nsweeps, stream);
    if (n <= 256) return run_vec<S, 4, 2, 2>(A, B, n, first, nsweeps, stream);
    if (n <= 448) return run_vec<S, 8, 4, 2>(A, B, n, first, nsweeps, stream);
    // odd rows put vectors across lines
    const double v8 = (n % 2 ? 7.3 : 6.5) * waves(8), v4 = (n % 2 ? 3.6 : 3.35) * waves(4);
    const double v1 = 1.03 * waves(1);
    if (v1 < std::min(v4, v8)) return run_points<S>(A, B, n, first, nsweeps, stream);
    if (v4 < v8) return run_vec<S, 4, 8, 4>(A, B, n, first, nsweeps, stream);
    return run_vec<S, 8, 8, 4>(A, B, n, first, nsweeps, stream);
  }
}

int heat_entry(int dtype, void* A, void* B, int64_t N, int64_t first, int64_t nsweeps, int tblock,
               void* stream) {
  NPBX_REQUIRE(N >= 0 && N <= 4096, "heat3d: N=%lld out of range", static_cast<long long>(N));
  NPBX_REQUIRE(nsweeps >= 0 && first >= 0, "heat3d: negative sweep count");
  NPBX_REQUIRE(tblock >= 0, "heat3d: negative tblock");
  if (N < 3 || nsweeps == 0) return NPBX_OK;
  NPBX_REQUIRE(A && B, "heat3d: null array");
  NPBX_REQUIRE(A != B, "heat3d: A and B must be distinct arrays");
  hipStream_t s = as_stream(stream);
  if (tblock >= 2)
    return tiled_sweeps(1, dtype, A, B, static_cast<int>(N), first, nsweeps, tblock, 0, s);
  return dispatch_dtype(dtype, [&](auto tag) {
    using S = decltype(tag);
    return run_sweeps<S>(static_cast<S*>(A), static_cast<S*>(B), static_cast<int>(N), first,
                         nsweeps, s);
  });
}

}  // namespace

int heat_batch_sweeps(int dtype, const std::vector<SweepGrid>& grids, bool enqueue,
                      hipStream_t stream, int64_t* launches, int64_t* tiles) {
  return dispatch_dtype(dtype, [&](auto tag) {
    return batch_sweeps<decltype(tag)>(dtype, grids, enqueue, stream, launches, tiles);
  });
}

}  // namespace npbx

extern "C" int npbx_heat3d(int dtype, void* A, void* B, int64_t N, int64_t tsteps, int tblock,
                           void* stream) {
  const int64_t iters = tsteps > 1 ? tsteps - 1 : 0;  // for t in range(1, TSTEPS)
  return npbx::heat_entry(dtype, A, B, N, 0, 2 * iters, tblock, stream);
}

extern "C" int npbx_heat3d_sweeps(int dtype, void* A, void* B, int64_t N, int64_t first,
                                  int64_t nsweeps, int tblock, void* stream) {
  return npbx::heat_entry(dtype, A, B, N, first, nsweeps, tblock, stream);
}
