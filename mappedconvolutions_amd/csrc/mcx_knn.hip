// k nearest neighbours: a walk over all reference points with a streaming top-k, and (second
// half of the file) a search over a uniform grid for points of one to three dimensions that
// gives the same result bit for bit.  The reference
// (include/util/cuda/knn.cuh:43-275) materialises the R x Q matrix of squared
// distances and insertion-sorts each column with one thread; here one thread owns
// one query, walks the reference points once and keeps its k best in registers,
// so HBM traffic is just the inputs and the [k,Q] outputs.  Reference points are
// read through wave-uniform (scalar) loads: every lane needs the same point.
//
// Contract kept from the reference: squared distance accumulated over the
// dimensions in order with fused multiply-adds, candidates enter only if strictly
// closer than the current k-th and go before the first strictly larger entry (so
// ties keep the lower reference index first), indices are 1-based, distances are
// square-rooted at the end.
#include <algorithm>
#include <cmath>
#include <initializer_list>

#include "mcx_device.h"

namespace mcx {
namespace {

constexpr int kThreads = 256;

__host__ __device__ constexpr size_t align_up256(size_t v) { return (v + 255) & ~(size_t)255; }

// Grid search (second half of this file): per batch element, at the start of its workspace slice
// Workgroups (per batch element) that share the bounding box and the clearing of the counters;
// the counting launch puts the boxes together, a lane each.
constexpr int kBoxParts = 64;
template <typename T>
struct GridHead {
  T lo[3], inv_h[3], h[3];
  int skewed;  // nonzero: a quarter of the points share one cell; the plain walk runs instead
  T part_lo[3][kBoxParts], part_hi[3][kBoxParts];  // bounding boxes of runs of the points
};
template <typename T>
struct alignas(sizeof(T) * 4) GridPoint {
  T c[3];
  int idx;  // 1-based index of the reference point
};

__device__ inline float fma_t(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ inline double fma_t(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ inline float min_t(float a, float b) { return __builtin_fminf(a, b); }
__device__ inline double min_t(double a, double b) { return __builtin_fmin(a, b); }
__device__ inline float sqrt_t(float v) { return sqrtf(v); }
__device__ inline double sqrt_t(double v) { return sqrt(v); }

template <typename T>
__device__ inline T inf_t() { return (T)__builtin_huge_valf(); }

// DT > 0: compile-time dimension, query coordinates live in registers.
// DT == 0: any dimension, coordinates re-read from memory (slow path).
template <typename T, int KMAX, int DT>
__global__ __launch_bounds__(kThreads) void knn_kernel(const T *__restrict__ ref,
                                                       const T *__restrict__ query,
                                                       int64_t *__restrict__ idx,
                                                       T *__restrict__ dist, int D, int R, int Q,
                                                       int k, const char *__restrict__ grid_ws,
                                                       size_t grid_slice) {
  const int b = blockIdx.y;
  // launched behind a grid search: only for batch elements whose grid was not worth walking
  if (grid_ws &&
      !reinterpret_cast<const GridHead<T> *>(grid_ws + (size_t)b * grid_slice)->skewed)
    return;
  const int q = blockIdx.x * kThreads + threadIdx.x;
  const bool live = q < Q;
  const int qc = live ? q : Q - 1;
  const T *rb = ref + (int64_t)b * D * R;
  const T *qb = query + (int64_t)b * D * Q;

  T qv[DT > 0 ? DT : 1];
#pragma unroll
  for (int d = 0; d < DT; d++) qv[d] = qb[(int64_t)d * Q + qc];

  T bd[KMAX];
  int bi[KMAX];
#pragma unroll
  for (int j = 0; j < KMAX; j++) {
    bd[j] = inf_t<T>();
    bi[j] = 0;
  }

  auto ssd_of = [&](int r) {
    T ssd = T(0);
    if (DT > 0) {
#pragma unroll
      for (int d = 0; d < DT; d++) {
        const T t = rb[(int64_t)d * R + r] - qv[d];
        ssd = fma_t(t, t, ssd);
      }
    } else {
      for (int d = 0; d < D; d++) {
        const T t = rb[(int64_t)d * R + r] - qb[(int64_t)d * Q + qc];
        ssd = fma_t(t, t, ssd);
      }
    }
    return ssd;
  };
  auto insert = [&](T ssd, int r) {
    if (ssd < bd[KMAX - 1]) {
      T cd = ssd;
      int ci = r + 1;
      bool shifting = false;
#pragma unroll
      for (int j = 0; j < KMAX; j++) {
        shifting = shifting || (cd < bd[j]);
        if (shifting) {
          const T td = bd[j];
          const int ti = bi[j];
          bd[j] = cd;
          bi[j] = ci;
          cd = td;
          ci = ti;
        }
      }
    }
  };
  // Reference points are taken kBatch at a time: their distances are independent work
  // (the wave-uniform loads of the next points overlap the arithmetic), and a single
  // comparison of the batch minimum decides whether any lane has to insert at all.
  constexpr int kBatch = 8;
  int r = 0;
  for (; r + kBatch <= R; r += kBatch) {
    T ssd[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; u++) ssd[u] = ssd_of(r + u);
    T m = ssd[0];
#pragma unroll
    for (int u = 1; u < kBatch; u++) m = min_t(m, ssd[u]);  // (a NaN yields to a number)
    if (m < bd[KMAX - 1]) {
#pragma unroll
      for (int u = 0; u < kBatch; u++) insert(ssd[u], r + u);  // in index order: ties keep it
    }
  }
  for (; r < R; r++) insert(ssd_of(r), r);
  if (!live) return;
#pragma unroll
  for (int j = 0; j < KMAX; j++) {
    if (j < k) {
      const int64_t o = ((int64_t)b * k + j) * Q + q;
      idx[o] = bi[j];
      dist[o] = bi[j] > 0 ? sqrt_t(bd[j]) : T(0);
    }
  }
}

template <typename T, int KMAX>
int launch_knn(const T *ref, const T *query, int64_t *idx, T *dist, int64_t B, int64_t D,
               int64_t R, int64_t Q, int64_t k, hipStream_t s) {
  dim3 grid(div_up(Q, kThreads), (unsigned)B);
#define MCX_KNN_LAUNCH(DT)                                                                        \
  hipLaunchKernelGGL((knn_kernel<T, KMAX, DT>), grid, dim3(kThreads), 0, s, ref, query, idx,     \
                     dist, (int)D, (int)R, (int)Q, (int)k, (const char *)nullptr, (size_t)0)
  switch (D) {
    case 1: MCX_KNN_LAUNCH(1); break;
    case 2: MCX_KNN_LAUNCH(2); break;
    case 3: MCX_KNN_LAUNCH(3); break;
    case 4: MCX_KNN_LAUNCH(4); break;
    default: MCX_KNN_LAUNCH(0); break;
  }
#undef MCX_KNN_LAUNCH
  MCX_HIP_CHECK_LAUNCH();
  return 0;
}

template <typename T>
int knn_t(const void *ref, const void *query, int64_t *idx, void *dist, int64_t B, int64_t D,
          int64_t R, int64_t Q, int64_t k, hipStream_t s) {
  const T *r = (const T *)ref, *q = (const T *)query;
  T *d = (T *)dist;
  if (k <= 8) return launch_knn<T, 8>(r, q, idx, d, B, D, R, Q, k, s);
  if (k <= 16) return launch_knn<T, 16>(r, q, idx, d, B, D, R, Q, k, s);
  if (k <= 32) return launch_knn<T, 32>(r, q, idx, d, B, D, R, Q, k, s);
  return launch_knn<T, 64>(r, q, idx, d, B, D, R, Q, k, s);
}


// ---------------------------------------------------------------------------------
// Grid search for points of one to three dimensions: the same result, bit for bit, as the
// walk over all reference points above (same distance arithmetic, same order (distance,
// index) of the k kept), found among the reference points of the grid cells around the
// query only.  The reference points are binned into a uniform grid over their bounding box
// (count, prefix sum, fill); a query walks the cells around its own in rings of growing
// Chebyshev radius and stops once its k-th distance is safely below the distance to the
// nearest face of the cube of cells it has seen (every point not seen lies beyond a face).
// Points arrive in no particular order, so ties are resolved by the index explicitly.
// Reference points with a non-finite coordinate can never enter a result (their distance
// is not smaller than anything) and are left out of the grid.
// ---------------------------------------------------------------------------------
constexpr int kGridThreads = 1024;

#ifndef MCX_KNN_CELLS_PER_POINT
#define MCX_KNN_CELLS_PER_POINT 2.0
#endif
constexpr double kCellsPerPoint = MCX_KNN_CELLS_PER_POINT;
struct GridShape {
  int g[3];
  int64_t cells;
};
// Cells per dimension from the number of points alone (about two points per cell of a
// uniformly filled box; the host needs the workspace size before any data is seen).
inline GridShape grid_shape(int64_t D, int64_t R) {
  GridShape s{{1, 1, 1}, 1};
  const double per = std::pow((double)std::max<int64_t>(R, 1) * kCellsPerPoint, 1.0 / (double)D);
  const int cap = D == 1 ? 65536 : D == 2 ? 512 : 64;
  const int g = (int)std::min<double>(cap, std::max(1.0, std::ceil(per)));
  for (int d = 0; d < (int)D; d++) s.g[d] = g;
  s.cells = (int64_t)s.g[0] * s.g[1] * s.g[2];
  return s;
}
template <typename T>
size_t grid_slice_bytes(int64_t D, int64_t R) {
  const GridShape s = grid_shape(D, R);
  return align_up256(sizeof(GridHead<T>)) + align_up256((size_t)(s.cells + 1) * 4) +
         align_up256((size_t)s.cells * 4) + align_up256((size_t)R * sizeof(GridPoint<T>));
}

template <typename T>
__device__ inline bool finite_t(T v) { return v - v == T(0); }

template <typename T, int D>
__device__ inline int cell_of(const GridHead<T> &h, const int *g, const T *c, int *cd) {
  int cell = 0;
#pragma unroll
  for (int d = D - 1; d >= 0; d--) {
    const int i = min(max((int)floor((c[d] - h.lo[d]) * h.inv_h[d]), 0), g[d] - 1);
    cd[d] = i;
    cell = cell * g[d] + i;
  }
  return cell;
}

// Bounding box of a run of the finite reference points, and a run of the counters cleared.
// (One workgroup for all of them took 24 us at 40 962 points and 85 184 cells.)
template <typename T, int D>
__global__ __launch_bounds__(256) void knn_grid_box_kernel(const T *__restrict__ ref,
                                                           char *__restrict__ ws, size_t slice,
                                                           int R, int cells) {
  __shared__ T smin[D][4], smax[D][4];
  const int b = blockIdx.y, part = blockIdx.x;
  const T *rb = ref + (int64_t)b * D * R;
  char *base = ws + (size_t)b * slice;
  GridHead<T> *head = reinterpret_cast<GridHead<T> *>(base);
  int *start = reinterpret_cast<int *>(base + align_up256(sizeof(GridHead<T>)));
  int *cursor = reinterpret_cast<int *>(reinterpret_cast<char *>(start) +
                                        align_up256((size_t)(cells + 1) * 4));
  T mn[D], mx[D];
#pragma unroll
  for (int d = 0; d < D; d++) {
    mn[d] = inf_t<T>();
    mx[d] = -inf_t<T>();
  }
  for (int r = part * 256 + threadIdx.x; r < R; r += kBoxParts * 256) {
    T c[D];
    bool ok = true;
#pragma unroll
    for (int d = 0; d < D; d++) {
      c[d] = rb[(int64_t)d * R + r];
      ok = ok && finite_t(c[d]);
    }
    if (ok) {
#pragma unroll
      for (int d = 0; d < D; d++) {
        mn[d] = c[d] < mn[d] ? c[d] : mn[d];
        mx[d] = c[d] > mx[d] ? c[d] : mx[d];
      }
    }
  }
#pragma unroll
  for (int d = 0; d < D; d++) {
    for (int o = 32; o > 0; o >>= 1) {
      const T a = __shfl_xor(mn[d], o), c = __shfl_xor(mx[d], o);
      mn[d] = a < mn[d] ? a : mn[d];
      mx[d] = c > mx[d] ? c : mx[d];
    }
    if ((threadIdx.x & 63) == 0) {
      smin[d][threadIdx.x >> 6] = mn[d];
      smax[d][threadIdx.x >> 6] = mx[d];
    }
  }
  __syncthreads();
  if (threadIdx.x < D) {
    const int d = threadIdx.x;
    T lo = smin[d][0], hi = smax[d][0];
    for (int w = 1; w < 4; w++) {
      lo = smin[d][w] < lo ? smin[d][w] : lo;
      hi = smax[d][w] > hi ? smax[d][w] : hi;
    }
    head->part_lo[d][part] = lo;
    head->part_hi[d][part] = hi;
  }
  for (int c = part * 256 + threadIdx.x; c < cells; c += kBoxParts * 256) cursor[c] = 0;
}

// The grid from the parts of the bounding box, by one wave: valid in its every lane.
template <typename T, int D>
__device__ inline void grid_of_box(const GridHead<T> &parts, const int *g, int lane, T *glo, T *gh,
                                   T *ginv) {
#pragma unroll
  for (int d = 0; d < 3; d++) {
    T lo = T(0), hi = T(0);
    if (d < D) {
      lo = parts.part_lo[d][lane];
      hi = parts.part_hi[d][lane];
      for (int o = 32; o > 0; o >>= 1) {
        const T a = __shfl_xor(lo, o), c = __shfl_xor(hi, o);
        lo = a < lo ? a : lo;
        hi = c > hi ? c : hi;
      }
    }
    const T width = hi - lo;  // not finite: no finite point, or the box overflows
    const bool usable = d < D && width > T(0) && finite_t(width);
    glo[d] = usable ? lo : T(0);
    gh[d] = usable ? width / (T)g[d] : T(0);
    ginv[d] = usable ? (T)g[d] / width : T(0);  // unusable: everything in cell 0
  }
}

template <typename T, int D>
__global__ __launch_bounds__(256) void knn_grid_count_kernel(const T *__restrict__ ref,
                                                            char *__restrict__ ws, size_t slice,
                                                            int R, int g0, int g1, int g2,
                                                            int cells, int fill) {
  static_assert(kBoxParts == 64, "a lane takes a part");
  const int b = blockIdx.y;
  const int r = blockIdx.x * 256 + threadIdx.x;
  const T *rb = ref + (int64_t)b * D * R;
  char *base = ws + (size_t)b * slice;
  GridHead<T> *head = reinterpret_cast<GridHead<T> *>(base);
  int *start = reinterpret_cast<int *>(base + align_up256(sizeof(GridHead<T>)));
  int *cursor = reinterpret_cast<int *>(reinterpret_cast<char *>(start) +
                                        align_up256((size_t)(cells + 1) * 4));
  GridPoint<T> *pts = reinterpret_cast<GridPoint<T> *>(reinterpret_cast<char *>(cursor) +
                                                       align_up256((size_t)cells * 4));
  const int g[3] = {g0, g1, g2};
  // (every wave puts the box together for itself; the counting launch leaves the grid in the
  // head for the launches that follow it)
  GridHead<T> h;
  grid_of_box<T, D>(*head, g, threadIdx.x & 63, h.lo, h.h, h.inv_h);
  if (!fill && blockIdx.x == 0 && threadIdx.x == 0) {
    for (int d = 0; d < 3; d++) {
      head->lo[d] = h.lo[d];
      head->h[d] = h.h[d];
      head->inv_h[d] = h.inv_h[d];
    }
    head->skewed = 0;
  }
  if (r >= R) return;
  T c[3] = {T(0), T(0), T(0)};
  bool ok = true;
#pragma unroll
  for (int d = 0; d < D; d++) {
    c[d] = rb[(int64_t)d * R + r];
    ok = ok && finite_t(c[d]);
  }
  if (!ok) return;
  int cd[3];
  const int cell = cell_of<T, D>(h, g, c, cd);
  if (!fill) {
    atomicAdd(&cursor[cell], 1);
  } else {
    GridPoint<T> p;
    p.c[0] = c[0]; p.c[1] = c[1]; p.c[2] = c[2];
    p.idx = r + 1;
    // (first come, first placed: points of about ascending index, so that of many at one distance
    // the first k stay and the rest are turned away; the other way round each displaces one)
    pts[start[cell + 1] - atomicAdd(&cursor[cell], -1)] = p;
  }
}

// counts (in cursor) -> offsets (exclusive prefix sum; start[cells] = number of binned points);
// also decides whether the grid is worth walking.  A workgroup takes kScanCells cells and adds up
// every count before them by itself: 85 184 cells are at most 340 KB to read from L2, where one
// workgroup walking all of them paid a round trip to memory and two barriers per 4096 cells (25 us
// against 6).
constexpr int kScanCells = kGridThreads * 4;
template <typename T>
__global__ __launch_bounds__(kGridThreads) void knn_grid_scan_kernel(char *__restrict__ ws,
                                                                    size_t slice, int cells,
                                                                    int R) {
  constexpr int kWaves = kGridThreads / 64;
  __shared__ int before_sum[kWaves], wave_sum[kWaves], biggest[kWaves];
  char *base = ws + (size_t)blockIdx.y * slice;
  GridHead<T> *head = reinterpret_cast<GridHead<T> *>(base);
  int *start = reinterpret_cast<int *>(base + align_up256(sizeof(GridHead<T>)));
  const int *cursor = reinterpret_cast<int *>(reinterpret_cast<char *>(start) +
                                              align_up256((size_t)(cells + 1) * 4));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c0 = blockIdx.x * kScanCells;
  const int4 *count4 = reinterpret_cast<const int4 *>(cursor);  // (256-byte aligned)
  int sum = 0;
#pragma unroll 4
  for (int i = threadIdx.x; i < c0 / 4; i += kGridThreads) {
    const int4 v = count4[i];
    sum += v.x + v.y + v.z + v.w;
  }
  const int c = c0 + threadIdx.x * 4;
  int v[4];
#pragma unroll
  for (int j = 0; j < 4; j++) v[j] = c + j < cells ? cursor[c + j] : 0;
  int big = max(max(v[0], v[1]), max(v[2], v[3]));
  const int mine = v[0] + v[1] + v[2] + v[3];
  int incl = mine;  // inclusive scan within the wave
  for (int o = 1; o < 64; o <<= 1) {
    const int t = __shfl_up(incl, o);
    if (lane >= o) incl += t;
  }
  for (int o = 32; o > 0; o >>= 1) {
    sum += __shfl_xor(sum, o);
    big = max(big, __shfl_xor(big, o));
  }
  if (lane == 63) {
    wave_sum[wave] = incl;
    before_sum[wave] = sum;
    biggest[wave] = big;
  }
  __syncthreads();
  int run = incl - mine;
  for (int w = 0; w < kWaves; w++) {
    run += before_sum[w];
    if (w < wave) run += wave_sum[w];
  }
#pragma unroll
  for (int j = 0; j < 4; j++) {
    if (c + j < cells) start[c + j] = run;
    run += v[j];
    if (c + j == cells - 1) start[cells] = run;
  }
  if (threadIdx.x == 0) {
    int m = 0;
    for (int w = 0; w < kWaves; w++) m = max(m, biggest[w]);
    if (m > max(256, R / 4)) head->skewed = 1;  // (every writer stores the same value)
  }
}

template <typename T, int KMAX, int D>
__global__ __launch_bounds__(kThreads) void knn_grid_kernel(
    const T *__restrict__ query, int64_t *__restrict__ idx, T *__restrict__ dist,
    const char *__restrict__ ws, size_t slice, int Q, int k, int g0, int g1, int g2, int cells) {
  const int b = blockIdx.y;
  const char *base = ws + (size_t)b * slice;
  const GridHead<T> head = *reinterpret_cast<const GridHead<T> *>(base);
  if (head.skewed) return;
  const int *start = reinterpret_cast<const int *>(base + align_up256(sizeof(GridHead<T>)));
  const GridPoint<T> *pts = reinterpret_cast<const GridPoint<T> *>(
      reinterpret_cast<const char *>(start) + align_up256((size_t)(cells + 1) * 4) +
      align_up256((size_t)cells * 4));
  const int q = blockIdx.x * kThreads + threadIdx.x;
  if (q >= Q) return;
  const T *qb = query + (int64_t)b * D * Q;
  const int g[3] = {g0, g1, g2};

  T qv[3] = {T(0), T(0), T(0)};
  bool finite = true;
#pragma unroll
  for (int d = 0; d < D; d++) {
    qv[d] = qb[(int64_t)d * Q + q];
    finite = finite && finite_t(qv[d]);
  }
  T bd[KMAX];
  int bi[KMAX];
#pragma unroll
  for (int j = 0; j < KMAX; j++) {
    bd[j] = inf_t<T>();
    bi[j] = 0;
  }
  // (cd, ci) goes before (d, i): closer, or as close with the lower index; an empty slot
  // (infinite distance, index 0) yields to any finite distance only
  auto before = [](T cd, int ci, T d, int i) { return cd < d || (cd == d && ci < i); };
  auto insert = [&](T ssd, int pi) {
    if (before(ssd, pi, bd[KMAX - 1], bi[KMAX - 1])) {
      T cd = ssd;
      int ci = pi;
      bool shifting = false;
#pragma unroll
      for (int j = 0; j < KMAX; j++) {
        shifting = shifting || before(cd, ci, bd[j], bi[j]);
        if (shifting) {
          const T td = bd[j];
          const int ti = bi[j];
          bd[j] = cd;
          bi[j] = ci;
          cd = td;
          ci = ti;
        }
      }
    }
  };
  // The points of cells cell_a .. cell_b, four at a time so that their loads are in flight
  // together (a load past the run re-reads its last point and is not used).
  constexpr int kUnroll = 4;
  auto scan = [&](int cell_a, int cell_b) {
    const int e = start[cell_b + 1];
    for (int r = start[cell_a]; r < e; r += kUnroll) {
      GridPoint<T> p[kUnroll];
#pragma unroll
      for (int u = 0; u < kUnroll; u++) p[u] = pts[min(r + u, e - 1)];
      T ssd[kUnroll];
#pragma unroll
      for (int u = 0; u < kUnroll; u++) {
        ssd[u] = T(0);
#pragma unroll
        for (int d = 0; d < D; d++) {
          const T t = p[u].c[d] - qv[d];
          ssd[u] = fma_t(t, t, ssd[u]);
        }
      }
#pragma unroll
      for (int u = 0; u < kUnroll; u++)
        if (r + u < e) insert(ssd[u], p[u].idx);
    }
  };

  if (finite && start[cells] > 0) {  // a query with a non-finite coordinate is near nothing
    int c[3] = {0, 0, 0};
    cell_of<T, D>(head, g, qv, c);
    // a dimension the points do not spread over (cell size 0) has them all in its cell 0
    int ge[3] = {1, 1, 1};
    T hmin = inf_t<T>();
    // largest coordinate magnitude of a cell face: the face lo + n * h is rounded to one unit in
    // the last place of that magnitude, and the cell index floor((c - lo) / h) of a point next to
    // face n is off by a few units in the last place of n, i.e. of (n * h) in coordinates
    T reach = T(0);
#pragma unroll
    for (int d = 0; d < D; d++) {
      if (head.h[d] > T(0)) {
        ge[d] = g[d];
        hmin = head.h[d] < hmin ? head.h[d] : hmin;
        const T lo = head.lo[d] < T(0) ? -head.lo[d] : head.lo[d];
        const T span = (T)g[d] * head.h[d];
        reach = lo + span > reach ? lo + span : reach;
      }
    }
    const int gmax = max(ge[0], max(ge[1], ge[2]));
    constexpr T kUlp = sizeof(T) == 4 ? T(1.1920929e-7) : T(2.220446049250313e-16);
    // a thousandth of a cell, plus the rounding above (which outgrows it on long one-dimensional
    // grids: 65536 cells in fp32 put a face off by hundredths of a cell)
    const T slack = hmin * T(1e-3) + T(16) * kUlp * reach;
    for (int rho = 0; rho < gmax; rho++) {
      // ring rho: rows of cells along the first dimension; rows on the ring's outer faces
      // are contiguous runs of cells (one run of points), the others contribute their ends
      const int z0 = max(c[2] - rho, 0), z1 = min(c[2] + rho, ge[2] - 1);
      const int y0 = max(c[1] - rho, 0), y1 = min(c[1] + rho, ge[1] - 1);
      const int xa = c[0] - rho, xb = c[0] + rho;
      for (int z = z0; z <= z1; z++) {
        for (int y = y0; y <= y1; y++) {
          const int row = (z * g1 + y) * g0;
          const bool face = (D > 2 && (z == c[2] - rho || z == c[2] + rho)) ||
                            (D > 1 && (y == c[1] - rho || y == c[1] + rho));
          if (face || rho == 0) {
            scan(row + max(xa, 0), row + min(xb, ge[0] - 1));
          } else {
            if (xa >= 0) scan(row + xa, row + xa);
            if (xb < ge[0]) scan(row + xb, row + xb);
          }
        }
      }
      // every point not seen lies beyond a face of the cube of cells seen that is not on the
      // grid's boundary; m: distance from the query to the nearest such face
      T m = inf_t<T>();
#pragma unroll
      for (int d = 0; d < D; d++) {
        if (c[d] - rho > 0) {
          const T f = head.lo[d] + (T)(c[d] - rho) * head.h[d];
          m = qv[d] - f < m ? qv[d] - f : m;
        }
        if (c[d] + rho < ge[d] - 1) {
          const T f = head.lo[d] + (T)(c[d] + rho + 1) * head.h[d];
          m = f - qv[d] < m ? f - qv[d] : m;
        }
      }
      if (!(m < inf_t<T>())) break;  // the whole grid has been seen
      T kth = bd[0];
#pragma unroll
      for (int j = 1; j < KMAX; j++) kth = j < k ? bd[j] : kth;
      // (the margins cover the rounding of cell assignment, faces and distances)
      const T safe = m - slack;
      if (safe > T(0) && kth < safe * safe * T(1.0 - 1e-5)) break;
    }
  }
#pragma unroll
  for (int j = 0; j < KMAX; j++) {
    if (j < k) {
      const int64_t o = ((int64_t)b * k + j) * Q + q;
      idx[o] = bi[j];
      dist[o] = bi[j] > 0 ? sqrt_t(bd[j]) : T(0);
    }
  }
}

// The k best so far of a lane in fp32, ordered by (distance, index); an empty slot (infinite
// distance, index 0) yields to any finite distance only.
// The pair is one 64-bit key, distance above index, read as a double: the bits of
// numbers that are not negative are ordered like the numbers, and no key is an infinity or NaN (a
// finite or infinite fp32 distance in the upper word is a finite double; a distance of zero makes
// a subnormal one, which the 64-bit unit keeps).  Entry j after an insertion of x is then
// max(entry j - 1, min(entry j, x)): two instructions an entry, where the comparisons and moves
// of a pair are about eight.
template <int KMAX>
struct TopK {
  double key[KMAX];
  __device__ static inline double key_of(float d, int i) {
    return __builtin_bit_cast(double, ((uint64_t)__builtin_bit_cast(unsigned, d) << 32) |
                                          (unsigned)i);
  }
  // (written out: the compiler would quiet every operand first, for fear of a signalling NaN)
  __device__ static inline double min2(double a, double b) {
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
  }
  __device__ static inline double max2(double a, double b) {
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
  }
  __device__ inline void init() {
#pragma unroll
    for (int j = 0; j < KMAX; j++) key[j] = key_of(inf_t<float>(), 0);
  }
  __device__ inline void insert(float ssd, int pi) {
    const double x = key_of(ssd, pi);
    if (!(x < key[KMAX - 1])) return;
#pragma unroll
    for (int j = KMAX - 1; j > 0; j--) key[j] = max2(key[j - 1], min2(key[j], x));
    key[0] = min2(key[0], x);
  }
  __device__ inline float dist(int j) const {
    return __builtin_bit_cast(float, (unsigned)(__builtin_bit_cast(uint64_t, key[j]) >> 32));
  }
  __device__ inline int index(int j) const { return (int)__builtin_bit_cast(uint64_t, key[j]); }
};

// Bound: vector instructions under divergence (a lane whose cells hold fewer points waits for the
// wave's fullest).  So the runs of points of a lane's cells go into a list in LDS first and each
// lane walks its own list through: the wave pays for the largest sum over its lanes, not for the
// sum of each row's largest, and the loads of the row bounds are in flight together.
// Rings beyond the first hold few points a lane still needs; rows that its k-th distance rules
// out are not listed.
// Measured, the kernel above -> this one (whole calls, us; Q queries among R points, k):
// sphere, 524 288 among 40 962, 8: 318 -> 151; 1 000 among 642, 1: 76 -> 30; cube, 262 144
// among 40 962, 8: 251 -> 136; plane 150 -> 84; line 122 -> 76; sphere, 50 000 among 10 000, 33:
// 2388 -> 189; 40 tight clusters, 100 000 among 40 962, 8: 1126 -> 381.  (All but the first pair
// hold the binning's own gain too, some 35 us among 40 962 points.)  In fp64 the key does not fit an instruction's operand and the same walk, with
// pairs, needs more registers than there are: 2.7 -> 9.8 ms at k = 33, 410 -> 496 us for the cube
// at k = 16 (and 265 -> 195 for the sphere at 8); fp64 keeps the kernel above.
constexpr int kCrowded = 256;  // points in a query's 27 cells
constexpr int kRuns = 12;  // runs listed per lane (24 KB of LDS: six workgroups a CU)
template <int KMAX, int D>
__global__ __launch_bounds__(kThreads) void knn_grid_lists_kernel(
    const float *__restrict__ query, int64_t *__restrict__ idx, float *__restrict__ dist,
    const char *__restrict__ ws, size_t slice, int Q, int k, int g0, int g1, int g2, int cells) {
  using T = float;
  const int b = blockIdx.y;
  const char *base = ws + (size_t)b * slice;
  const GridHead<T> head = *reinterpret_cast<const GridHead<T> *>(base);
  if (head.skewed) return;
  const int *start = reinterpret_cast<const int *>(base + align_up256(sizeof(GridHead<T>)));
  const GridPoint<T> *pts = reinterpret_cast<const GridPoint<T> *>(
      reinterpret_cast<const char *>(start) + align_up256((size_t)(cells + 1) * 4) +
      align_up256((size_t)cells * 4));
  const int q = blockIdx.x * kThreads + threadIdx.x;
  if (q >= Q) return;
  const T *qb = query + (int64_t)b * D * Q;
  const int g[3] = {g0, g1, g2};

  T qv[3] = {T(0), T(0), T(0)};
  bool finite = true;
#pragma unroll
  for (int d = 0; d < D; d++) {
    qv[d] = qb[(int64_t)d * Q + q];
    finite = finite && finite_t(qv[d]);
  }
  TopK<KMAX> best;
  best.init();
  __shared__ int2 runs[kRuns][kThreads];  // (a lane reads only what it wrote: no barrier)
  int listed = 0;
  auto kth_dist = [&]() __attribute__((always_inline)) {
    // (the largest of the first k.  They are in order; but written as the choice of entry k - 1,
    // it is compiled to an access at a variable index, and the list then lives in scratch memory)
    T kth = best.dist(0);
#pragma unroll
    for (int j = 1; j < KMAX; j++) {
      const T d = best.dist(j);
      kth = j < k && d > kth ? d : kth;
    }
    return kth;
  };
  // On a line, between points far apart, thousands of rings hold nothing: there the k-th distance
  // is kept from the last walk that found something (40 962 points in 20 tight clusters, 200 000
  // queries, k = 8: 8640 -> 5450 us; with more dimensions its register costs more than it saves).
  T kept = inf_t<T>();
  auto kth_so_far = [&]() __attribute__((always_inline)) { return D == 1 ? kept : kth_dist(); };
  // The points of the listed runs, four at a time so that their loads are in flight together
  // (a load past the run re-reads its last point and is not used).
  constexpr int kUnroll = 4;
  auto walk = [&]() __attribute__((always_inline)) {
    if (D == 1 && listed == 0) return;
    int next = 0, r = 0, e = 0;
    for (;;) {
      if (r >= e) {
        if (next == listed) break;
        const int2 run = runs[next++][threadIdx.x];
        r = run.x;
        e = run.y;
      }
      GridPoint<T> p[kUnroll];
#pragma unroll
      for (int u = 0; u < kUnroll; u++) p[u] = pts[min(r + u, e - 1)];
      T ssd[kUnroll];
#pragma unroll
      for (int u = 0; u < kUnroll; u++) {
        ssd[u] = T(0);
#pragma unroll
        for (int d = 0; d < D; d++) {
          const T t = p[u].c[d] - qv[d];
          ssd[u] = fma_t(t, t, ssd[u]);
        }
      }
#pragma unroll
      for (int u = 0; u < kUnroll; u++)
        if (r + u < e) best.insert(ssd[u], p[u].idx);
      r += kUnroll;
    }
    listed = 0;
    if (D == 1) kept = kth_dist();
  };
  auto list = [&](int r, int e) __attribute__((always_inline)) {
    if (r < e) runs[listed++][threadIdx.x] = make_int2(r, e);
  };

  if (finite && start[cells] > 0) {  // a query with a non-finite coordinate is near nothing
    int c[3] = {0, 0, 0};
    const int cell = cell_of<T, D>(head, g, qv, c);
    // a dimension the points do not spread over (cell size 0) has them all in its cell 0
    int ge[3] = {1, 1, 1};
    T hmin = inf_t<T>();
    // largest coordinate magnitude of a cell face: the face lo + n * h is rounded to one unit in
    // the last place of that magnitude, and the cell index floor((c - lo) / h) of a point next to
    // face n is off by a few units in the last place of n, i.e. of (n * h) in coordinates
    T reach = T(0);
#pragma unroll
    for (int d = 0; d < D; d++) {
      if (head.h[d] > T(0)) {
        ge[d] = g[d];
        hmin = head.h[d] < hmin ? head.h[d] : hmin;
        const T lo = head.lo[d] < T(0) ? -head.lo[d] : head.lo[d];
        const T span = (T)g[d] * head.h[d];
        reach = lo + span > reach ? lo + span : reach;
      }
    }
    const int gmax = max(ge[0], max(ge[1], ge[2]));
    constexpr T kUlp = 1.1920929e-7f;
    // a thousandth of a cell, plus the rounding above (which outgrows it on long one-dimensional
    // grids: 65536 cells in fp32 put a face off by hundredths of a cell)
    const T slack = hmin * T(1e-3) + T(16) * kUlp * reach;
    // a lower bound on the distance to the points of cells n along dimension d, squared
    auto gap2 = [&](int d, int n) {
      T f = T(0);
      if (n > c[d]) f = head.lo[d] + (T)n * head.h[d] - qv[d];
      if (n < c[d]) f = qv[d] - (head.lo[d] + (T)(n + 1) * head.h[d]);
      f -= slack;
      return f > T(0) ? f * f : T(0);
    };
    // the query's cell and its neighbours at once: a wave whose 64 lanes all find their k in the
    // one cell is rare, and each row of cells is one run of points.  Where the points crowd (some
    // 60 on a sphere, 14 in a cube filled evenly) the one cell comes first, so that its k-th
    // distance rules the neighbours out.
    bool crowded;
    {
      const int x0 = max(c[0] - 1, 0), x1 = min(c[0] + 1, ge[0] - 1) + 1;
      int ra[9], re[9];
#pragma unroll
      for (int i = 0; i < 9; i++) {
        const int z = c[2] + i / 3 - 1, y = c[1] + i % 3 - 1;
        ra[i] = re[i] = 0;
        if (z >= 0 && z < ge[2] && y >= 0 && y < ge[1]) {
          const int row = (z * g1 + y) * g0;
          ra[i] = start[row + x0];
          re[i] = start[row + x1];
        }
      }
      int held = 0;
#pragma unroll
      for (int i = 0; i < 9; i++) held += re[i] - ra[i];
      crowded = held > kCrowded;
      if (crowded) {
        list(start[cell], start[cell + 1]);
      } else {
#pragma unroll
        for (int i = 0; i < 9; i++) list(ra[i], re[i]);
      }
    }
    bool first = true;
    for (int rho = crowded ? 0 : 1; rho < max(gmax, 2); rho++) {
      const int z0 = max(c[2] - rho, 0), z1 = min(c[2] + rho, ge[2] - 1);
      const int y0 = max(c[1] - rho, 0), y1 = min(c[1] + rho, ge[1] - 1);
      const int xa = c[0] - rho, xb = c[0] + rho;
      int z = first ? z1 + 1 : z0, y = y0;  // the next row of the ring
      first = false;
      do {
        // ring rho: rows of cells along the first dimension; rows on the ring's outer faces
        // are contiguous runs of cells (one run of points), the others contribute their ends.
        // A row that lies beyond the k-th distance holds none of the k (the margin is that of
        // the test below).
        const T kth = kth_so_far();
        while (z <= z1 && listed <= kRuns - 2) {
          const T gyz = (D > 2 ? gap2(2, z) : T(0)) + (D > 1 ? gap2(1, y) : T(0));
          if (!(kth < gyz * T(1.0 - 1e-5))) {
            const int row = (z * g1 + y) * g0;
            const bool face = (D > 2 && (z == c[2] - rho || z == c[2] + rho)) ||
                              (D > 1 && (y == c[1] - rho || y == c[1] + rho));
            if (face) {
              list(start[row + max(xa, 0)], start[row + min(xb, ge[0] - 1) + 1]);
            } else {
              if (xa >= 0 && !(kth < (gyz + gap2(0, xa)) * T(1.0 - 1e-5)))
                list(start[row + xa], start[row + xa + 1]);
              if (xb < ge[0] && !(kth < (gyz + gap2(0, xb)) * T(1.0 - 1e-5)))
                list(start[row + xb], start[row + xb + 1]);
            }
          }
          if (++y > y1) {
            y = y0;
            z++;
          }
        }
        walk();
      } while (z <= z1);
      // every point not seen lies beyond a face of the cube of cells seen that is not on the
      // grid's boundary; m: distance from the query to the nearest such face
      T m = inf_t<T>();
#pragma unroll
      for (int d = 0; d < D; d++) {
        if (c[d] - rho > 0) {
          const T f = head.lo[d] + (T)(c[d] - rho) * head.h[d];
          m = qv[d] - f < m ? qv[d] - f : m;
        }
        if (c[d] + rho < ge[d] - 1) {
          const T f = head.lo[d] + (T)(c[d] + rho + 1) * head.h[d];
          m = f - qv[d] < m ? f - qv[d] : m;
        }
      }
      if (!(m < inf_t<T>())) break;  // the whole grid has been seen
      const T kth = kth_so_far();
      // (the margins cover the rounding of cell assignment, faces and distances)
      const T safe = m - slack;
      if (safe > T(0) && kth < safe * safe * T(1.0 - 1e-5)) break;
    }
  }
#pragma unroll
  for (int j = 0; j < KMAX; j++) {
    if (j < k) {
      const int64_t o = ((int64_t)b * k + j) * Q + q;
      idx[o] = best.index(j);
      dist[o] = best.index(j) > 0 ? sqrt_t(best.dist(j)) : T(0);
    }
  }
}

template <typename T, int KMAX, int D>
int launch_knn_grid(const T *ref, const T *query, int64_t *idx, T *dist, void *workspace,
                    int64_t B, int64_t R, int64_t Q, int64_t k, hipStream_t s) {
  const GridShape gs = grid_shape(D, R);
  const size_t slice = grid_slice_bytes<T>(D, R);
  char *ws = (char *)workspace;
  const int cells = (int)gs.cells;
  hipLaunchKernelGGL((knn_grid_box_kernel<T, D>), dim3(kBoxParts, (unsigned)B), dim3(256), 0, s,
                     ref, ws, slice, (int)R, cells);
  MCX_HIP_CHECK_LAUNCH();
  const dim3 rgrid(div_up(R, 256), (unsigned)B);
  hipLaunchKernelGGL((knn_grid_count_kernel<T, D>), rgrid, dim3(256), 0, s, ref, ws, slice, (int)R,
                     gs.g[0], gs.g[1], gs.g[2], cells, 0);
  MCX_HIP_CHECK_LAUNCH();
  hipLaunchKernelGGL(knn_grid_scan_kernel<T>, dim3(div_up(cells, kScanCells), (unsigned)B),
                     dim3(kGridThreads), 0, s, ws, slice, cells, (int)R);
  MCX_HIP_CHECK_LAUNCH();
  hipLaunchKernelGGL((knn_grid_count_kernel<T, D>), rgrid, dim3(256), 0, s, ref, ws, slice, (int)R,
                     gs.g[0], gs.g[1], gs.g[2], cells, 1);
  MCX_HIP_CHECK_LAUNCH();
  const dim3 qgrid(div_up(Q, kThreads), (unsigned)B);
  if constexpr (sizeof(T) == 4)
    hipLaunchKernelGGL((knn_grid_lists_kernel<KMAX, D>), qgrid, dim3(kThreads), 0, s, query, idx,
                       dist, ws, slice, (int)Q, (int)k, gs.g[0], gs.g[1], gs.g[2], cells);
  else
    hipLaunchKernelGGL((knn_grid_kernel<T, KMAX, D>), qgrid, dim3(kThreads), 0, s, query, idx,
                       dist, ws, slice, (int)Q, (int)k, gs.g[0], gs.g[1], gs.g[2], cells);
  MCX_HIP_CHECK_LAUNCH();
  // the plain walk, for batch elements whose grid came out skewed (it returns at once otherwise)
  hipLaunchKernelGGL((knn_kernel<T, KMAX, D>), qgrid, dim3(kThreads), 0, s, ref, query, idx, dist,
                     (int)D, (int)R, (int)Q, (int)k, (const char *)ws, slice);
  MCX_HIP_CHECK_LAUNCH();
  return 0;
}

// The grid pays once there are enough reference points to skip.
inline bool grid_applies(int64_t D, int64_t R) { return D >= 1 && D <= 3 && R >= 512; }

template <typename T>
int knn_grid_t(const void *ref, const void *query, int64_t *idx, void *dist, void *workspace,
               int64_t B, int64_t D, int64_t R, int64_t Q, int64_t k, hipStream_t s) {
  const T *r = (const T *)ref, *q = (const T *)query;
  T *d = (T *)dist;
#define MCX_KNN_GRID(KMAX)                                                                  \
  switch (D) {                                                                              \
    case 1: return launch_knn_grid<T, KMAX, 1>(r, q, idx, d, workspace, B, R, Q, k, s);     \
    case 2: return launch_knn_grid<T, KMAX, 2>(r, q, idx, d, workspace, B, R, Q, k, s);     \
    default: return launch_knn_grid<T, KMAX, 3>(r, q, idx, d, workspace, B, R, Q, k, s);    \
  }
  if (k <= 8) { MCX_KNN_GRID(8) }
  if (k <= 16) { MCX_KNN_GRID(16) }
  if (k <= 32) { MCX_KNN_GRID(32) }
  MCX_KNN_GRID(64)
#undef MCX_KNN_GRID
}

}  // namespace
}  // namespace mcx

extern "C" size_t mcx_knn_workspace(int64_t B, int64_t D, int64_t R, int dtype) {
  if (B <= 0 || R <= 0 || !mcx::grid_applies(D, R)) return 0;
  if (dtype == MCX_F32) return (size_t)B * mcx::grid_slice_bytes<float>(D, R);
  if (dtype == MCX_F64) return (size_t)B * mcx::grid_slice_bytes<double>(D, R);
  return 0;
}

extern "C" int mcx_knn(const void *ref, const void *query, int64_t *idx, void *dist,
                       void *workspace, size_t workspace_bytes, int64_t B, int64_t D, int64_t R,
                       int64_t Q, int64_t k, int dtype, void *stream) {
  if (!ref || !query || !idx || !dist) return MCX_E_NULL;
  for (int64_t v : {B, D, R, Q, k, D * R, D * Q})
    if (v <= 0 || v > 0x7fffffffLL) return MCX_E_SHAPE;
  if (k > 64 || B > 65535) return MCX_E_SHAPE;
  if (dtype != MCX_F32 && dtype != MCX_F64) return MCX_E_DTYPE;
  hipStream_t s = (hipStream_t)stream;
  const size_t need = mcx_knn_workspace(B, D, R, dtype);
  if (workspace && need > 0) {
    if (workspace_bytes < need) return MCX_E_WORKSPACE;
    if (dtype == MCX_F32)
      return mcx::knn_grid_t<float>(ref, query, idx, dist, workspace, B, D, R, Q, k, s);
    return mcx::knn_grid_t<double>(ref, query, idx, dist, workspace, B, D, R, Q, k, s);
  }
  if (dtype == MCX_F32) return mcx::knn_t<float>(ref, query, idx, dist, B, D, R, Q, k, s);
  return mcx::knn_t<double>(ref, query, idx, dist, B, D, R, Q, k, s);
}
