// fp64 form of the three products (gather-product, product-scatter, weight gradient; roles in
// mcx_conv_generic.hip) over channel-last records.  In the planar layout every corner of every
// tap of every channel is an 8-byte access in a cache line of its own; a record holds all
// channels of a pixel side by side, so a corner is one run of lines that LPR neighbouring
// lanes read (or add to) together.  The operand that the map reaches is copied into records
// in the caller's workspace (the scattered destination: accumulated there and copied back);
// without a workspace the scalar kernels run.  All arithmetic is fp64 on the vector units: the
// fp64 matrix instructions have the same rate here.
// Bound: random record reads and fp64 atomics.  Measured at one image of 200x500 pixels, 10 -> 1
// channels, nine taps of a shuffled map (scalar kernels -> these): forward
// 210 -> 36 us (7 of them the copy), input gradient 1585 -> 375 us (the atomics: 36 M of them
// as 3.6 M records; 2 x 8 lanes per record of 10 channels 385), weight gradient 579 -> 70 us.
// Where a map is coherent the scalar kernels can be the faster ones: see "where the map decides"
// and "where records pay" below.
#include <algorithm>

#include "mcx_conv.h"
#include "mcx_device.h"

namespace mcx {
namespace {

constexpr int kThreads = 256;

// Lanes per record.  A reading lane handles two channels, so a pass covers 2 * LPR; a lane that
// adds handles one.
template <int LPR>
struct RecShape {
  static constexpr int kLocs = kThreads / LPR;  // map locations per workgroup
  static constexpr int kCh = 2 * LPR;           // channels per pass
  // taps resolved per pass (their cache is what limits the workgroups per CU)
  static constexpr int kTaps = LPR == 2 ? 5 : 9;
};

// Record stride in doubles: 16-byte pairs for reading.
inline int64_t read_stride(int64_t channels) { return (channels + 1) & ~(int64_t)1; }
// Records that atomics add to.  Requests are of 64 bytes: up to eight channels a power of two and
// from 17 on a multiple of eight, so that no run of eight straddles a boundary (five channels
// without a pad, shuffled map of 256x512: 224 -> 330 us).  Nine to sixteen lie side by side:
// neighbouring records then share requests, and where they do not it costs nothing (ten channels
// padded to sixteen, coherent 502 -> 341 us, shuffled 450 -> 445).
inline int64_t add_stride(int64_t channels) {
  for (int64_t s = 2; s <= 8; s *= 2)
    if (channels <= s) return s;
  return channels <= 16 ? (channels + 1) & ~(int64_t)1 : (channels + 7) & ~(int64_t)7;
}
inline int lanes_per_record(int64_t channels) { return channels <= 4 ? 2 : channels <= 8 ? 4 : 8; }

// *coherent = 1 if in three of four samples of the map (up to 1024 taps) the next location's tap
// points at the pixel beside, else 0: what decides between planes and records where neither form
// is better for every map.  Block 0; the others clear `count` pairs of doubles, it helps.
__global__ __launch_bounds__(kThreads) void begin_records_kernel(const double *__restrict__ map,
                                                                 int64_t N, int K, int pm,
                                                                 int nearest,
                                                                 int *__restrict__ coherent,
                                                                 double2 *__restrict__ clear,
                                                                 int64_t count) {
  if (coherent && blockIdx.x == 0) {
    constexpr int kSamples = 4 * kThreads;
    int beside = 0;
    for (int i = threadIdx.x; i < kSamples; i += kThreads) {
      // (spread by the golden ratio, not by a stride that could meet a row's end every time;
      // N > 1 where the map is asked, n <= N - 2)
      const uint64_t u = (uint32_t)i * 2654435769u;
      const int64_t n = (int64_t)((u * (uint64_t)(N - 1)) >> 32);
      const int64_t e = (n * K + i % K) * pm, e2 = e + (int64_t)K * pm;
      double x = map[e * 2], y = map[e * 2 + 1], x2 = map[e2 * 2], y2 = map[e2 * 2 + 1];
      if (nearest) {
        x = round_half_away(x), y = round_half_away(y);
        x2 = round_half_away(x2), y2 = round_half_away(y2);
      } else {
        x = mcx_floor(x), y = mcx_floor(y), x2 = mcx_floor(x2), y2 = mcx_floor(y2);
      }
      const double d = x2 - x;
      beside += __syncthreads_count(y == y2 && (d == 1.0 || d == -1.0));
    }
    if (threadIdx.x == 0) *coherent = beside * 4 >= kSamples * 3 ? 1 : 0;
  }
  const int64_t stride = (int64_t)gridDim.x * kThreads;
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < count; i += stride)
    clear[i] = make_double2(0.0, 0.0);
}

// `unless` below: a word that ends the kernel at once where it is not zero (NULL: always runs).

// [B][C][N] -> records [B][N + 1][stride]; the last record of an image is all zeros (what a
// corner outside the image reads), as are the channels beyond C.
__global__ __launch_bounds__(kThreads) void to_records_kernel(const double *__restrict__ x,
                                                              double *__restrict__ rec, int C,
                                                              int stride, int64_t N,
                                                              const int *__restrict__ unless) {
  if (unless && *unless != 0) return;
  const int64_t n = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  const int b = blockIdx.z;
  if (n > N) return;
  const double *src = x + (int64_t)b * C * N + (n < N ? n : 0);
  double2 *dst = reinterpret_cast<double2 *>(rec + ((int64_t)b * (N + 1) + n) * stride);
  const int c_end = min(stride, (int)(blockIdx.y + 1) * 16);
  for (int c = blockIdx.y * 16; c < c_end; c += 2) {
    double2 v = make_double2(0.0, 0.0);
    if (n < N) {
      if (c < C) v.x = src[(int64_t)c * N];
      if (c + 1 < C) v.y = src[(int64_t)(c + 1) * N];
    }
    dst[c >> 1] = v;
  }
}

// records [B][N][stride] -> [B][C][N], plus bias; the bias alone where `bias_only` says so
__global__ __launch_bounds__(kThreads) void from_records_kernel(const double *__restrict__ rec,
                                                                const double *__restrict__ bias,
                                                                double *__restrict__ y, int C,
                                                                int stride, int64_t N,
                                                                const int *__restrict__ bias_only) {
  const int64_t n = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  const int b = blockIdx.z;
  if (n >= N) return;
  const double2 *src = reinterpret_cast<const double2 *>(rec + ((int64_t)b * N + n) * stride);
  double *dst = y + (int64_t)b * C * N + n;
  const bool skip = bias_only && *bias_only != 0;
  const int c_end = min(C, (int)(blockIdx.y + 1) * 16);
  for (int c = blockIdx.y * 16; c < c_end; c += 2) {
    const double2 v = skip ? make_double2(0.0, 0.0) : src[c >> 1];
    dst[(int64_t)c * N] = v.x + (bias ? bias[c] : 0.0);
    if (c + 1 < C) dst[(int64_t)(c + 1) * N] = v.y + (bias ? bias[c + 1] : 0.0);
  }
}

// Tap (n, k) of interpolation point p as NC (record index, weight) pairs; a corner outside the
// image, or of weight zero, gets the index `none`.
template <int NC>
__device__ inline void resolve_records(const double *__restrict__ map,
                                       const double *__restrict__ iw, int64_t e, int h, int w,
                                       bool wrap, int none, int *off, double *wt, int step) {
  const double x = map[e * 2], y = map[e * 2 + 1];
  const double scale = iw ? iw[e] : 1.0;
  if constexpr (NC == 1) {
    Tap<double, kInterpNearest> t;
    t.set(x, y, h, w);
    off[0] = t.off < 0 ? none : t.off;
    wt[0] = scale;
  } else {
    // (beside a corner that counts, one that does not weighs zero whatever the tap's scale: an
    // infinite one times the zero it reads would make the whole sample NaN)
    auto put = [&](const auto &t) {
      bool any = false;
#pragma unroll
      for (int i = 0; i < 4; i++) any |= t.off[i] >= 0;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        off[i * step] = t.off[i] < 0 ? none : t.off[i];
        wt[i * step] = t.wt[i] * (any && t.off[i] < 0 ? 0.0 : scale);
      }
    };
    if (wrap) {
      Tap<double, kInterpBispherical> t;
      t.set(x, y, h, w);
      put(t);
    } else {
      Tap<double, kInterpBilinear> t;
      t.set(x, y, h, w);
      put(t);
    }
  }
}

// The taps [k0, k0 + taps) of a workgroup's locations into its cache, [corner][tap][location].
template <int NC, int LPR, int TAPS = RecShape<LPR>::kTaps>
__device__ inline void fill_tap_cache(const double *__restrict__ map,
                                      const double *__restrict__ iw, int n0, int N, int K, int pm,
                                      int p, int k0, int taps, int h, int w, bool wrap, int none,
                                      int *s_off, double *s_wt) {
  using S = RecShape<LPR>;
  constexpr int kStep = TAPS * S::kLocs;
  for (int e = threadIdx.x; e < taps * S::kLocs; e += kThreads) {
    const int l = e / taps, t = e - l * taps;
    const int slot = t * S::kLocs + l;
    if (n0 + l < N) {
      resolve_records<NC>(map, iw, ((int64_t)(n0 + l) * K + k0 + t) * pm + p, h, w, wrap, none,
                          s_off + slot, s_wt + slot, kStep);
    } else {
#pragma unroll
      for (int i = 0; i < NC; i++) {
        s_off[i * kStep + slot] = none;
        s_wt[i * kStep + slot] = 0.0;
      }
    }
  }
}

// y[b,o,n] = bias[o] + sum_{g,k} W[o,g,k] * sample(src[b,g], map[n,k]).  A location belongs to
// LPR lanes; every lane sums its two channels into OT outputs, the lanes' sums are added at
// the end.  Taps and the weights of a pass sit in LDS.
template <int NC, int LPR, int OT>
__global__ __launch_bounds__(kThreads) void gather_records_kernel(
    const double *__restrict__ rec, const double *__restrict__ map, const double *__restrict__ iw,
    const double *__restrict__ w, const double *__restrict__ bias, double *__restrict__ y, int G,
    int stride, int O, int SH, int SW, int N, int K, int P, int wrap,
    const int *__restrict__ unless) {
  if (unless && *unless != 0) return;
  using S = RecShape<LPR>;
  constexpr int kStep = S::kTaps * S::kLocs;
  __shared__ int s_off[NC * kStep];
  __shared__ double s_wt[NC * kStep];
  __shared__ double2 s_w[S::kTaps * OT * LPR];
  const int loc = threadIdx.x / LPR, j = threadIdx.x % LPR;
  const int n0 = blockIdx.x * S::kLocs, o0 = blockIdx.y * OT, b = blockIdx.z;
  const int64_t SN = (int64_t)SH * SW;
  const double *recb = rec + (int64_t)b * (SN + 1) * stride;
  const int pm = P == 0 ? 1 : P;
  double acc[OT];
#pragma unroll
  for (int o = 0; o < OT; o++) acc[o] = 0.0;
  for (int k0 = 0; k0 < K; k0 += S::kTaps) {
    const int taps = min(S::kTaps, K - k0);
    for (int g0 = 0; g0 < stride; g0 += S::kCh) {
      __syncthreads();
      for (int i = threadIdx.x; i < taps * OT * LPR; i += kThreads) {
        const int jj = i % LPR, o = i / LPR % OT, t = i / (LPR * OT);
        const int g = g0 + 2 * jj;
        double2 v = make_double2(0.0, 0.0);
        if (o0 + o < O) {
          const double *row = w + ((int64_t)(o0 + o) * G + g) * K + k0 + t;
          if (g < G) v.x = row[0];
          if (g + 1 < G) v.y = row[K];
        }
        s_w[i] = v;
      }
      for (int p = 0; p < pm; p++) {
        if (p) __syncthreads();
        fill_tap_cache<NC, LPR>(map, iw, n0, N, K, pm, p, k0, taps, SH, SW, wrap != 0, (int)SN,
                                s_off, s_wt);
        __syncthreads();
        if (g0 + 2 * j < stride) {
          const double *src = recb + g0 + 2 * j;
#pragma unroll 3
          for (int t = 0; t < taps; t++) {
            double2 d[NC];
#pragma unroll
            for (int i = 0; i < NC; i++)
              d[i] = *reinterpret_cast<const double2 *>(
                  src + (int64_t)s_off[i * kStep + t * S::kLocs + loc] * stride);
            double vx = 0.0, vy = 0.0;
#pragma unroll
            for (int i = 0; i < NC; i++) {
              const double a = s_wt[i * kStep + t * S::kLocs + loc];
              vx = mcx_fma(a, d[i].x, vx);
              vy = mcx_fma(a, d[i].y, vy);
            }
            if (g0 + 2 * j + 1 >= G) vy = 0.0;  // (an odd last channel's pad, should `a` be infinite)
#pragma unroll
            for (int o = 0; o < OT; o++) {
              const double2 ww = s_w[(t * OT + o) * LPR + j];
              acc[o] = mcx_fma(ww.y, vy, mcx_fma(ww.x, vx, acc[o]));
            }
          }
        }
      }
    }
  }
#pragma unroll
  for (int o = 0; o < OT; o++) {
#pragma unroll
    for (int m = LPR / 2; m > 0; m >>= 1) acc[o] += __shfl_xor(acc[o], m);
    if (o % LPR == j && o0 + o < O && n0 + loc < N)
      y[((int64_t)b * O + o0 + o) * N + n0 + loc] = acc[o] + (bias ? bias[o0 + o] : 0.0);
  }
}

// rec[b, corner] += weight * sum_s W[s,d,k] * src[b,s,n]: the products of a pass of taps stay
// in registers, one channel a lane, then go out corner by corner: an atomic instruction adds to
// whole records of up to sixteen channels (128 bytes).
template <int NC, int LPR>
__global__ __launch_bounds__(kThreads) void scatter_records_kernel(
    const double *__restrict__ src, const double *__restrict__ map, const double *__restrict__ iw,
    const double *__restrict__ w, double *__restrict__ rec, int S_, int D, int stride, int DH,
    int DW, int N, int K, int P, int wrap, const int *__restrict__ unless) {
  if (unless && *unless != 0) return;
  using S = RecShape<LPR>;
  constexpr int kStep = S::kTaps * S::kLocs;
  constexpr int kSrc = 16;  // source channels per pass
  constexpr int kCh = LPR;
  __shared__ int s_off[NC * kStep];
  __shared__ double s_wt[NC * kStep];
  __shared__ double s_w[S::kTaps * kSrc * kCh];
  __shared__ double s_src[kSrc * S::kLocs];
  const int loc = threadIdx.x / LPR, j = threadIdx.x % LPR;
  const int n0 = blockIdx.x * S::kLocs, d0 = blockIdx.y * kCh, b = blockIdx.z;
  const int64_t DN = (int64_t)DH * DW;
  double *recb = rec + (int64_t)b * DN * stride + d0 + j;
  const bool live = d0 + j < D;
  const int pm = P == 0 ? 1 : P;
  for (int k0 = 0; k0 < K; k0 += S::kTaps) {
    const int taps = min(S::kTaps, K - k0);
    double acc[S::kTaps];
#pragma unroll
    for (int t = 0; t < S::kTaps; t++) acc[t] = 0.0;
    for (int s0 = 0; s0 < S_; s0 += kSrc) {
      const int ns = min(kSrc, S_ - s0);
      __syncthreads();
      for (int i = threadIdx.x; i < ns * S::kTaps * kCh; i += kThreads) {
        const int t = i % S::kTaps, c = i / S::kTaps % kCh, ss = i / (S::kTaps * kCh);
        s_w[(ss * S::kTaps + t) * kCh + c] =
            (t < taps && d0 + c < D) ? w[((int64_t)(s0 + ss) * D + d0 + c) * K + k0 + t] : 0.0;
      }
      for (int i = threadIdx.x; i < ns * S::kLocs; i += kThreads) {
        const int l = i % S::kLocs, ss = i / S::kLocs;
        s_src[i] = n0 + l < N ? src[((int64_t)b * S_ + s0 + ss) * N + n0 + l] : 0.0;
      }
      __syncthreads();
      for (int ss = 0; ss < ns; ss++) {
        const double v = s_src[ss * S::kLocs + loc];
#pragma unroll
        for (int t = 0; t < S::kTaps; t++) {
          acc[t] = mcx_fma(s_w[(ss * S::kTaps + t) * kCh + j], v, acc[t]);
        }
      }
    }
    for (int p = 0; p < pm; p++) {
      __syncthreads();
      fill_tap_cache<NC, LPR>(map, iw, n0, N, K, pm, p, k0, taps, DH, DW, wrap != 0, -1, s_off,
                              s_wt);
      __syncthreads();
#pragma unroll
      for (int t = 0; t < S::kTaps; t++) {
#pragma unroll
        for (int i = 0; i < NC; i++) {
          const int slot = i * kStep + t * S::kLocs + loc;
          const int off = t < taps ? s_off[slot] : -1;
          if (live && off >= 0) atomic_add(recb + (int64_t)off * stride, s_wt[slot] * acc[t]);
        }
      }
    }
  }
}

// part[range][k][a][g] = sum over a range of (b, n) of plain[b,a,n] * sample(gath[b,g], map[n,k]).
// A workgroup takes AT plain channels, 2 * LPR gathered ones and KT taps.  A tile is one run of kLocs
// locations; for one tap it is kSub, whose record reads are in flight together.
// KT is 1, or kGradTaps over up to four plain channels where there are taps and locations enough (grad_shape): the
// taps of a location are one piece of the map, and one by one each workgroup reads the lines of all of them;
// neighbouring taps often meet each other's records too.  Three, not as many as a lane has registers for the sums of:
// with nine, two waves a SIMD instead of four, coherent maps were slower than tap by tap (whole weight gradient, 10 -> 1 channels,
// nine taps, us, tap by tap, three and nine: 100 000 locations, shuffled pixels 70, 47, 60, coherent 43, 42, 58; 300 000 240, 117,
// 132 and 131, 95, 125).
constexpr int kGradTaps = 3;
template <int NC, int LPR, int AT, int KT>
__global__ __launch_bounds__(kThreads) void weight_grad_records_kernel(
    const double *__restrict__ plain, const double *__restrict__ rec,
    const double *__restrict__ map, const double *__restrict__ iw, double *__restrict__ part,
    int A, int G, int stride, int GH, int GW, int N, int K, int P, int wrap, int tiles_per_img,
    int64_t total_tiles, int ranges) {
  using S = RecShape<LPR>;
  constexpr int kSub = KT > 1 ? 1 : LPR == 2 ? 2 : 4;
  constexpr int kTile = kSub * S::kLocs;
  constexpr int kSlots = KT * kTile;  // of the tap cache: [tap][location]
  __shared__ int s_off[NC * kSlots];
  __shared__ double s_wt[NC * kSlots];
  __shared__ double s_plain[AT * kTile];
  const int loc = threadIdx.x / LPR, j = threadIdx.x % LPR;
  const int kgroups = (K + KT - 1) / KT;
  const int k0 = (int)(blockIdx.x % kgroups) * KT, range = blockIdx.x / kgroups;
  const int taps = min(KT, K - k0);
  const int a0 = blockIdx.y * AT, g0 = blockIdx.z * S::kCh;
  const int64_t GN = (int64_t)GH * GW;
  const int pm = P == 0 ? 1 : P;
  const bool live = g0 + 2 * j < stride;
  double2 acc[KT][AT];
#pragma unroll
  for (int t = 0; t < KT; t++)
#pragma unroll
    for (int a = 0; a < AT; a++) acc[t][a] = make_double2(0.0, 0.0);
  const int64_t t0 = total_tiles * range / ranges, t1 = total_tiles * (range + 1) / ranges;
  for (int64_t tile = t0; tile < t1; tile++) {
    const int b = (int)(tile / tiles_per_img);
    const int n0 = (int)(tile - (int64_t)b * tiles_per_img) * kTile;
    const double *src = rec + (int64_t)b * (GN + 1) * stride + g0 + 2 * j;
    for (int p = 0; p < pm; p++) {
      __syncthreads();
      if (p == 0)
        for (int i = threadIdx.x; i < AT * kTile; i += kThreads) {
          const int l = i % kTile, a = a0 + i / kTile;
          s_plain[i] = (a < A && n0 + l < N) ? plain[((int64_t)b * A + a) * N + n0 + l] : 0.0;
        }
      if constexpr (KT > 1) {
        fill_tap_cache<NC, LPR, KT>(map, iw, n0, N, K, pm, p, k0, taps, GH, GW, wrap != 0, (int)GN,
                                    s_off, s_wt);
      } else {
        for (int l = threadIdx.x; l < kTile; l += kThreads) {
          if (n0 + l < N) {
            resolve_records<NC>(map, iw, ((int64_t)(n0 + l) * K + k0) * pm + p, GH, GW, wrap != 0,
                                (int)GN, s_off + l, s_wt + l, kTile);
          } else {
#pragma unroll
            for (int i = 0; i < NC; i++) {
              s_off[i * kTile + l] = (int)GN;
              s_wt[i * kTile + l] = 0.0;
            }
          }
        }
      }
      __syncthreads();
      if (live) {
        // units, whose records are in flight together: the taps of a location, or one tap's locations
        constexpr int kUnits = KT > 1 ? KT : kSub;
        double2 d[kUnits][NC];
#pragma unroll
        for (int u = 0; u < kUnits; u++) {
          // (past the last tap it is read again and not used)
          const int v = KT > 1 ? min(u, taps - 1) : u;
#pragma unroll
          for (int i = 0; i < NC; i++)
            d[u][i] = *reinterpret_cast<const double2 *>(
                src + (int64_t)s_off[i * kSlots + v * S::kLocs + loc] * stride);
        }
#pragma unroll
        for (int u = 0; u < kUnits; u++) {
          if (KT > 1 && u >= taps) break;
          double vx = 0.0, vy = 0.0;
#pragma unroll
          for (int i = 0; i < NC; i++) {
            const double f = s_wt[i * kSlots + u * S::kLocs + loc];
            vx = mcx_fma(f, d[u][i].x, vx);
            vy = mcx_fma(f, d[u][i].y, vy);
          }
#pragma unroll
          for (int a = 0; a < AT; a++) {
            const double g = s_plain[a * kTile + (KT > 1 ? 0 : u * S::kLocs) + loc];
            double2 &sum = acc[KT > 1 ? u : 0][a];
            sum.x = mcx_fma(g, vx, sum.x);
            sum.y = mcx_fma(g, vy, sum.y);
          }
        }
      }
    }
  }
  // sum over the locations' lanes of each wave, then over the four waves through LDS
  __shared__ double2 s_red[kThreads / 64][KT * AT][LPR];
#pragma unroll
  for (int t = 0; t < KT; t++)
#pragma unroll
    for (int a = 0; a < AT; a++) {
#pragma unroll
      for (int m = 32; m >= LPR; m >>= 1) {
        acc[t][a].x += __shfl_xor(acc[t][a].x, m);
        acc[t][a].y += __shfl_xor(acc[t][a].y, m);
      }
      if ((int)(threadIdx.x & 63) < LPR) s_red[threadIdx.x >> 6][t * AT + a][j] = acc[t][a];
    }
  __syncthreads();
  for (int i = threadIdx.x; i < taps * AT * LPR; i += kThreads) {
    const int ta = i / LPR, jj = i % LPR, g = g0 + 2 * jj, k = k0 + ta / AT, a = ta % AT;
    double2 v = s_red[0][ta][jj];
    for (int q = 1; q < kThreads / 64; q++) {
      v.x += s_red[q][ta][jj].x;
      v.y += s_red[q][ta][jj].y;
    }
    if (a0 + a < A) {
      double *out = part + (((int64_t)range * K + k) * A + a0 + a) * G + g;
      if (g < G) out[0] = v.x;
      if (g + 1 < G) out[1] = v.y;
    }
  }
}

// gw[a][g][k] = sum over the ranges of part[range][k][a][g]: a wave per element
__global__ __launch_bounds__(kThreads) void reduce_records_kernel(const double *__restrict__ part,
                                                                  double *__restrict__ gw, int AG,
                                                                  int K, int ranges) {
  const int64_t e = (int64_t)blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (e >= (int64_t)AG * K) return;
  double v = 0.0;
  for (int r = lane; r < ranges; r += 64) v += part[(int64_t)r * AG * K + e];
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m);
  if (lane == 0) {
    const int64_t k = e / AG, ag = e - k * AG;
    gw[ag * K + k] = v;
  }
}

// ---- scattering before the product ----
// With few source channels (S) and more destination ones (D) it is S values per corner that are
// added, into a plane per (tap, source channel), and the product that follows reads every plane
// once:  T[k][s][p] = sum over the corners on p of weight * src[s],  dst[d][p] = sum W[s][d][k] T[k][s][p].
// The two corners of a row are neighbouring lanes and neighbouring doubles: one request of 64 bytes
// for both (a record of ten channels takes one and a half for either), and under a coherent map a
// wave's 32 pixels are as many neighbours.
// A double of a plane that nothing was added to keeps its first value, -0: its product is left
// out, so that an infinite W does not make NaN where no corner lies.  (What -0 adds is nothing.)
// Bound: the requests of the additions, and clearing the planes.  1 -> 10 channels, nine taps, one
// image of 200x500, shuffled: 375 -> 120 us for the whole
// product (16 channels 388 -> 123); see planes_scatter_applies.
constexpr unsigned long long kUntouched = 0x8000000000000000ull;

__global__ __launch_bounds__(kThreads) void begin_planes_kernel(double2 *__restrict__ t,
                                                                int64_t count) {
  const int64_t stride = (int64_t)gridDim.x * kThreads;
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < count; i += stride)
    t[i] = make_double2(-0.0, -0.0);
}

// NC == 4: two lanes a map location, one for either column of corners.
template <int NC>
__global__ __launch_bounds__(kThreads) void scatter_planes_kernel(
    const double *__restrict__ src, const double *__restrict__ map, const double *__restrict__ iw,
    double *__restrict__ planes, int S, int DH, int DW, int N, int K, int pm, int wrap) {
  constexpr int kCols = NC == 4 ? 2 : 1;
  const int n = blockIdx.x * (kThreads / kCols) + threadIdx.x / kCols;
  const int col = threadIdx.x % kCols, k = blockIdx.y, b = blockIdx.z;
  if (n >= N) return;
  const int64_t DN = (int64_t)DH * DW;
  double *t = planes + ((int64_t)b * K + k) * S * DN;
  const double *v = src + (int64_t)b * S * N + n;
  for (int p = 0; p < pm; p++) {
    int off[NC];
    double wt[NC];
    resolve_records<NC>(map, iw, ((int64_t)n * K + k) * pm + p, DH, DW, wrap != 0, -1, off, wt, 1);
#pragma unroll
    for (int r = 0; r < (NC == 4 ? 2 : 1); r++) {
      const int o0 = off[(2 * r) % NC], o1 = off[(2 * r + 1) % NC];
      const double a0 = wt[(2 * r) % NC], a1 = wt[(2 * r + 1) % NC];
      const int o = col ? o1 : o0;
      const double a = col ? a1 : a0;
      if (o < 0) continue;
      // (a product of -0 is added as +0: the pixel has been added to)
      for (int c = 0; c < S; c++) atomic_add(t + c * DN + o, a * v[(int64_t)c * N] + 0.0);
    }
  }
}

constexpr int kPlaneD = 16;    // destination channels per workgroup
constexpr int kPlanes = 64;    // planes of an image, at most
constexpr int kPlaneRun = 8;   // planes whose loads are in flight
// The weights sit in LDS and eight planes are read together: a plane of a small image, whose few
// waves have nothing else to do meanwhile, takes 0.64 us
// instead of 0.95 (25 taps of 64x128, 1 -> 10 channels: the whole product 51 -> 45 us).
__global__ __launch_bounds__(kThreads) void product_planes_kernel(
    const double *__restrict__ planes, const double *__restrict__ w,
    const double *__restrict__ bias, double *__restrict__ dst, int S, int D, int64_t DN, int K) {
  __shared__ double s_w[kPlanes][kPlaneD];
  const int64_t p = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  const int d0 = blockIdx.y * kPlaneD, b = blockIdx.z, count = K * S;
  for (int i = threadIdx.x; i < count * kPlaneD; i += kThreads) {
    const int q = i / kPlaneD, k = q / S, c = q - k * S, d = min(d0 + i % kPlaneD, D - 1);
    s_w[q][i % kPlaneD] = w[((int64_t)c * D + d) * K + k];
  }
  const double *t = planes + (int64_t)b * count * DN + min(p, DN - 1);
  double acc[kPlaneD];
#pragma unroll
  for (int d = 0; d < kPlaneD; d++) acc[d] = bias && d0 + d < D ? bias[d0 + d] : 0.0;
  __syncthreads();
  for (int q0 = 0; q0 < count; q0 += kPlaneRun) {
    double v[kPlaneRun];
#pragma unroll
    for (int j = 0; j < kPlaneRun; j++) v[j] = t[(int64_t)min(q0 + j, count - 1) * DN];
#pragma unroll
    for (int j = 0; j < kPlaneRun; j++) {
      if (q0 + j >= count) break;
      const bool touched = __builtin_bit_cast(unsigned long long, v[j]) != kUntouched;
#pragma unroll
      for (int d = 0; d < kPlaneD; d++)
        acc[d] = touched ? mcx_fma(s_w[q0 + j][d], v[j], acc[d]) : acc[d];
    }
  }
  if (p >= DN) return;
#pragma unroll
  for (int d = 0; d < kPlaneD; d++)
    if (d0 + d < D) dst[((int64_t)b * D + d0 + d) * DN + p] = acc[d];
}

size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

// Tiles, ranges and channel blocks of the weight gradient: about 2048 workgroups, eight per CU; of several
// taps, whose registers leave room for four or three, 1024 or 768.
struct GradShape {
  int lpr, at, taps;
  int64_t tiles_per_img, total, ranges, ablocks, gblocks, kgroups;
};
GradShape grad_shape(int64_t B, int64_t A, int64_t G, int64_t N, int64_t K) {
  GradShape q;
  q.lpr = lanes_per_record(G);
  q.at = A == 1 ? 1 : A <= 4 ? 4 : 16;
  q.ablocks = (A + q.at - 1) / q.at;
  q.gblocks = (read_stride(G) + 2 * q.lpr - 1) / (2 * q.lpr);
  // Several taps a workgroup where there are taps and locations enough and the taps fill eight ninths of the
  // workgroups': with fewer, workgroups of one tap are more and have the loads of four locations in flight (whole weight gradients,
  // us, one tap and three, shuffled and coherent maps.  10 -> 1 channels, 67 000 locations, six taps 35, 31 and 28, 28; seven 40,
  // 35 and 30, 33; eight 47, 36 and 33, 33; nine 47, 37 and 33, 33; ten 47, 41 and 35, 36; 25 98, 67 and 61, 60; 49 500, nine 35, 30 and
  // 27, 28; 100 000, four 41, 38 and 29, 34; five 41, 38 and 31, 34; six 51, 38 and 36, 35.  From 196 608 locations on five taps are
  // enough: 300 000, four 115, 86 and 68, 73; five 140, 87 and 77, 72; ten 263, 144 and 133, 115.  2 -> 1, 67 000, six 21, 21 and 18,
  // 18; nine 27, 22 and 23, 19.  Two to four plain channels, whose sums take the registers of a wave, nine coherent taps:
  // 4 -> 2 50 000 23, 24; 66 000 27, 26; 10 -> 4 66 000 37, 37; ten taps 100 000 46, 55; 25 66 000 64, 73; 150 000 145, 145.)
  const bool filled = K * 9 >= (K + kGradTaps - 1) / kGradTaps * kGradTaps * 8;
  const bool several = q.at == 1   ? (filled && K >= 6 && B * N >= 1 << 16) || (K >= 5 && B * N >= 3 << 16)
                       : q.at == 4 ? filled && K >= 8 && B * N >= (K > 9 ? 1 << 17 : 1 << 16)
                                   : false;
  const int64_t taps = several ? kGradTaps : 1;
  q.taps = (int)taps;
  const int64_t tile = (taps > 1 ? 1 : q.lpr == 2 ? 2 : 4) * (kThreads / q.lpr);
  q.tiles_per_img = (N + tile - 1) / tile;
  q.total = B * q.tiles_per_img;
  q.kgroups = (K + taps - 1) / taps;
  const int64_t per_range = q.kgroups * q.ablocks * q.gblocks;
  q.ranges = std::max<int64_t>(1, std::min(q.total, (taps == 1 ? 2048 : q.at == 1 ? 1024 : 768) / per_range));
  return q;
}

bool wraps(int interp) { return canonical_interp(interp) == kInterpBispherical; }

int make_records(const double *x, double *rec, int64_t B, int64_t C, int64_t N, hipStream_t s,
                 const int *unless = nullptr) {
  const int64_t stride = read_stride(C);
  const dim3 grid(div_up(N + 1, kThreads), div_up(stride, 16), (unsigned)B);
  hipLaunchKernelGGL(to_records_kernel, grid, dim3(kThreads), 0, s, x, rec, (int)C, (int)stride, N,
                     unless);
  MCX_HIP_CHECK_LAUNCH();
  return 0;
}

// Whether the map is examined (coherent) and `count` doubles cleared.
int begin_records(const double *map, int64_t N, int64_t K, int64_t P, int interp, int *coherent,
                  double *clear, int64_t count, hipStream_t s) {
  const unsigned blocks =
      (unsigned)std::max<int64_t>(1, std::min<int64_t>((count / 2 + 1023) / 1024, 8192));
  hipLaunchKernelGGL(begin_records_kernel, dim3(blocks), dim3(kThreads), 0, s, map, N, (int)K,
                     (int)(P == 0 ? 1 : P), canonical_interp(interp) == kInterpNearest ? 1 : 0,
                     coherent, (double2 *)clear, count / 2);
  MCX_HIP_CHECK_LAUNCH();
  return 0;
}

size_t gather_record_bytes(int64_t B, int64_t G, int64_t SN) {
  return align256((size_t)(B * (SN + 1) * read_stride(G)) * sizeof(double));
}
size_t scatter_record_bytes(int64_t B, int64_t D, int64_t DN) {
  return align256((size_t)(B * DN * add_stride(D)) * sizeof(double));
}

// ---- where the map decides ----
// Neither form is better for every map, and which kind the map is only the device knows: it is
// examined, both forms are launched, one returns at once.  That costs 5 to 9 us a call, which the
// rules' lines leave below the difference.  (us, scalar / records / with the map examined)
// One or two taps: those of a coherent map are reads of neighbouring pixels, which planes serve as
// well, without the copy.  362x724, 64 -> 8 channels, one tap: 102 / 330 / 111, shuffled
// 503 / 338 / 346; 16 -> 8, two taps 54 / 88 / 64, shuffled 243 / 90 / 98, but 16 -> 32 157 / 148,
// and at 256x512 64 -> 8 of two taps 175 / 127, 64 -> 32 of one 174 / 163.
bool gather_asks_map(int64_t B, int64_t G, int64_t O, int64_t N, int64_t K) {
  return N > 1 && G > 1 && (K == 1 || (K == 2 && O <= 16)) && B * N >= 196608 &&
         B * N * G >= ((int64_t)3 << 20);
}
// Scattering: neighbouring lanes of the scalar kernel add to neighbouring pixels of a plane, eight
// a request, where records take a request or two each.  256x512, nine taps, latitude map: 1 -> 10
// channels 124 / 142 / 134, 4 -> 5 66 / 106 / 78, 1 -> 17 203 / 292 / 224; fractional rows and
// columns 1 -> 10 278 / 341 / 288; shuffled 2008 / 445 / 450.  (64x128 1 -> 10: 19 / 18 / 26.)  From
// nine source channels on the products cost the scalar kernel what it saves (16 -> 5 98 / 113, 16 ->
// 24 360 / 325), except where the last of three or more runs of eight holds a channel or two
// (16 -> 17 239 / 315).
bool scatter_asks_map(int64_t B, int64_t S, int64_t N, int64_t K) {
  return N > 1 && S <= 8 && B * N * K >= ((int64_t)1 << 20);
}

}  // namespace

// A grid has at most 65535 workgroups in its second and third direction.
static bool records_fit(int64_t B, int64_t C1, int64_t C2, int64_t K) {
  return B <= 65535 && C1 <= 65535 && C2 <= 65535 && K <= 2048;
}

// Where records pay (us, scalar kernel against records; 8x8 to 500x1000 pixels, one image unless
// said otherwise, coherent and shuffled maps).
// The scalar gather is one launch less and walks G * K samples per thread one after the other.
// Few of them are sooner done, unless there are locations enough to fill the card many times
// over: 8x8, two channels of 4 taps to one 5.5 / 7.7, to eight 8.4 / 7.9, 64 of 9 taps 653 / 40;
// 500x1000, 2 -> 32 of 4 taps 105 / 77, shuffled 500 / 104.  One channel has no neighbours to
// share a line with: 128x256 9 taps 8 / 10, 256x512 10 / 15; 362x724 33 / 28, shuffled 56 / 45, to
// 32 channels 117 / 75.
bool records_gather_applies(int64_t B, int64_t G, int64_t O, int64_t N, int64_t K) {
  if (!records_fit(B, G, O, K)) return false;
  const bool large = B * N >= 196608;
  if (G == 1) return large && K >= 9;
  return G * K >= (O >= 4 ? 8 : 16) || (large && G * K >= 3);
}

// The scalar scatter loses from two destination channels on (16x16 20 / 11 at ten; 256x512
// shuffled 2008 / 450); with one on either side it writes what it must: 8.6 / 10.8, 203 / 214.
bool records_scatter_applies(int64_t B, int64_t S, int64_t D, int64_t K) {
  return records_fit(B, S, D, K) && (S > 1 || D > 1);
}

// The scalar weight gradient has one workgroup per (gathered channel, tap, eight plain channels)
// walk all locations: short walks beat three launches as long as the workgroups are few.  10 -> 1
// channels, 9 taps: 32x32 6.0 / 10.5, 45x45 9 / 10, 64x64 13 / 10, 91x91 28 / 12; 64 -> 64
// 16x16 20 / 22 (9.4 M products), 45x45 98 / 57; 128 -> 128 8x8 51 / 42 (9.4 M).
bool records_weight_grad_applies(int64_t B, int64_t A, int64_t G, int64_t N, int64_t K) {
  if (!records_fit(B, A, G, K)) return false;
  return B * N >= 2048 || A * G * K * B * N >= ((int64_t)1 << 23);
}

// Scattering before the product, where the source channels are few beside the destination's (us for
// the scalar kernel or records, as the rules above have it, against this; one image, shuffled maps,
// coherent ones in brackets).  Nine taps of 90x180: 1 -> 6 34 / 28 (35 / 27), 1 -> 10 61 / 28 (46 / 27),
// 1 -> 64 213 / 30, 2 -> 12 63 / 49 (52 / 46), 2 -> 32 112 / 50, 4 -> 64 217 / 94; of 200x500 1 -> 10
// 375 / 121 (108 / 61), 1 -> 4 187 / 117 (48 / 57), 2 -> 5 205 / 221, 5 -> 16 390 / 525 (157 / 231).  Other
// taps of 90x180, 1 -> 10: 25 151 / 69, 64 378 / 160; of 500x1000 one 218 / 66, 25 4494 / 1284, 64
// 11397 / 3261.
// A pixel of the product reads its planes eight at a time, however few pixels there are: a plane
// is 0.64 us and 100 ps a location, a record 28 ps a location, tap and channel, and 3 us more for all.
// Nine taps of 10x20 4 -> 64 23 / 36, of 32x64 2 -> 12 23 / 25, of 64x128 38 / 33 (31 / 34); 25 taps of
// 10x20 1 -> 10 24 / 26, of 32x64 30 / 31, of 45x90 49 / 35 (39 / 34); 64 taps of 45x90 1 -> 6 64 / 77, of
// 64x128 107 / 105.  (Taps outside the image all meet in one pixel: nine taps of a shuffled 60x90 with
// such a border 1 -> 10 37 / 20, 2 -> 12 40 / 30.)
// The planes are K * S doubles a pixel to clear and to read: not many more than additions, or than a
// record.  (64 taps of one channel take up to ten times a record's scratch; with less than they need
// records run.)
static bool planes_scatter_applies(int64_t B, int64_t S, int64_t D, int64_t DN, int64_t N, int64_t K) {
  return D >= 6 * S && K * S <= kPlanes && (S * DN <= 2 * N || K * S <= D) &&
         K * (B * N * (28 * add_stride(D) - 100 * S) - 640000 * S) > -3000000;
}
static size_t planes_bytes(int64_t B, int64_t S, int64_t DN, int64_t K) {
  return align256((size_t)(B * K * S * DN + 1) * sizeof(double));
}

#define MCX_LPR(C, CALL)              \
  switch (lanes_per_record(C)) {      \
    case 2: { CALL(2) } break;        \
    case 4: { CALL(4) } break;        \
    default: { CALL(8) } break;       \
  }

// (the word about the map last)
size_t records_gather_bytes(int64_t B, int64_t G, int64_t O, int64_t SN, int64_t N, int64_t K) {
  return gather_record_bytes(B, G, SN) + (gather_asks_map(B, G, O, N, K) ? 256 : 0);
}

int records_gather_product(const double *src, const double *map, const double *iw, const double *w,
                           const double *bias, double *y, void *ws, int64_t B, int64_t G,
                           int64_t O, int64_t SH, int64_t SW, int64_t N, int64_t K, int64_t P,
                           int interp, hipStream_t s) {
  double *rec = (double *)ws;
  int *coherent = nullptr;
  if (gather_asks_map(B, G, O, N, K)) {
    coherent = (int *)((char *)ws + gather_record_bytes(B, G, SH * SW));
    if (int rc = begin_records(map, N, K, P, interp, coherent, nullptr, 0, s)) return rc;
  }
  if (int rc = make_records(src, rec, B, G, SH * SW, s, coherent)) return rc;
  const int stride = (int)read_stride(G);
  const bool one = canonical_interp(interp) == kInterpNearest;
#define MCX_RUN(NC, LPR, OT)                                                                     \
  hipLaunchKernelGGL((gather_records_kernel<NC, LPR, OT>),                                       \
                     dim3(div_up(N, kThreads / LPR), div_up(O, OT), (unsigned)B), dim3(kThreads), \
                     0, s, rec, map, iw, w, bias, y, (int)G, stride, (int)O, (int)SH, (int)SW,   \
                     (int)N, (int)K, (int)P, wraps(interp) ? 1 : 0, coherent);
#define MCX_OT(NC, LPR)                             \
  if (O == 1) { MCX_RUN(NC, LPR, 1) }               \
  else if (O <= 4) { MCX_RUN(NC, LPR, 4) }          \
  else { MCX_RUN(NC, LPR, 16) }
#define MCX_NC(LPR) if (one) { MCX_OT(1, LPR) } else { MCX_OT(4, LPR) }
  MCX_LPR(G, MCX_NC)
#undef MCX_NC
#undef MCX_OT
#undef MCX_RUN
  MCX_HIP_CHECK_LAUNCH();
  if (!coherent) return 0;
  return generic_gather_product<double>(src, map, iw, w, bias, y, B, G, O, SH, SW, N, K, P, interp,
                                        s, coherent);
}

// (what the form that runs with enough scratch takes, and what the call can do with)
size_t records_scatter_bytes(int64_t B, int64_t S, int64_t D, int64_t DN, int64_t N, int64_t K) {
  if (planes_scatter_applies(B, S, D, DN, N, K)) return planes_bytes(B, S, DN, K);
  return scatter_record_bytes(B, D, DN) + (scatter_asks_map(B, S, N, K) ? 256 : 0);
}
size_t records_scatter_min_bytes(int64_t B, int64_t S, int64_t D, int64_t DN, int64_t N, int64_t K) {
  const size_t records = scatter_record_bytes(B, D, DN) + (scatter_asks_map(B, S, N, K) ? 256 : 0);
  return std::min(records, records_scatter_bytes(B, S, D, DN, N, K));
}

int records_product_scatter(const double *src, const double *map, const double *iw,
                            const double *w, const double *bias, double *dst, void *ws,
                            size_t ws_bytes, int64_t B, int64_t S, int64_t D, int64_t DH, int64_t DW,
                            int64_t N, int64_t K, int64_t P, int interp, hipStream_t s) {
  const int64_t DN = DH * DW;
  if (planes_scatter_applies(B, S, D, DN, N, K) && ws_bytes >= planes_bytes(B, S, DN, K)) {
    double *planes = (double *)ws;
    const int64_t pairs = (B * K * S * DN + 1) / 2;
    const unsigned blocks =
        (unsigned)std::max<int64_t>(1, std::min<int64_t>((pairs + 1023) / 1024, 8192));
    hipLaunchKernelGGL(begin_planes_kernel, dim3(blocks), dim3(kThreads), 0, s, (double2 *)ws, pairs);
    const int pm = (int)(P == 0 ? 1 : P);
#define MCX_RUN(NC, LOCS)                                                                        \
  hipLaunchKernelGGL((scatter_planes_kernel<NC>), dim3(div_up(N, LOCS), (unsigned)K, (unsigned)B), \
                     dim3(kThreads), 0, s, src, map, iw, planes, (int)S, (int)DH, (int)DW, (int)N, \
                     (int)K, pm, wraps(interp) ? 1 : 0)
    if (canonical_interp(interp) == kInterpNearest) { MCX_RUN(1, kThreads); }
    else { MCX_RUN(4, kThreads / 2); }
#undef MCX_RUN
    hipLaunchKernelGGL(product_planes_kernel,
                       dim3(div_up(DN, kThreads), div_up(D, kPlaneD), (unsigned)B), dim3(kThreads), 0,
                       s, planes, w, bias, dst, (int)S, (int)D, DN, (int)K);
    MCX_HIP_CHECK_LAUNCH();
    return 0;
  }
  double *rec = (double *)ws;
  const int64_t stride = add_stride(D);
  int *coherent = scatter_asks_map(B, S, N, K)
                      ? (int *)((char *)ws + scatter_record_bytes(B, D, DN))
                      : nullptr;
  if (int rc = begin_records(map, N, K, P, interp, coherent, rec, B * DN * stride, s)) return rc;
  const bool one = canonical_interp(interp) == kInterpNearest;
#define MCX_RUN(NC, LPR)                                                                          \
  hipLaunchKernelGGL((scatter_records_kernel<NC, LPR>),                                           \
                     dim3(div_up(N, kThreads / LPR), div_up(D, LPR), (unsigned)B),                \
                     dim3(kThreads), 0, s, src, map, iw, w, rec, (int)S, (int)D, (int)stride,     \
                     (int)DH, (int)DW, (int)N, (int)K, (int)P, wraps(interp) ? 1 : 0, coherent);
#define MCX_NC(LPR) if (one) { MCX_RUN(1, LPR) } else { MCX_RUN(4, LPR) }
  if (D <= 2) { MCX_NC(2) }
  else if (D <= 4) { MCX_NC(4) }
  else if (D <= 8) { MCX_NC(8) }
  else { MCX_NC(16) }
#undef MCX_NC
#undef MCX_RUN
  MCX_HIP_CHECK_LAUNCH();
  hipLaunchKernelGGL(from_records_kernel, dim3(div_up(DN, kThreads), div_up(D, 16), (unsigned)B),
                     dim3(kThreads), 0, s, rec, bias, dst, (int)D, (int)stride, DN, coherent);
  MCX_HIP_CHECK_LAUNCH();
  if (!coherent) return 0;
  return generic_product_scatter<double>(src, map, iw, w, dst, B, S, D, DH, DW, N, K, P, interp, s,
                                         coherent);
}

size_t records_weight_grad_bytes(int64_t B, int64_t A, int64_t G, int64_t GN, int64_t N,
                                 int64_t K) {
  const GradShape q = grad_shape(B, A, G, N, K);
  return gather_record_bytes(B, G, GN) + align256((size_t)(q.ranges * K * A * G) * sizeof(double));
}

int records_weight_grad(const double *plain, const double *gath, const double *map,
                        const double *iw, double *gw, void *ws, int64_t B, int64_t A, int64_t G,
                        int64_t GH, int64_t GW, int64_t N, int64_t K, int64_t P, int interp,
                        hipStream_t s) {
  double *rec = (double *)ws;
  double *part = (double *)((char *)ws + gather_record_bytes(B, G, GH * GW));
  if (int rc = make_records(gath, rec, B, G, GH * GW, s)) return rc;
  const GradShape q = grad_shape(B, A, G, N, K);
  const bool one = canonical_interp(interp) == kInterpNearest;
#define MCX_RUN_TAPS(NC, LPR, AT, KT)                                                            \
  hipLaunchKernelGGL((weight_grad_records_kernel<NC, LPR, AT, KT>),                              \
                     dim3((unsigned)(q.ranges * q.kgroups), (unsigned)q.ablocks, (unsigned)q.gblocks),   \
                     dim3(kThreads), 0, s, plain, rec, map, iw, part, (int)A, (int)G,            \
                     (int)read_stride(G), (int)GH, (int)GW, (int)N, (int)K, (int)P,              \
                     wraps(interp) ? 1 : 0, (int)q.tiles_per_img, q.total, (int)q.ranges);
#define MCX_RUN(NC, LPR, AT)                                          \
  if (q.taps == 1) { MCX_RUN_TAPS(NC, LPR, AT, 1) }                   \
  else { MCX_RUN_TAPS(NC, LPR, AT, (AT <= 4 ? kGradTaps : 1)) }
#define MCX_AT(NC, LPR)                             \
  if (q.at == 1) { MCX_RUN(NC, LPR, 1) }            \
  else if (q.at == 4) { MCX_RUN(NC, LPR, 4) }       \
  else { MCX_RUN(NC, LPR, 16) }
#define MCX_NC(LPR) if (one) { MCX_AT(1, LPR) } else { MCX_AT(4, LPR) }
  MCX_LPR(G, MCX_NC)
#undef MCX_NC
#undef MCX_AT
#undef MCX_RUN_TAPS
#undef MCX_RUN
  MCX_HIP_CHECK_LAUNCH();
  hipLaunchKernelGGL(reduce_records_kernel, dim3(div_up(A * G * K, kThreads / 64)), dim3(kThreads),
                     0, s, part, gw, (int)(A * G), (int)K, (int)q.ranges);
  MCX_HIP_CHECK_LAUNCH();
  return 0;
}
#undef MCX_LPR

}  // namespace mcx
