// Weight gradient of fp32 images over maps whose neighbouring pixels sample neighbouring pixels
// (every kernel of an equirectangular projection: along a row of the image a tap moves with the
// pixel), on the bf16 matrix instructions with both operands split into three bf16 parts as in
// mcx_conv_split.hip.
//   gW[a,g,k] = sum_{b,n} plain[b,a,n] * sample(gath[b,g], map[n,k])
//   * The sum runs over pixels, so a lane's matrix operand is eight consecutive pixels of one
//     channel.  Where the eight taps of such a group read a run of neighbouring pixels, a thread
//     fetches the run - nine elements, or sixteen for taps two pixels apart - with two to four
//     16-byte loads per row of corners instead of two loads per sample: the texture path takes
//     four lanes per clock whatever the width, which had cost as much as the fp32 matrix
//     instructions (16 loads x 16 clocks for a unit of 8 samples a thread).  It interpolates and
//     splits the eight samples and leaves them in LDS as fragments of the matrix instruction,
//     which the four waves multiply by sixteen plain channels each, whose fragments they keep in
//     registers for all taps of a tile.
//   * resolve_runs_kernel finds the runs, once per call: per (group, tap) the run's offset under
//     either row of corners and the corner weights of its pixels.  A run that jumps once (the seam
//     of a wrapping map: one group in 64 of a row of 512) is fetched element by element, a group
//     that is none corner by corner.
//   * Maps with more groups that are no runs than the gain bears (RunPlan::limit), and sums that are
//     not finite (an infinity or NaN among the operands, or values the split does not hold) are left to
//     weight_grad_mfma_kernel, whose launch follows: state[0] says that this kernel has done the
//     work, state[1] that a sum was not finite.  Where resolve_runs_kernel sees at once that the map has
//     no runs, it resolves the taps for that kernel instead.
// Bound: vector and matrix instructions, which take turns (90 + 24 a unit: 65 % of the time at the
// clock that it runs at, 2.0 GHz), and the LDS round trip and barrier of a unit, which three waves
// per SIMD do not quite cover.  A wave of 32 plain channels (half the LDS reads) needs 250 registers,
// and at two waves per SIMD everything is waited for: 820 us where this takes 735.
// Measured in one run each, fp32 instructions -> this: 8 x 64 -> 64 channels of 256 x 512, nine taps:
// 793 -> 672 us; 3 x 24 -> 40 of 125 x 250, fractional rows, 100 -> 66; transposed 4 x 64 -> 32 from
// 128 x 256 onto twice that (taps two pixels apart) 105 -> 71.
// Accuracy: the instruction rounds its sums downwards, so that 24 of them a tile lose up to 24 units
// of the last place, all one way.  The products of the leading parts, 16 bits each, are summed in an
// accumulator of their own, which rounds next to nothing; what the other five lose is 2^-8 of that;
// and the sign of every other tile is turned.  Distance from 64 bits in 2-norm, in units of 1e-7, fp32
// instructions / one accumulator / this, 16 -> 64 channels, nine taps:
//   pixels     operands normal       positive             behind a ReLU
//   128        1.49 / 1.55 / 0.70    0.93 / 1.25 / 0.67   0.61 / 1.11 / 0.52
//   256        1.53 / 1.60 / 0.72    0.71 / 0.93 / 0.58   0.55 / 0.88 / 0.48
//   2 048      2.14 / 1.67 / 0.90    0.60 / 0.52 / 0.45   0.51 / 0.53 / 0.46
//   131 072    3.73 / 2.87 / 2.57    1.14 / 1.14 / 1.13   1.13 / 1.13 / 1.13
//   1 048 576  7.21 / 3.02 / 2.71    1.15 / 1.13 / 1.13   1.11 / 1.13 / 1.13
// (2 to 64 pixels 0.3 to 0.7 against 0.3 to 1.5; two of a hundred values not zero 0.33 to 2.6 against
// 0.32 to 2.7.)
#include "mcx_conv.h"
#include "mcx_conv_runs.h"
#include "mcx_mfma_common.h"

namespace mcx {
namespace {

constexpr int kRunThreads = 256;
constexpr int kRunA = 64;          // plain channels per workgroup
constexpr int kRunTaps = 9;        // taps per workgroup, at most
constexpr int kRunStatWords = 1024;

// Groups of eight pixels are numbered strip by strip, a strip being up to eight groups wide: the
// tiles of a workgroup then follow one another down the image, and the rows that the taps of one
// tile read are in the L2 for the next (row by row, the 64 workgroups of an XCD touch 21 MB
// between two uses of a row: 2.1 GB from memory instead of 0.8 at 8 x 64 channels of 256 x 512).
constexpr int kStrip = 8;
struct GroupPlace {
  int row, col;  // of the group's first pixel
};
__device__ inline GroupPlace group_place(int g, int MH, int gpr) {
  const int strip = g / (MH * kStrip), in = g - strip * (MH * kStrip);
  const int width = min(kStrip, gpr - strip * kStrip);
  const int row = in / width;
  return GroupPlace{row, (strip * kStrip + in - row * width) * 8};
}

// What a (group, tap) reads.  kind 0: `upper` and `lower` are the byte offsets of the run under
// either row of corners.  kElements: elements from `at` on lie `jump` bytes further (behind the seam of
// a wrapping map), or the run reaches past its plane: fetched one by one.  kCorners: no run.
struct RunDesc {
  int upper, lower, jump, kind_at;  // kind in the two lowest bits, `at` above them
};
constexpr int kElements = 1, kCorners = 2, kNowhere = 64;

// desc[group][tap]; wts[group][tap][row of corners][pixel][2]: corner weights, scaled for the
// split; offs (same shape): byte offsets of the corners, where the group is no run.  stats[block]:
// {4 * groups that are no runs + 2 * (these tables were not written) + (a corner of the lower row has
// a weight), groups fetched element by element}.  Eight lanes share a group.  wanted: the tables are,
// should the map have runs.
template <int NCORN, int ST>
__global__ __launch_bounds__(256) void resolve_runs_kernel(
    const float *__restrict__ map, const float *__restrict__ iw, RunDesc *__restrict__ desc,
    float2 *__restrict__ wts, uint2 *__restrict__ offs, int2 *__restrict__ stats,
    int *__restrict__ state, int GH, int GW, int MH, int MW, int K, int wrap, int weighted,
    int wanted, const TapTable taps) {
  __shared__ int count[3];
  if (threadIdx.x < 3) count[threadIdx.x] = 0;
  if (blockIdx.x == 0 && threadIdx.x == 0) state[1] = 0;
  __syncthreads();
  const int gpr = (MW + 7) >> 3;
  const int total = MH * gpr * K * 8;
  const int lane = threadIdx.x & 63, first = lane & 56;
  int no_runs = 0, elements = 0;
  bool lower = false;
  auto of_group = [&](bool x) {
    return (unsigned)(__builtin_amdgcn_ballot_w64(x) >> first) & 0xffu;
  };
  // One pixel of a (group, tap) q; returns the kind of its group (the same in its
  // eight lanes).  `write`: into the tables.
  auto examine = [&](int q, int e, bool exists, bool write) __attribute__((always_inline)) {
    const int g = q / K, k = q - g * K;
    const GroupPlace at_px = group_place(g, MH, gpr);
    const int row = at_px.row, j = at_px.col + e;
    const bool live = exists && j < MW;
    const int64_t s = ((int64_t)row * MW + min(j, MW - 1)) * K + k;
    const float2 xy = reinterpret_cast<const float2 *>(map)[s];
    const float scale = live ? (weighted ? iw[s] * kSplitScale : kSplitScale) : 0.f;
    PairTap<NCORN> tap;
    resolve_pairs<NCORN, 1>(xy.x, xy.y, GH, GW, wrap != 0, scale, tap);
    // run of the first corner in use (as the offset its element 0 would have), the first element
    // that is not on it, and the run from there on
    int run[2] = {0, 0}, jump[2] = {0, 0}, at[2] = {kNowhere, kNowhere};
    bool any[2] = {false, false}, fits = true;
#pragma unroll
    for (int r = 0; r < (NCORN == 4 ? 2 : 1); r++) {
      float w[2] = {tap.wt[(2 * r) % NCORN], NCORN == 4 ? tap.wt[(2 * r + 1) % NCORN] : 0.f};
      int o[2] = {(int)tap.off[(2 * r) % NCORN], (int)tap.off[(2 * r + 1) % NCORN]};
      const unsigned u0 = of_group(w[0] != 0.f), u1 = of_group(w[1] != 0.f);
      const int e0 = u0 ? __builtin_ctz(u0) : 7, e1 = u1 ? __builtin_ctz(u1) : 7;
      const int i0 = u0 ? ST * e0 : 127, i1 = u1 ? ST * e1 + 1 : 127;
      const int ia = min(i0, i1);
      any[r] = ia != 127;
      const int s0 = __shfl(o[0], first + e0), s1 = __shfl(o[1], first + e1);
      run[r] = any[r] ? (i0 < i1 ? s0 : s1) - ia : 0;
      const bool off0 = w[0] != 0.f && o[0] - ST * e != run[r];
      const bool off1 = w[1] != 0.f && o[1] - (ST * e + 1) != run[r];
      const unsigned m0 = of_group(off0), m1 = of_group(off1);
      const int f0 = m0 ? __builtin_ctz(m0) : 7, f1 = m1 ? __builtin_ctz(m1) : 7;
      const int j0 = m0 ? ST * f0 : 127, j1 = m1 ? ST * f1 + 1 : 127;
      const int ja = min(j0, j1);
      const int t0 = __shfl(o[0], first + f0), t1 = __shfl(o[1], first + f1);
      if (ja != 127) {
        at[r] = ja;
        jump[r] = (j0 <= j1 ? t0 : t1) - ja - run[r];
      }
#pragma unroll
      for (int c = 0; c < 2; c++) {
        const int i = ST * e + c;
        fits = fits && (w[c] == 0.f || o[c] == run[r] + i + (i >= at[r] ? jump[r] : 0));
      }
      if (exists && write) wts[(int64_t)(q * 2 + r) * 8 + e] = make_float2(w[0], w[1]);
      if (r == 1) lower |= any[1];
    }
    if (NCORN == 1 && exists && write) wts[(int64_t)(q * 2 + 1) * 8 + e] = make_float2(0.f, 0.f);
    // both rows break at the same element, or one of them is not in use
    if (!any[0]) at[0] = at[1], jump[0] = jump[1];
    const bool same = !any[1] || (at[1] == at[0] && jump[1] == jump[0]);
    const bool no_run = of_group(!(fits && same)) != 0;
    bool inside = at[0] == kNowhere;
#pragma unroll
    for (int r = 0; r < 2; r++) inside = inside && run[r] >= 0 && run[r] + 7 * ST + 1 < GH * GW;
    if (no_run && exists && write) {
#pragma unroll
      for (int r = 0; r < 2; r++)
        offs[(int64_t)(q * 2 + r) * 8 + e] =
            NCORN == 4 ? make_uint2(tap.off[2 * r % NCORN] * 4u, tap.off[(2 * r + 1) % NCORN] * 4u)
                       : make_uint2(tap.off[0] * 4u, tap.off[0] * 4u);
    }
    if (e == 0 && exists && write) {
      RunDesc d{run[0] * 4, run[1] * 4, jump[0] * 4, inside ? 0 : at[0] * 4 + kElements};
      if (no_run) d = RunDesc{0, 0, 0, kNowhere * 4 + kCorners};
      desc[q] = d;
    }
    return no_run ? kCorners : inside ? 0 : kElements;
  };
  // Maps without runs (a shuffled one) are not worth these tables: more than four of 32 groups spread
  // over the map, the same for every block, are none (500x1000 shuffled, 10 -> 1 channels: with tables
  // 2220 us for the call, 2121 so).  The general kernel's taps are resolved instead, which also finds
  // out whether corners of the lower row are in use; if the samples have shown that they are, nothing
  // is left to do.
  const int e = threadIdx.x & 7;
  const int sample = (int)(((uint64_t)((threadIdx.x >> 3) * 2654435769u) * (uint64_t)(total >> 3)) >> 32);
  const bool tables = __syncthreads_count(examine(sample, e, true, false) == kCorners) <= 4 * 8 && wanted;
  if (tables) {
    for (int t = blockIdx.x * 256 + threadIdx.x; t < ((total + 63) & ~63); t += gridDim.x * 256) {
      const bool exists = t < total;
      const int kind = examine(min(t, total - 1) >> 3, e, exists, true);
      no_runs += exists && e == 0 && kind == kCorners ? 1 : 0;
      elements += exists && e == 0 && kind == kElements ? 1 : 0;
    }
  } else if (NCORN == 4 && !__syncthreads_or(lower)) {
    const int64_t entries = (int64_t)taps.tiles * K * kTilePx;
    for (int64_t i = blockIdx.x * 256 + threadIdx.x; i < entries; i += gridDim.x * 256) {
      const int p = (int)(i & (kTilePx - 1)), tk = (int)(i / kTilePx);
      const int tile = tk / K, k = tk - tile * K;
      const int tile_y = tile / taps.tiles_x, tile_x = tile - tile_y * taps.tiles_x;
      const int gi = tile_y * (kTilePx >> taps.tw_shift) + (p >> taps.tw_shift);
      const int gj = (tile_x << taps.tw_shift) + (p & ((1 << taps.tw_shift) - 1));
      const int64_t s = ((int64_t)min(gi, MH - 1) * MW + min(gj, MW - 1)) * K + k;
      const float2 xy = reinterpret_cast<const float2 *>(map)[s];
      const float scale = gi < MH && gj < MW ? (weighted ? iw[s] : 1.f) : 0.f;
      PairTap<NCORN> tap;
      resolve_pairs<NCORN, 4>(xy.x, xy.y, GH, GW, wrap != 0, scale, tap);
      lower |= tap.wt[2 % NCORN] != 0.f || tap.wt[3 % NCORN] != 0.f;
      taps.table[i] = make_uint4(tap.off[0], tap.off[1 % NCORN], __builtin_bit_cast(unsigned, tap.wt[0]),
                                 __builtin_bit_cast(unsigned, tap.wt[1 % NCORN]));
    }
  }
  if (!tables) no_runs = threadIdx.x == 0 ? total / 8 / (int)gridDim.x + 1 : 0;
  if (no_runs) atomicAdd(&count[0], no_runs);
  if (elements) atomicAdd(&count[2], elements);
  if (lower) count[1] = 1;
  __syncthreads();
  if (threadIdx.x == 0) stats[blockIdx.x] = make_int2(4 * count[0] + (tables ? 0 : 2) + count[1], count[2]);
}

struct RunArgs {
  const float *plain, *gath;
  const RunDesc *desc;
  const uint2 *offs;
  const float *wts;
  const int2 *stats;
  int *state;
  float *part, *sum_part;  // sum_part: NULL, or per-range sums of the plain operand
  int A, G, GH, GW, MH, MW, K, stat_words;
  int groups;              // of an image: MH * ceil(MW / 8)
  int tiles_per_img, total_tiles, ranges, cblocks;
  int64_t limit;           // see RunPlan
};

constexpr int kTileGroups = 16;  // 128 pixels

struct RunLds {
  // Weights of a (tap, group): up to 32 floats and four that keep eight lanes' 16-byte reads on
  // different banks (with one row of corners 16 and four).
  uint4 samples[2][3][4 * 64];  // [buffer][part][fragment of 32 pixels]
  float weights[kRunTaps * kTileGroups * 36];
  RunDesc desc[kRunTaps * kTileGroups];
};

// A workgroup multiplies a block of samples, 16 gathered channels x 128 pixels of a tap, by 64 plain
// channels, a wave 16 of them.  NR: rows of corners in use; ST: pixels between the taps of
// neighbouring pixels.
template <int NR, int ST>
__device__ inline void weight_grad_runs(const RunArgs &s, RunLds &lds) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  typedef int i32x4 __attribute__((ext_vector_type(4)));
  constexpr int NV = ST == 1 ? 9 : 16;  // elements of a run
  constexpr int kRow = 16 * NR + 4;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, lq = lane >> 4;  // of the matrix operands
  // The run a thread fetches, interpolates and splits: channel pc, group pg (lanes of four along
  // the groups, which are neighbours in memory).
  const int pc = lane >> 2, pg = (lane & 3) + 4 * wave;
  const int item = xcd_contiguous_tile(blockIdx.x, gridDim.x);
  const int cg = item % s.cblocks, range = item / s.cblocks;
  const int a0 = blockIdx.y * kRunA + 16 * wave;
  const int passes = gridDim.z;  // taps of this pass: as even as they go
  const int k_base = (int)((int64_t)s.K * blockIdx.z / passes);
  const int ktaps = (int)((int64_t)s.K * (blockIdx.z + 1) / passes) - k_base;
  const int g0 = cg * 16;
  const int N = s.MH * s.MW, gpr = (s.MW + 7) >> 3;
  const unsigned plane = (unsigned)(s.GH * s.GW) * 4u;
  const int chan = (int)((unsigned)min(g0 + pc, s.G - 1) * plane);
  const int tpr = (s.total_tiles + s.ranges - 1) / s.ranges;
  const int t_begin = min(range * tpr, s.total_tiles), t_end = min(t_begin + tpr, s.total_tiles);
  // place of a lane's fragment words: eight lanes that write (two channels, four groups) and eight
  // that read together (four and four channels of neighbouring groups) fall on different banks
  auto place = [](int group, int channel) {
    return (group & 3) * 16 + (channel ^ ((group & 1) * 2 + (group & 2) * 4));
  };
  const int write_at = wave * 64 + place(pg, pc), read_at = place(lq, l15);

  floatx4 acc[kRunTaps];
#pragma unroll
  for (int k = 0; k < kRunTaps; k++) acc[k] = floatx4{0.f, 0.f, 0.f, 0.f};
  float plain_sum = 0.f;
  const bool sums = s.sum_part && cg == 0 && blockIdx.z == 0;

  // Where a tile lies (wave-uniform, stepped from tile to tile: divisions cost as much as products)
  const int strip_groups = s.MH * kStrip;
  int b = t_begin / s.tiles_per_img, first = (t_begin - b * s.tiles_per_img) * kTileGroups;
  int strip = first / strip_groups, in = first - strip * strip_groups;
  int buf = 0;
  for (int tile = t_begin; tile < t_end; ++tile) {
    const int live = min(kTileGroups, s.groups - first);
    // (sixteen groups of one full strip)
    const bool plain_tile =
        live == kTileGroups && (strip + 1) * kStrip <= gpr && in + kTileGroups <= strip_groups;
    const auto img = plane_buf(s.gath + (int64_t)b * s.G * (plane >> 2), (unsigned)s.G * plane);
    // (every other tile is multiplied with its sign turned and subtracted, so that what the sums
    // lose does not add up)
    const float sign = (tile & 1) ? -1.f : 1.f;
    int t0 = tid;  // (opaque: nothing of the preparation is kept in registers through the products)
    asm volatile("" : "+v"(t0));
    // the plain operand: sixteen rows of the tile, split into fragments in registers
    bf16x8 a[4][3];
    {
      const unsigned rows_bytes = (unsigned)s.A * (unsigned)N * 4u;
      const auto rows = plane_buf(s.plain + (int64_t)b * s.A * N, rows_bytes);
      const unsigned row_off = (unsigned)min(a0 + (t0 & 15), s.A - 1) * (unsigned)N;
      f32x4 raw[4][2];
      int n_live[4];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int gl = 4 * q + ((t0 >> 4) & 3);
        int row, col;
        if (plain_tile) {
          row = (in + gl) >> 3;
          col = (strip * kStrip + ((in + gl) & (kStrip - 1))) * 8;
          n_live[q] = s.MW - col;
        } else {
          const GroupPlace px = group_place(first + min(gl, live - 1), s.MH, gpr);
          row = px.row;
          col = px.col;
          n_live[q] = gl < live ? s.MW - col : 0;
        }
        const unsigned off = (row_off + (unsigned)(row * s.MW + col)) * 4u;
#pragma unroll
        for (int i = 0; i < 2; i++)
          raw[q][i] = __builtin_bit_cast(
              f32x4, __builtin_amdgcn_raw_buffer_load_b128(rows, (int)off + 16 * i, 0, 0));
        // (a row's last group that reaches past the image: element by element)
        if (__builtin_amdgcn_ballot_w64(off + 32u > rows_bytes) != 0) {
#pragma unroll
          for (int e = 0; e < 8; e++)
            raw[q][e >> 2][e & 3] = __builtin_bit_cast(
                float, __builtin_amdgcn_raw_buffer_load_b32(rows, (int)off + 4 * e, 0, 0));
        }
      }
      __syncthreads();  // everyone is done with the previous tile's taps
      // the taps: [tap][group][row of corners][16 floats]
      const int64_t q0 = (int64_t)first * s.K + k_base;
      const f32x4 *wt = reinterpret_cast<const f32x4 *>(s.wts) + q0 * 8;
      for (int i = t0; i < ktaps * (kTileGroups * NR * 4); i += kRunThreads) {
        const int w = i & 3, r = (i >> 2) % NR, gk = (i >> 2) / NR;
        const int gl = gk % kTileGroups, k = gk / kTileGroups;
        f32x4 x = wt[(unsigned)((min(gl, live - 1) * s.K + k) * 8 + r * 4 + w)];
        if (gl >= live) x = f32x4{0.f, 0.f, 0.f, 0.f};
        *reinterpret_cast<f32x4 *>(&lds.weights[gk * kRow + 16 * r + 4 * w]) = x;
      }
      if (t0 < ktaps * kTileGroups)
        reinterpret_cast<i32x4 *>(lds.desc)[t0] = reinterpret_cast<const i32x4 *>(
            s.desc)[q0 + min(t0 % kTileGroups, live - 1) * s.K + t0 / kTileGroups];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; e++) x[e] = raw[q][e >> 2][e & 3];
        if (__builtin_amdgcn_ballot_w64(n_live[q] < 8) != 0) {
#pragma unroll
          for (int e = 0; e < 8; e++) x[e] = e < n_live[q] ? x[e] : 0.f;
        }
        if (sums) {
          float sum = 0.f;
#pragma unroll
          for (int e = 0; e < 8; e++) sum += x[e];
          plain_sum += sum;
          // (added here and now: put off to the tile's end, the summands take 32 registers)
          asm volatile("" : "+v"(plain_sum));
        }
#pragma unroll
        for (int e = 0; e < 8; e++) x[e] *= sign * kSplitScale;
        split8(x, a[q]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __syncthreads();

    float v[NR][NV];
    i32x4 d;
    // the loads of the unit of tap k
    auto issue = [&](int k) __attribute__((always_inline)) {
      d = reinterpret_cast<const i32x4 *>(lds.desc)[k * kTileGroups + pg];
      if (__builtin_amdgcn_ballot_w64((d[3] & 3) != 0) == 0) {
#pragma unroll
        for (int r = 0; r < NR; r++) {
          const int off = d[r] + chan;
#pragma unroll
          for (int i = 0; i < NV / 4; i++) {
            const f32x4 q = __builtin_bit_cast(
                f32x4, __builtin_amdgcn_raw_buffer_load_b128(img, off + 16 * i, 0, 0));
#pragma unroll
            for (int e = 0; e < 4; e++) v[r][4 * i + e] = q[e];
          }
          if constexpr (NV % 4 == 1)
            v[r][NV - 1] = __builtin_bit_cast(
                float, __builtin_amdgcn_raw_buffer_load_b32(img, off + 4 * (NV - 1), 0, 0));
        }
      } else {
#pragma unroll
        for (int r = 0; r < NR; r++) {
          int off = d[r] + chan;
          asm volatile("" : "+v"(off));  // (one offset, not one per element, through the products)
#pragma unroll
          for (int e = 0; e < NV; e++)
            v[r][e] = __builtin_bit_cast(
                float, __builtin_amdgcn_raw_buffer_load_b32(
                           img, off + (e >= d[3] >> 2 ? d[2] : 0) + 4 * e, 0, 0));
        }
      }
    };
    // interpolates and splits what issue() fetched, into the samples' buffer
    auto stage = [&](int k) __attribute__((always_inline)) {
      const f32x4 *wp =
          reinterpret_cast<const f32x4 *>(&lds.weights[(k * kTileGroups + pg) * kRow]);
      float sv[8];
#pragma unroll
      for (int r = 0; r < NR; r++) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const f32x4 w = wp[4 * r + i];
#pragma unroll
          for (int h = 0; h < 2; h++) {
            const int e = 2 * i + h;
            const float c = v[r][ST * e];
            sv[e] = r == 0 ? w[2 * h] * c : __builtin_fmaf(w[2 * h], c, sv[e]);
            sv[e] = __builtin_fmaf(w[2 * h + 1], v[r][ST * e + 1], sv[e]);
          }
        }
      }
      if (d[3] & kCorners) {
        int p0 = pg;
        asm volatile("" : "+v"(p0));
        const int64_t q = ((int64_t)(first + min(p0, live - 1)) * s.K + k_base + k) * 16;
#pragma unroll
        for (int h = 0; h < 2 * NR; h++) {  // four pixels of a row of corners at a time
          const int r = h >> 1, e0 = 4 * (h & 1);
          uint2 o[4];
#pragma unroll
          for (int e = 0; e < 4; e++) o[e] = s.offs[q + 8 * r + e0 + e];
          float c0[4], c1[4];
#pragma unroll
          for (int e = 0; e < 4; e++) {
            c0[e] = __builtin_bit_cast(
                float, __builtin_amdgcn_raw_buffer_load_b32(img, (int)o[e].x + chan, 0, 0));
            c1[e] = __builtin_bit_cast(
                float, __builtin_amdgcn_raw_buffer_load_b32(img, (int)o[e].y + chan, 0, 0));
          }
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const f32x4 w = wp[4 * r + (e0 + e) / 2];
            const int i = 2 * (e & 1);
            sv[e0 + e] = r == 0 ? w[i] * c0[e] : __builtin_fmaf(w[i], c0[e], sv[e0 + e]);
            sv[e0 + e] = __builtin_fmaf(w[i + 1], c1[e], sv[e0 + e]);
          }
        }
      }
      bf16x8 p[3];
      split8(sv, p);
#pragma unroll
      for (int part = 0; part < 3; part++)
        lds.samples[buf][part][write_at] = __builtin_bit_cast(uint4, p[part]);
    };
    issue(0);
#pragma unroll
    for (int k = 0; k < kRunTaps; k++) {
      if (k < ktaps) {
        buf ^= 1;
        stage(k);
        __syncthreads();
        if (k + 1 < ktaps) issue(k + 1);
        // (a quarter of the pixels ahead of its products, and no more: the registers)
        bf16x8 bq[2][3];
        auto samples = [&](int q) __attribute__((always_inline)) {
#pragma unroll
          for (int part = 0; part < 3; part++)
            bq[q & 1][part] =
                __builtin_bit_cast(bf16x8, lds.samples[buf][part][q * 64 + read_at]);
        };
        samples(0);
        // (the leading parts' products apart from the others: see the head of the file)
        floatx4 p = floatx4{0.f, 0.f, 0.f, 0.f}, low = p;
        constexpr int pa[5] = {2, 0, 1, 1, 0}, pb[5] = {0, 2, 1, 0, 1};
#pragma unroll
        for (int q = 0; q < 4; q++) {
          if (q < 3) samples(q + 1);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < 5; i++)  // (smallest first)
            low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[q][pa[i]], bq[q & 1][pb[i]], low, 0, 0, 0);
          p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[q][0], bq[q & 1][0], p, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) acc[k][i] = __builtin_fmaf(sign, p[i] + low[i], acc[k][i]);
      }
    }
    first += kTileGroups;
    in += kTileGroups;
    if (first >= s.groups) {
      first = strip = in = 0;
      b++;
    }
    if (in >= strip_groups) {
      in -= strip_groups;
      strip++;
    }
  }

  if (sums) {
    float t = plain_sum;
    t += __shfl_xor(t, 16);
    t += __shfl_xor(t, 32);
    if (lq == 0 && a0 + l15 < s.A) s.sum_part[(int64_t)range * s.A + a0 + l15] = t;
  }
  const int A4 = (s.A + 3) & ~3;
  float *pr = s.part + (int64_t)range * A4 * s.G * s.K;
  bool bad = false;
#pragma unroll
  for (int k = 0; k < kRunTaps; k++) {
    const int g = g0 + l15, c = a0 + 4 * lq;
    if (k < ktaps && c < s.A && g < s.G) {
      floatx4 o = acc[k];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        if (c + i < s.A) bad |= !(__builtin_fabsf(o[i]) <= 3.402823466e+38f);
        o[i] *= kSplitUnscale;
      }
      *reinterpret_cast<floatx4 *>(&pr[((int64_t)(k_base + k) * s.G + g) * A4 + c]) = o;
    }
  }
  if (__builtin_amdgcn_ballot_w64(bad) != 0 && lane == 0) s.state[1] = 1;
}

template <int ST>
__global__ __launch_bounds__(kRunThreads, 3) void weight_grad_runs_kernel(const RunArgs s) {
  __shared__ __attribute__((aligned(16))) RunLds lds;
  __shared__ int totals[kRunThreads / 64][3];
  int no_runs = 0, elements = 0, bits = 0;
  for (int i = threadIdx.x; i < s.stat_words; i += kRunThreads) {
    const int2 of_block = s.stats[i];
    no_runs += of_block.x >> 2;
    bits |= of_block.x;
    elements += of_block.y;
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    no_runs += __shfl_xor(no_runs, m);
    bits |= __shfl_xor(bits, m);
    elements += __shfl_xor(elements, m);
  }
  if ((threadIdx.x & 63) == 0) {
    totals[threadIdx.x >> 6][0] = no_runs;
    totals[threadIdx.x >> 6][1] = bits;
    totals[threadIdx.x >> 6][2] = elements;
  }
  __syncthreads();
  no_runs = bits = elements = 0;
#pragma unroll
  for (int w = 0; w < kRunThreads / 64; w++) {
    no_runs += totals[w][0];
    bits |= totals[w][1];
    elements += totals[w][2];
  }
  const bool two_rows = (bits & 1) != 0;
  const bool runs = (int64_t)no_runs * (two_rows ? 448 : 160) +
                            (int64_t)elements * (two_rows ? 56 : 10) <= s.limit &&
                    (int64_t)no_runs * 8 <= (int64_t)s.groups * s.K;
  if (blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0 && threadIdx.x == 0) {
    s.state[0] = runs ? 1 : 0;
    s.state[2] = two_rows ? 4 : 0;
    s.state[3] = (bits & 2) != 0 && !two_rows ? 1 : 0;
  }
  if (!runs) return;
  if (two_rows)
    weight_grad_runs<2, ST>(s, lds);
  else
    weight_grad_runs<1, ST>(s, lds);
}

struct RunTables {
  RunDesc *desc;
  uint2 *offs;
  float2 *wts;
  int2 *stats;
  int *state;
  RunTables(const RunPlan &p, char *t) {
    desc = reinterpret_cast<RunDesc *>(t);
    wts = reinterpret_cast<float2 *>(t + p.desc_bytes);
    offs = reinterpret_cast<uint2 *>(t + p.desc_bytes + p.wts_bytes);
    stats = reinterpret_cast<int2 *>(t + p.desc_bytes + 2 * p.wts_bytes);
    state = reinterpret_cast<int *>(stats + kRunStatWords);
  }
};

}  // namespace

RunPlan run_plan(int64_t B, int64_t A, int64_t G, int64_t GW, int64_t MH, int64_t MW, int64_t K) {
  RunPlan p{};
  // taps of neighbouring pixels are taken to be as far apart as the images' widths say
  p.st = 2 * GW >= 3 * MW ? 2 : 1;
  p.cblocks = (int)((G + 15) / 16);
  p.ablocks = (int)((A + kRunA - 1) / kRunA);
  p.groups = (int)(MH * ((MW + 7) / 8));
  p.tiles_per_img = (p.groups + kTileGroups - 1) / kTileGroups;
  p.total_tiles = B * p.tiles_per_img;
  // Three workgroups fit a CU, and a tile takes a workgroup its time however few there are: 1.5 us a
  // tap and 1.9 for the rest (under taps of one row; a tenth more where they are two pixels apart, and
  // somewhat more where all three share the taps of one tile).  The taps are cut, to three at least, where
  // tiles then come out evenly: 16 x 64 -> 64 channels of 32 x 64, nine taps at a time 59 us, three 52;
  // 4 x 16 -> 32 of 128 x 256 64 and 53; 2 x 128 -> 128 of 45 x 90 in two parts 58 and 54.
  const int64_t per_tile = (int64_t)p.cblocks * p.ablocks, least = (K + kRunTaps - 1) / kRunTaps;
  constexpr int64_t kSlots = 768;
  for (int64_t passes = least; passes <= std::max(least, (K + 2) / 3); passes++) {
    const int64_t ranges = std::min(std::max<int64_t>(1, kSlots / (per_tile * passes)), p.total_tiles);
    const int64_t turns = (ranges * per_tile * passes + kSlots - 1) / kSlots;
    const double us = (double)(turns * ((p.total_tiles + ranges - 1) / ranges)) *
                      (1.5 * (double)((K + passes - 1) / passes) + 1.9) *
                      (p.st == 2 ? 1.1 : 1.0) * (1.0 + 0.08 * (double)(passes - least));
    if (p.passes == 0 || us < p.us) {
      p.us = us;
      p.passes = (int)passes;
      p.ranges = (int)ranges;
    }
  }
  const int64_t entries = (int64_t)p.groups * K * 8;
  p.stat_words = (int)std::min<int64_t>(kRunStatWords, (entries + 255) / 256);
  p.desc_bytes = align256((size_t)p.groups * K * sizeof(RunDesc));
  p.wts_bytes = align256((size_t)p.groups * K * 128);
  return p;
}
// The operands' images are addressed as buffers of less than 2 GiB (the sign bit of an offset and
// its two lowest bits are free), the table's entries with 32 bits.
bool runs_apply(int64_t B, int64_t A, int64_t G, int64_t GH, int64_t GW, int64_t MH, int64_t MW,
                int64_t K, int64_t P) {
  return P <= 1 && GH > 1 && G * GH * GW < (1LL << 29) && A * MH * MW < (1LL << 29) &&
         MH * ((MW + 7) / 8) * K < (1LL << 27) && B * MH * MW < (1LL << 33) && A <= 64 * 65535;
}
// desc, weights, corner offsets, statistics and the state words
size_t run_table_bytes(const RunPlan &p) {
  return p.desc_bytes + 2 * p.wts_bytes + align256(kRunStatWords * sizeof(int2)) + align256(kRunStateWords * 4);
}

void set_run_limit(RunPlan &p, int64_t K, double general_us) {
  const double gain = general_us / p.us - 1.0;
  p.limit = gain < 0 ? -1 : (int64_t)(gain * 16 * (double)p.groups * (double)K);
}

int *run_state(const RunPlan &p, char *tables) { return RunTables(p, tables).state; }

int resolve_runs(const RunPlan &p, char *tables, const float *map, const float *iw, int64_t GH,
                 int64_t GW, int64_t MH, int64_t MW, int64_t K, int ncorn, int wrap, int weighted,
                 const TapTable &taps, hipStream_t stream) {
  const RunTables t(p, tables);
#define MCX_RESOLVE(NCORN, ST)                                                                     \
  hipLaunchKernelGGL((resolve_runs_kernel<NCORN, ST>), dim3((unsigned)p.stat_words), dim3(256), 0, \
                     stream, map, iw, t.desc, t.wts, t.offs, t.stats, t.state, (int)GH, (int)GW,   \
                     (int)MH, (int)MW, (int)K, wrap, weighted, p.limit >= 0 ? 1 : 0, taps)
  if (ncorn == 1) {
    if (p.st == 2) { MCX_RESOLVE(1, 2); } else { MCX_RESOLVE(1, 1); }
  } else {
    if (p.st == 2) { MCX_RESOLVE(4, 2); } else { MCX_RESOLVE(4, 1); }
  }
#undef MCX_RESOLVE
  MCX_HIP_CHECK_LAUNCH();
  return 0;
}

int weight_grad_by_runs(const RunPlan &p, char *tables, const float *plain, const float *gath,
                        float *part, float *sum_part, int64_t A, int64_t G, int64_t GH, int64_t GW,
                        int64_t MH, int64_t MW, int64_t K, hipStream_t stream) {
  const RunTables t(p, tables);
  RunArgs a{};
  a.plain = plain; a.gath = gath; a.part = part; a.sum_part = sum_part;
  a.desc = t.desc; a.wts = reinterpret_cast<const float *>(t.wts); a.offs = t.offs;
  a.stats = t.stats; a.state = t.state;
  a.A = (int)A; a.G = (int)G; a.GH = (int)GH; a.GW = (int)GW; a.MH = (int)MH; a.MW = (int)MW;
  a.K = (int)K; a.stat_words = p.stat_words; a.groups = p.groups;
  a.tiles_per_img = p.tiles_per_img; a.total_tiles = (int)p.total_tiles; a.ranges = p.ranges;
  a.cblocks = p.cblocks; a.limit = p.limit;
  // (where the work is the general kernel's in any case, one workgroup says so)
  const dim3 grid = p.limit < 0 ? dim3(1)
                                : dim3((unsigned)(p.ranges * p.cblocks), (unsigned)p.ablocks,
                                       (unsigned)p.passes);
  if (p.st == 2)
    hipLaunchKernelGGL(weight_grad_runs_kernel<2>, grid, dim3(kRunThreads), 0, stream, a);
  else
    hipLaunchKernelGGL(weight_grad_runs_kernel<1>, grid, dim3(kRunThreads), 0, stream, a);
  MCX_HIP_CHECK_LAUNCH();
  return 0;
}

}  // namespace mcx
