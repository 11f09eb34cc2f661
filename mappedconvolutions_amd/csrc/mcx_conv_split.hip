// fp32 gather-product on the bf16 matrix instructions, without giving up fp32: every operand is
// split exactly into three bf16 parts (8 + 8 + 8 significant bits, round to nearest each, the
// remainders exact; the decomposition into leading part and remainders is Dekker's, Numerische
// Mathematik 18, 1971), and of the nine partial products six are summed in fp32 by the matrix unit.
// Each of the other three is at most 2^-25 of the product, all of them 2^-24 (half a unit in the
// last place of fp32; their root mean square over random operands is about 2^-26.5), and a matrix
// instruction adds 16 products per rounding of its sum where the fp32 one adds 2.  Distance from the
// 64-bit result over that of the fp32 instructions, in 2-norm, at 6 to 128 channels and 1 to 49 taps:
// normal and positive operands 0.45 to 1.05, above one by more than 0.01 only over nine, ten, 17 and
// 18 channels (the partly filled chunk rounds like a full one).  Samples half of which are zero, as
// behind a ReLU, favour the fp32 instructions, which round nothing where both products are zero:
// 0.6 to 1.1 where taps interpolate, 0.6 to 1.3 where they read whole pixels (128 channels, nine
// taps: 5.0e-7 against 4.4e-7, with dense samples 5.2e-7 against 6.1e-7).  A second set of
// accumulators for the five small products would round the large sums once a unit instead of six
// times; its 32 registers are not there (144 spilled at three waves per SIMD).
// v_mfma_f32_32x32x16_bf16 does sixteen times the work of v_mfma_f32_32x32x2_f32 per clock, so six
// of them cost 384 clocks a unit (one tap x 16 channels x 32 pixels x 64 outputs) where the fp32
// form costs 1024.
//   * Interpolation weights and product weights are scaled by 2^24 before they are split, the sums by
//     2^-48 at the end: exact, and the lowest bit of the smallest fp32 number (2^-149) is then a
//     normal bf16.  (Without it parts below 2^-133 are lost, and with them bits of operands smaller
//     than 2^-110: 216 products of 2^-124 and 2^30 came out 4e-4 off in 2-norm, now 2.4e-7.)
//   * What the split cannot represent - an infinity or NaN among the operands, whose
//     remainders are NaN, samples or weights from 2^104 up, or sums from 2^80 up - always ends as a
//     value that is not finite.  A wave that sees one sets its tile's flag, and the fp32 kernel,
//     whose launch follows every launch of these with the same tiles, recomputes the tiles that
//     have it (in its general form: a flagged tile costs both kernels).  8 x 64 channels of
//     256 x 512 -> 64 forward: no NaN 599 us, one element 607, a quarter of the rows 766, all
//     1285 (the fp32 kernel alone, in its two-pair form: 715 to 730; one flag for the whole
//     product: 1300 in every case with a NaN).  2 x 24 -> 40 of 125 x 250, where the fp32 kernel's
//     workgroups all run at once: 35, 59, 72, 72 (47).
//   * In the planar kernel a lane gathers, interpolates and splits exactly the elements its matrix
//     B operand holds (lane (l31, lhi): channels lhi * 8 .. + 7 of pixel l31 of the wave), so only
//     the weights, pre-split by the packing launch, pass through LDS.
// Bound: the matrix instructions (384 clocks a unit) and the vector instructions around them
// (some 60 x 4), which all but take turns, and what three waves per SIMD leave exposed of the
// loads' latency.  Measured in one run each, fp32 instructions -> these: 8 x 64 channels of
// 256 x 512 -> 64, nine taps: forward 798 -> 597 us, input gradient 768 -> 597 us (547 to 600 for
// the product over the cards seen); 4 x 64 -> 32 channels onto 256 x 512 (transposed) 379 -> 269 us;
// mesh of 40 962 vertices, 4 x 64 -> 128 channels, four points a tap: forward 411 -> 292 us, input
// gradient (both levels in one pass) 952 -> 509 us.
#include "mcx_conv_split.h"
#include "mcx_mfma_common.h"

namespace mcx {
namespace {

constexpr int kThreads = 256;
// Channels between the two halves of chunk c of a planar source.
__device__ inline int split_upper_half(int c, int G) {
  const int rem = G - c * 16;
  return rem >= 16 ? 8 : rem > 8 ? rem - 8 : 0;
}

// The weights of a unit through LDS: [part][kg][output][8 channels], double buffered.  NB: blocks of
// 32 outputs a workgroup computes.
template <int NB>
struct SplitWeights {
  static constexpr int kPieces = 3 * 2 * 32 * NB;                         // of 16 bytes
  static constexpr int kPer = (kPieces + kThreads - 1) / kThreads;        // per thread
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  unsigned off[kPer];
  int tid;
  bool last_round;  // (wave-uniform) this wave stores a piece in the last, partial round
  __device__ inline void init(int t, int Opad, int o0) {
    tid = t;
    last_round = __builtin_amdgcn_readfirstlane(t >> 6) * 64 + (kPer - 1) * kThreads < kPieces;
#pragma unroll
    for (int j = 0; j < kPer; j++) {
      const int i = min(t + j * kThreads, kPieces - 1);  // (a last, partial round is not stored)
      off[j] = (unsigned)((i / (32 * NB)) * Opad + o0 + i % (32 * NB)) * 16u;
    }
  }
  __device__ inline void load(plane_buf_t r, unsigned unit_off, u32x4 *v) const {
#pragma unroll
    for (int j = 0; j < kPer; j++)
      v[j] = __builtin_bit_cast(
          u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off[j], (int)unit_off, 0));
  }
  __device__ inline void store(uint4 *lds, const u32x4 *v) const {
#pragma unroll
    for (int j = 0; j < kPer; j++)
      if ((j + 1) * kThreads <= kPieces || last_round)
        *reinterpret_cast<u32x4 *>(lds + tid + j * kThreads) = v[j];
  }
};

template <int NB>
__device__ inline void read_split_weights(const uint4 *lds, int l31, int lhi, bf16x8 (*a)[3]) {
#pragma unroll
  for (int m = 0; m < NB; m++)
#pragma unroll
    for (int part = 0; part < 3; part++)
      a[m][part] =
          __builtin_bit_cast(bf16x8, lds[(part * 2 + lhi) * (32 * NB) + 32 * m + l31]);
}
template <int NB>
__device__ inline void split_products(const bf16x8 (*a)[3], const bf16x8 *b, floatx16 *acc) {
  // (smallest first; the chains of the output blocks are independent)
  constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
  for (int t = 0; t < 6; t++)
#pragma unroll
    for (int m = 0; m < NB; m++)
      acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[m][pa[t]], b[pb[t]], acc[m], 0, 0, 0);
}

// The workgroup's biases, in LDS before its first barrier.
template <int NB>
__device__ inline void split_bias(const SplitArgs &s, float *lds, int o0) {
  if (threadIdx.x < 32 * NB)
    lds[threadIdx.x] =
        s.bias && o0 + (int)threadIdx.x < s.O ? s.bias[o0 + (int)threadIdx.x] : 0.f;
}

// Bias, addend and stores of a lane's pixel; flags a tile with a result that is not finite.  (No
// load after the first store: a wait for it would be one for the stores before it as well, 500 clocks an
// output, a quarter of the kernel's time at nine taps of 64 channels.)
template <int NB, int AT_ONCE>
__device__ inline void split_epilogue(const SplitArgs &s, floatx16 *acc, const float *bias, int tile,
                                      int b, int o0, int ei, int ej, int lhi) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  const int64_t N = (int64_t)s.OH * s.OW;
  bool bad = false;
  if (ei < s.OH && ej < s.OW) {
    const int64_t n = (int64_t)ei * s.OW + ej;
    float *yb = s.y + ((int64_t)b * s.O + o0 + lhi * 4) * N + n;
#pragma unroll
    for (int m = 0; m < NB; m++)
#pragma unroll
      for (int i = 0; i < 16; i++) {
        bad |= !(__builtin_fabsf(acc[m][i]) <= 3.402823466e+38f);
        acc[m][i] = __builtin_fmaf(acc[m][i], kSplitUnscale,
                                   bias[32 * m + (i >> 2) * 8 + lhi * 4 + (i & 3)]);
      }
    if (s.addend && s.gate && s.gate[1] > 0) {
      const float *ab = s.addend + ((int64_t)b * N + n) * s.Opad + o0 + lhi * 4;
      auto add4 = [&](int m, int g, f32x4 v) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; i++) acc[m][4 * g + i] += v[i];
      };
      // (Those of outputs that there are.  Of AT_ONCE blocks they are read before the first is used: 4 x 64 -> 128 channels over
      // 40 962 vertices, input gradient 649 us with the test before each use, so 645; of more blocks, they spill.)
#pragma unroll
      for (int m0 = 0; m0 < NB; m0 += AT_ONCE) {
        f32x4 more[AT_ONCE][4];
#pragma unroll
        for (int m = m0; m < m0 + AT_ONCE && m < NB; m++)
#pragma unroll
          for (int g = 0; g < 4; g++)
            if (o0 + 32 * m + 8 * g < s.O) {
              more[m - m0][g] = *reinterpret_cast<const f32x4 *>(ab + 32 * m + 8 * g);
              if constexpr (AT_ONCE == 1) add4(m, g, more[0][g]);
            }
        if constexpr (AT_ONCE > 1) {
#pragma unroll
          for (int m = m0; m < m0 + AT_ONCE && m < NB; m++)
#pragma unroll
            for (int g = 0; g < 4; g++)
              if (o0 + 32 * m + 8 * g < s.O) add4(m, g, more[m - m0][g]);
          if (NB > AT_ONCE) __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    if (o0 + 32 * NB <= s.O) {
#pragma unroll
      for (int m = 0; m < NB; m++)
#pragma unroll
        for (int i = 0; i < 16; i++) yb[(int64_t)(32 * m + (i >> 2) * 8 + (i & 3)) * N] = acc[m][i];
    } else {
#pragma unroll
      for (int m = 0; m < NB; m++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
          const int o = 32 * m + (i >> 2) * 8 + (i & 3);
          if (o0 + lhi * 4 + o < s.O) yb[(int64_t)o * N] = acc[m][i];
        }
    }
  }
  if (__builtin_amdgcn_ballot_w64(bad) != 0 && (threadIdx.x & 63) == 0)
    s.nonfinite[tile] = 1;  // (every writer stores the same value)
}

// Planar images.  NE: (offset, weight) entries per tap, 1 or 4; with 4, tiles none of whose taps
// uses a later entry run with the leading two.  NB: blocks of 32 outputs.
//
// The taps go in groups.  In memory (in_memory): two entries of a tap that are neighbours in memory for
// every pixel of the tile (the corners of a row, two contributions of a transposed map) are
// fetched with one 8-byte load; the texture path takes 16 to 25 clocks for a wave's load whatever its
// width, and 16 single loads a unit would cost it as much as the fp32 matrix instructions did.
//
// WINDOW: with four entries a tap that is still 16 loads a unit, and one block of outputs has few
// matrix instructions to hide even eight.  Where the entries of a group's 128 pixels lie in a small box of
// the source - those of every kernel over an image do, but next to the poles and at random maps - the
// box goes into LDS, 16 channels at a time, four channels of a pixel in 16 bytes (a wave copies four of the
// channels with 16-byte loads, the next chunk's on their way while this one's are multiplied), and an
// entry is two 16-byte reads of LDS.  A group whose box is too large is tried again in threes of taps, then
// goes the way through memory.
constexpr int kMemCache = 12;            // entries a pixel of a group in memory, offsets of 32 bits
constexpr int kWinCache = 12;            // of a group in a window, offsets of 16 bits
constexpr int kTapBytes = kMemCache * kTilePx * 8;
constexpr int kWinPx = 256;              // pixels of a window

// Where pixel i of a window lies: fours of pixels that eight lanes store together are on different banks.
__device__ inline int window_place(int i) { return i ^ ((i >> 3) & 3); }

// q / d for 0 <= q < 2^31, 0 < d, where the quotient is below 2^16: the estimate is off by one at most.
__device__ inline int quotient(int q, int d, float inv) {
  int r = (int)((float)q * inv);
  r -= r * d > q ? 1 : 0;
  r += (r + 1) * d <= q ? 1 : 0;
  return r;
}

template <int NE, int NB, bool WINDOW>  // (windows for four entries only)
__global__ __launch_bounds__(kThreads, NB > 2 ? 2 : !WINDOW && (NE == 1 || NB == 1) ? 4 : 3) void
gather_product_split_kernel(const SplitArgs s) {
  __shared__ __attribute__((aligned(16))) uint4 Wt[2][SplitWeights<NB>::kPieces];
  __shared__ __attribute__((aligned(16))) float4 Win[4][kWinPx];  // [channel / 4][pixel]
  __shared__ __attribute__((aligned(16))) char TapMem[kTapBytes];
  __shared__ __attribute__((aligned(16))) int box[6][4];  // largest values by wave
  __shared__ __attribute__((aligned(16))) float Bias[32 * NB];
  __shared__ int unpaired;
  static_assert(!WINDOW || NE == 4, "four entries");
  if (s.gate && ((*s.gate == 0) != (s.run_if_zero != 0))) return;
  const int tid = threadIdx.x;
  const int tile = xcd_contiguous_tile(blockIdx.x, gridDim.x);
  const int b = tile / s.tiles_per_img;
  const int t_in = tile - b * s.tiles_per_img;
  const int tile_y = t_in / s.tiles_x, tile_x = t_in - tile_y * s.tiles_x;
  const int tw_mask = (1 << s.tw_shift) - 1, th = kTilePx >> s.tw_shift;
  bool leading = false;
  if (NE == 4 && s.pair_mask) {
    leading = !later_pairs_in_use(s.pair_mask, s.mask_words);
    if (!leading && s.row_mask) {
      int any = 0;
      for (int r = tile_y * th; r < min(tile_y * th + th, s.OH); r++) any |= s.row_mask[r];
      leading = any == 0;
    }
  }
  const int o0 = blockIdx.y * (32 * NB);
  const int N = s.OH * s.OW;
  const unsigned plane_bytes = (unsigned)s.SH * (unsigned)s.SW * 4u;
  const int chunks = s.Gpad / kGC;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l31 = lane & 31, lhi = lane >> 5;
  const int pe = wave * 32 + l31;
  const auto img = plane_buf(s.src + (int64_t)b * s.G * s.SH * s.SW, (unsigned)s.G * plane_bytes);
  const auto wbuf = plane_buf(s.w, (unsigned)s.K * chunks * 6u * s.Opad * 16u);
  const unsigned w_unit = 6u * s.Opad * 16u;

  // resolving role: pixel p of the tile, every other tap
  const int p = tid & (kTilePx - 1), half = tid >> 7;
  const int gi = tile_y * th + (p >> s.tw_shift), gj = (tile_x << s.tw_shift) + (p & tw_mask);
  const bool live = gi < s.OH && gj < s.OW;
  const int64_t n_g = live ? (int64_t)gi * s.OW + gj : 0;

  floatx16 acc[NB];
#pragma unroll
  for (int m = 0; m < NB; m++)
#pragma unroll
    for (int i = 0; i < 16; i++) acc[m][i] = 0.f;
  SplitWeights<NB> wts;
  wts.init(tid, s.Opad, o0);
  split_bias<NB>(s, Bias, o0);
  int buf = 0;

  // ---- a group in a window: rows of `cols` pixels, a multiple of four, from (row0, col0) on, columns
  // cyclic, fours of them next to each other in the source ----
  uint16_t *const win_off = reinterpret_cast<uint16_t *>(TapMem);  // (place in the window)
  float *const win_wt = reinterpret_cast<float *>(TapMem + kWinCache * kTilePx * 2);
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  auto units_in_window = [&](int k0, int kn, auto na_tag, int row0, int col0, int cols,
                             int rows) __attribute__((always_inline)) {
    constexpr int NA = decltype(na_tag)::value;
    // the four pixels that this lane copies, of this wave's four channels of every chunk
    const int fours = cols >> 2;
    const int r = quotient(lane, fours, 1.f / (float)fours);
    int x4 = col0 + 4 * (lane - r * fours);
    x4 -= x4 >= s.SW ? s.SW : 0;
    const unsigned from =
        lane < rows * fours ? (unsigned)((row0 + r) * s.SW + x4) * 4u : kOobOffset;
    const unsigned to = (unsigned)(wave * kWinPx + window_place(4 * lane)) * 16u;  // (in Win)
    f32x4 held[4];
    // (the last chunk, which may hold few channels, comes first: its products round small sums)
    auto fetch = [&](int c) __attribute__((always_inline)) {
      const int cc = max(chunks - 1 - c, 0), last = s.G - 1 - cc * kGC;
      const int first = cc * kGC + (wave >> 1 ? split_upper_half(cc, s.G) : 0);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const unsigned so = (unsigned)(first + min((wave & 1) * 4 + i, last)) * plane_bytes;
        held[i] = __builtin_bit_cast(
            f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                       img, (int)from, (int)__builtin_amdgcn_readfirstlane(so), 0));
      }
    };
    auto fill = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < 4; j++)
        *reinterpret_cast<f32x4 *>(reinterpret_cast<char *>(&Win[0][0]) + (to ^ (j * 16u))) =
            f32x4{held[0][j], held[1][j], held[2][j], held[3][j]};
    };
    f32x4 v[2][NA];
    float wgt[NA];
    typename SplitWeights<NB>::u32x4 wv[SplitWeights<NB>::kPer];
    auto load_weights = [&](int kl, int c) __attribute__((always_inline)) {
      const int unit = (k0 + kl) * chunks + max(chunks - 1 - c, 0);
      wts.load(wbuf, __builtin_amdgcn_readfirstlane((unsigned)unit * w_unit), wv);
    };
    auto read = [&](int kl) __attribute__((always_inline)) {
      unsigned at[NA];
#pragma unroll
      for (int i = 0; i < NA; i++) at[i] = win_off[(kl * kTilePx + pe) * NA + i] * 16u;
#pragma unroll
      for (int i = 0; i < NA; i++)
#pragma unroll
        for (int q = 0; q < 2; q++)
          v[q][i] = *reinterpret_cast<const f32x4 *>(reinterpret_cast<const char *>(&Win[q][0]) +
                                                     at[i] + (unsigned)lhi * (2u * kWinPx * 16u));
#pragma unroll
      for (int i = 0; i < NA; i++) wgt[i] = win_wt[(kl * kTilePx + pe) * NA + i];
    };
    // One unit: its samples split, the next one's weights and samples on their way, the products.  The
    // next chunk's pixels (FIRST: after the loads of the weights that the next unit waits for) have two units' time.
    auto unit = [&](int kl, int c, auto first_tag) __attribute__((always_inline)) {
      constexpr bool FIRST = decltype(first_tag)::value;
      const bool turn = kl + 1 == kn;
      const int next = turn ? 0 : kl + 1;  // (past the last unit it is read again)
      bf16x8 bq[3];
      float sv[8];
#pragma unroll
      for (int ch = 0; ch < 8; ch++) {
        sv[ch] = wgt[0] * v[ch >> 2][0][ch & 3];
#pragma unroll
        for (int i = 1; i < NA; i++) sv[ch] = __builtin_fmaf(wgt[i], v[ch >> 2][i][ch & 3], sv[ch]);
      }
      split8(sv, bq);
      wts.store(Wt[buf], wv);
      load_weights(next, turn ? c + 1 : c);
      if constexpr (FIRST) fetch(c + 1);
      __syncthreads();  // the weights are there, and every wave has read this unit's samples
      if (turn && c + 1 < chunks) {
        fill();
        __syncthreads();
      }
      read(next);
      bf16x8 a[NB][3];
      read_split_weights<NB>(Wt[buf], l31, lhi, a);
      split_products<NB>(a, bq, acc);
      buf ^= 1;
    };
    fetch(0);
    load_weights(0, 0);
    fill();
    __syncthreads();
    read(0);
    for (int c = 0; c < chunks; c++) {
      unit(0, c, std::true_type());
      if (kn > 1) {
        unit(1, c, std::false_type());
        for (int kl = 2; kl < kn; kl++) unit(kl, c, std::false_type());
      }
    }
  };
  // Resolves taps k0 .. k0 + kn - 1 and multiplies them if they fit a window; returns 1 then, else at
  // least 2: one more than the windows that their box would fill.
  const float inv_sw = 1.f / (float)s.SW;
  auto in_window = [&](int k0, int kn, auto na_tag) __attribute__((always_inline)) {
    constexpr int NA = decltype(na_tag)::value;
    constexpr int kMine = NA == 4 ? 2 : 3;  // of three or six taps
    // (every load is issued before the first is used; past the group's end its last tap is read)
    float2 raw[kMine][NA];
    float raw_w[kMine];
#pragma unroll
    for (int j = 0; j < kMine; j++) {
      const int k = k0 + min(half + 2 * j, kn - 1);
      raw_w[j] = 1.f;
      if (s.packed) {
        // pre-resolved entries [tap][slot][pixel]: (pixel index as bits, weight)
#pragma unroll
        for (int i = 0; i < NA; i++)
          raw[j][i] = reinterpret_cast<const float2 *>(s.map)[((int64_t)k * 4 + i) * N + n_g];
      } else {
        const int64_t e = n_g * s.K + k;
        raw[j][0] = reinterpret_cast<const float2 *>(s.map)[e];
        if (s.weighted) raw_w[j] = s.iw[e];
      }
    }
    unsigned cell[kMine][NA];  // row << 16 | column
    // largest row, column, column with the left half of the image moved to the right of the other
    // (a seam), and the same of their negatives
    int most[6];
#pragma unroll
    for (int i = 0; i < 6; i++) most[i] = -0x7fffffff;
#pragma unroll
    for (int j = 0; j < kMine; j++) {
      const int kl = half + 2 * j;
      if (kl < kn) {
        float wt[NA];
        int y[NA], x[NA];
        if (s.packed) {
#pragma unroll
          for (int i = 0; i < NA; i++) {
            const float2 q = raw[j][i];
            wt[i] = live ? q.y * kSplitScale : 0.f;
            const int e = wt[i] != 0.f ? __builtin_bit_cast(int, q.x) : 0;
            y[i] = quotient(e, s.SW, inv_sw);
            x[i] = e - y[i] * s.SW;
          }
        } else {
          CoordTap<4> t;
          resolve_coords<4>(raw[j][0].x, raw[j][0].y, s.SH, s.SW, s.wrap != 0,
                            live ? raw_w[j] * kSplitScale : 0.f, t);
#pragma unroll
          for (int i = 0; i < NA; i++) {
            wt[i] = (t.ok >> i) & 1u ? t.wt[i] : 0.f;
            y[i] = t.yy[i];
            x[i] = t.xx[i];
          }
        }
#pragma unroll
        for (int i = 0; i < NA; i++) {
          const bool use = wt[i] != 0.f;
          const int turned = x[i] < s.SW / 2 ? x[i] + s.SW : x[i];
          most[0] = max(most[0], use ? y[i] : -0x7fffffff);
          most[1] = max(most[1], use ? -y[i] : -0x7fffffff);
          most[2] = max(most[2], use ? x[i] : -0x7fffffff);
          most[3] = max(most[3], use ? -x[i] : -0x7fffffff);
          most[4] = max(most[4], use ? turned : -0x7fffffff);
          most[5] = max(most[5], use ? -turned : -0x7fffffff);
          cell[j][i] = use ? (unsigned)y[i] << 16 | (unsigned)x[i] : 0xffffffffu;
          win_wt[(kl * kTilePx + p) * NA + i] = wt[i];
        }
      }
    }
#pragma unroll
    for (int i = 0; i < 6; i++) {
      most[i] = wave_max(most[i]);
      if (lane == 0) box[i][wave] = most[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 6; i++)
      most[i] = __builtin_amdgcn_readfirstlane(
          max(max(box[i][0], box[i][1]), max(box[i][2], box[i][3])));
    const bool none = most[0] < 0;  // no entry in use: pixel 0 stands for all
    const int plain = most[2] + most[3], turned = most[4] + most[5];
    const int rows = none ? 1 : most[0] + most[1] + 1;
    const int row0 = none ? 0 : -most[1];
    int col0 = none ? 0 : plain <= turned ? -most[3] : -most[5];
    col0 -= col0 >= s.SW ? s.SW : 0;
    int cols = none ? 1 : min(plain, turned) + 1;
    // fours of columns, none of which has the seam inside
    const bool seam = col0 + cols > s.SW;
    if (seam) {
      const int back = (col0 - s.SW) & 3;
      cols += back;
      col0 -= back;
    }
    cols = (cols + 3) & ~3;
    if (!seam && col0 + cols > s.SW) col0 = s.SW - cols;
    if (cols > kWinPx || rows > kWinPx || rows * cols > kWinPx || cols > s.SW || col0 < 0)
      return max(2, 1 + (int)(min((unsigned)rows, 0xffffu) * min((unsigned)cols, 0xffffu) / kWinPx));
#pragma unroll
    for (int j = 0; j < kMine; j++) {
      const int kl = half + 2 * j;
      if (kl < kn) {
#pragma unroll
        for (int i = 0; i < NA; i++) {
          int x = (int)(cell[j][i] & 0xffffu) - col0;
          x += x < 0 ? s.SW : 0;
          const int at = ((int)(cell[j][i] >> 16) - row0) * cols + x;
          win_off[(kl * kTilePx + p) * NA + i] =
              (uint16_t)(cell[j][i] == 0xffffffffu ? 0 : window_place(at));
        }
      }
    }
    units_in_window(k0, kn, na_tag, row0, col0, cols, rows);
    return 1;
  };

  // ---- a group in memory ----
  // (Arrays of their own where four entries have no window to share the memory with: the compiler then moves reads of one
  // past writes of the other.  Input gradient of 3 x 139 -> 61 channels of 44 x 88 78 us in one, 73; 1 x 40 -> 100 of 60 x 120,
  // 5 x 5, 210 and 195.)
  constexpr bool kOwn = !WINDOW && NE == 4;
  __shared__ __attribute__((aligned(16))) unsigned OwnOff[kOwn ? kMemCache * kTilePx : 1];
  __shared__ __attribute__((aligned(16))) float OwnWt[kOwn ? kMemCache * kTilePx : 1];
  unsigned *const TapOff = kOwn ? OwnOff : reinterpret_cast<unsigned *>(TapMem);
  float *const TapWt = kOwn ? OwnWt : reinterpret_cast<float *>(TapMem + kMemCache * kTilePx * 4);
  // its units: chunk-major, the tap fastest (a chunk's source rows stay in cache)
  auto units_of = [&](int k0, int kn, auto na_tag, auto paired_tag) __attribute__((always_inline)) {
    constexpr int NA = decltype(na_tag)::value;
    constexpr bool PAIRED = decltype(paired_tag)::value;
    constexpr int NL = PAIRED ? NA / 2 : NA;  // loads per channel
    // Units whose loads are in flight.  With one, every unit waits out what its 12 matrix
    // instructions do not cover of a load's latency: 657 us a product at 8 x 64 channels of
    // 256 x 512 -> 64, 9 taps.  (Two of four single loads a channel do not fit the registers.)
    constexpr int kDepth = NL * (PAIRED ? 2 : 1) <= 2 ? 2 : 1;
    const int units = chunks * kn;
    float v[kDepth][8][NA];
    float wgt[kDepth][NA];
    typename SplitWeights<NB>::u32x4 wv[kDepth][SplitWeights<NB>::kPer];
    int kl = 0, c = 0;  // the unit whose loads are issued next
    // (issued unconditionally, past the last unit too, where it reads the last chunk again: a
    // load behind a branch would make every wait a full one)
    auto issue = [&](int d) __attribute__((always_inline)) {
      const int cc = min(c, chunks - 1);
      unsigned off[NL];
      const unsigned upper =
          (unsigned)__builtin_amdgcn_readfirstlane((int)((unsigned)split_upper_half(cc, s.G) *
                                                         plane_bytes));
#pragma unroll
      for (int i = 0; i < NL; i++)
        off[i] = TapOff[(kl * kTilePx + pe) * NA + (PAIRED ? 2 * i : i)] + (lhi ? upper : 0u);
#pragma unroll
      for (int i = 0; i < NA; i++) wgt[d][i] = TapWt[(kl * kTilePx + pe) * NA + i];
      wts.load(wbuf, __builtin_amdgcn_readfirstlane((unsigned)((k0 + kl) * chunks + cc) * w_unit),
               wv[d]);
      const int last = s.G - 1 - cc * kGC;  // (channels past the last one: weights of zero)
#pragma unroll
      for (int ch = 0; ch < 8; ch++) {
        const unsigned so = __builtin_amdgcn_readfirstlane((unsigned)(cc * kGC + min(ch, last)) *
                                                           plane_bytes);
#pragma unroll
        for (int i = 0; i < NL; i++) {
          if constexpr (PAIRED) {
            const float_pair q = __builtin_bit_cast(
                float_pair, __builtin_amdgcn_raw_buffer_load_b64(img, (int)off[i], (int)so, 0));
            v[d][ch][2 * i] = q.x;
            v[d][ch][2 * i + 1] = q.y;
          } else {
            v[d][ch][i] = __builtin_bit_cast(
                float, __builtin_amdgcn_raw_buffer_load_b32(img, (int)off[i], (int)so, 0));
          }
        }
      }
      if (++kl == kn) {
        kl = 0;
        ++c;
      }
    };
    bf16x8 bq[3];
    auto stage = [&](int d) __attribute__((always_inline)) {
      float sv[8];
#pragma unroll
      for (int ch = 0; ch < 8; ch++) {
        sv[ch] = wgt[d][0] * v[d][ch][0];
#pragma unroll
        for (int i = 1; i < NA; i++) sv[ch] = __builtin_fmaf(wgt[d][i], v[d][ch][i], sv[ch]);
      }
      split8(sv, bq);
      wts.store(Wt[buf], wv[d]);
    };
#pragma unroll
    for (int d = 0; d < kDepth; d++) issue(d);
    int u = 0;
    for (; u + kDepth <= units; u += kDepth) {
#pragma unroll
      for (int d = 0; d < kDepth; d++) {
        stage(d);
        __syncthreads();
        issue(d);
        {
          bf16x8 a[NB][3];
          read_split_weights<NB>(Wt[buf], l31, lhi, a);
          split_products<NB>(a, bq, acc);
        }
        buf ^= 1;
      }
    }
#pragma unroll
    for (int d = 0; d < kDepth - 1; d++) {
      if (u + d < units) {
        stage(d);
        __syncthreads();
        {
          bf16x8 a[NB][3];
          read_split_weights<NB>(Wt[buf], l31, lhi, a);
          split_products<NB>(a, bq, acc);
        }
        buf ^= 1;
      }
    }
  };
  auto in_memory = [&](int from, int count, auto na_tag) __attribute__((always_inline)) {
    constexpr int NA = decltype(na_tag)::value;
    constexpr int TG = (NE == 1 ? kMemCache / 2 : kMemCache) / NA;
    for (int k0 = from; k0 < from + count; k0 += TG) {
      const int kn = min(TG, from + count - k0);
      __syncthreads();  // the previous group's units are done with the cache
      if (tid == 0) unpaired = NA == 1 ? 1 : 0;
      __syncthreads();
      for (int kl = half; kl < kn; kl += 2) {
        unsigned off[4];
        float wt[4];
        if (s.packed) {
          // pre-resolved entries [tap][slot][pixel]: (pixel index as bits, weight)
#pragma unroll
          for (int i = 0; i < NA; i++) {
            const float2 q =
                reinterpret_cast<const float2 *>(s.map)[((int64_t)(k0 + kl) * 4 + i) * N + n_g];
            off[i] = __builtin_bit_cast(unsigned, q.x) * 4u;
            wt[i] = live ? q.y * kSplitScale : 0.f;
          }
        } else {
          const int64_t e = n_g * s.K + k0 + kl;
          const float scale = live ? (s.weighted ? s.iw[e] * kSplitScale : kSplitScale) : 0.f;
          PairTap<NE> t;
          resolve_pairs<NE, 4>(s.map[e * 2], s.map[e * 2 + 1], s.SH, s.SW, s.wrap != 0, scale, t);
#pragma unroll
          for (int i = 0; i < NA; i++) {
            off[i] = t.off[i];
            wt[i] = t.wt[i];
          }
        }
        if constexpr (NA > 1) {
          bool fits = plane_bytes >= 8u;
#pragma unroll
          for (int i = 0; i < NA; i += 2) {
            // entries i and i + 1 as two neighbours, where they are (an entry of weight zero
            // may move anywhere)
            const bool u0 = wt[i] != 0.f, u1 = wt[i + 1] != 0.f;
            if (u0 && u1) {
              if (off[i] == off[i + 1] + 4u) {
                const unsigned o = off[i];
                const float w = wt[i];
                off[i] = off[i + 1];
                wt[i] = wt[i + 1];
                off[i + 1] = o;
                wt[i + 1] = w;
              }
              fits = fits && off[i] + 4u == off[i + 1];
            } else if (plane_bytes >= 8u) {
              const unsigned o = u0 ? off[i] : u1 ? off[i + 1] : 0u;
              const float w = u0 ? wt[i] : u1 ? wt[i + 1] : 0.f;
              const bool end = o + 4u >= plane_bytes;  // the plane's last pixel: its left neighbour
              off[i] = end ? o - 4u : o;
              off[i + 1] = off[i] + 4u;
              wt[i] = end ? 0.f : w;
              wt[i + 1] = end ? w : 0.f;
            }
          }
          if (!fits) unpaired = 1;  // (every writer stores the same value)
        }
#pragma unroll
        for (int i = 0; i < NA; i++) {
          TapOff[(kl * kTilePx + p) * NA + i] = off[i];
          TapWt[(kl * kTilePx + p) * NA + i] = wt[i];
        }
      }
      __syncthreads();
      if constexpr (NA > 1) {
        if (!__builtin_amdgcn_readfirstlane(unpaired)) {
          units_of(k0, kn, na_tag, std::true_type());
          continue;
        }
      }
      units_of(k0, kn, na_tag, std::false_type());
    }
  };
  auto run = [&](auto na_tag) __attribute__((always_inline)) {
    constexpr int NA = decltype(na_tag)::value;
    // (two entries a tap of 64 outputs and more: as fast in memory, with the registers of a third wave)
    if constexpr (!WINDOW || (NA == 2 && NB > 1)) {
      in_memory(0, s.K, na_tag);
    } else {
      constexpr int kMost = kWinCache / NA < 6 ? kWinCache / NA : 6, kFew = 3;
      // (groups of one size, as far as it goes; a window that holds six taps' pixels holds three of nearly
      // twice the spread)
      const int groups = (s.K + kMost - 1) / kMost;
      int kg = (s.K + groups - 1) / groups;
      const bool small = s.SH <= 0xffff && s.SW <= 0xffff;
      for (int k0 = 0; k0 < s.K;) {
        const int kn = min(kg, s.K - k0);
        __syncthreads();  // the previous group's units are done with the taps and the window
        const int size = small ? in_window(k0, kn, na_tag) : 2;
        if (size > 1) {
          if (small && kn > kFew && size < 3) {
            kg = kFew;
            continue;
          }
          __syncthreads();
          if constexpr (NA == 2) {
            // (the others hardly fit, and six taps at a time are better off in memory than three: the map of every
            // other pixel, samples of 8 x 32 channels of 256 x 512 -> 24 of 128 x 256, 102 us, so 83)
            in_memory(k0, s.K - k0, na_tag);
            return;
          }
          in_memory(k0, kn, na_tag);
        }
        k0 += kn;
      }
    }
  };
  if (NE == 4 && leading)
    run(std::integral_constant<int, NE == 4 ? 2 : 1>());
  else
    run(std::integral_constant<int, NE>());
  split_epilogue<NB, (NE == 4 && NB > 1 ? 2 : 1)>(s, acc, Bias, tile, b, o0, tile_y * th + (pe >> s.tw_shift),
                     (tile_x << s.tw_shift) + (pe & tw_mask), lhi);
}

// Channel-last sources (mesh signals).  Four neighbouring lanes read the 64 bytes of a record's
// sixteen channels of a chunk together, two pixels a lane, interpolate them and hand them
// through LDS to the lane whose matrix operand they are: a load then meets 16 lines, where lanes that
// read their own operand's 32 bytes meet 64.  Mesh of 40 962 vertices, 4 x 64 -> 128 channels, four
// points a tap: forward 300 -> 253 us, input gradient 520 -> 417.
// Tap-major, a tap's entries in registers; NE entries a tap, and with TWO (a
// transposed map with a second level) four more where any lane of the wave uses one: both levels
// go through one product.
template <int NE, bool TWO, int NB>
__global__ __launch_bounds__(kThreads, TWO || NE * NB > 8 ? 2 : 3) void gather_product_split_cl_kernel(const SplitArgs s) {
  constexpr int NT = TWO ? NE + 4 : NE;
  __shared__ __attribute__((aligned(16))) uint4 Wt[2][SplitWeights<NB>::kPieces];
  constexpr int kSampleLd = kGC + 4;  // (eight lanes' 16-byte accesses on different banks)
  __shared__ __attribute__((aligned(16))) float Samples[kTilePx][kSampleLd];
  __shared__ __attribute__((aligned(16))) float Bias[32 * NB];
  if (s.gate && ((*s.gate == 0) != (s.run_if_zero != 0))) return;
  const int tid = threadIdx.x;
  const int tile = xcd_contiguous_tile(blockIdx.x, gridDim.x);
  const int b = tile / s.tiles_per_img;
  const int t_in = tile - b * s.tiles_per_img;
  const int tile_y = t_in / s.tiles_x, tile_x = t_in - tile_y * s.tiles_x;
  const int tw_mask = (1 << s.tw_shift) - 1, th = kTilePx >> s.tw_shift;
  const int o0 = blockIdx.y * (32 * NB);
  const int N = s.OH * s.OW;
  const int chunks = s.Gpad / kGC;
  const unsigned record = (unsigned)s.Gpad * 4u;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l31 = lane & 31, lhi = lane >> 5;
  const int pe = wave * 32 + l31;
  const int ei = tile_y * th + (pe >> s.tw_shift), ej = (tile_x << s.tw_shift) + (pe & tw_mask);
  // the two pixels of the wave whose records this lane reads, four channels of each
  const int qc = (lane & 3) * 4, qp = wave * 32 + (lane >> 2);
  bool live[2];
  int64_t n[2];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int px = qp + 16 * h;
    const int qi = tile_y * th + (px >> s.tw_shift), qj = (tile_x << s.tw_shift) + (px & tw_mask);
    live[h] = qi < s.OH && qj < s.OW;
    n[h] = live[h] ? (int64_t)qi * s.OW + qj : 0;
  }
  const int64_t pixels = (int64_t)s.SH * s.SW;
  const auto img = plane_buf(s.src + (int64_t)b * pixels * s.Gpad, (unsigned)pixels * record);
  const auto wbuf = plane_buf(s.w, (unsigned)s.K * chunks * 6u * s.Opad * 16u);
  const unsigned w_unit = 6u * s.Opad * 16u;

  floatx16 acc[NB];
#pragma unroll
  for (int m = 0; m < NB; m++)
#pragma unroll
    for (int i = 0; i < 16; i++) acc[m][i] = 0.f;
  SplitWeights<NB> wts;
  wts.init(tid, s.Opad, o0);
  split_bias<NB>(s, Bias, o0);

  const bool packed = TWO || s.packed;  // (only a transposed map has a second level)
  // entries of a tap as they come from memory, fetched a tap ahead
  float2 raw[2][NT];
  float raw_w[2][NE];
  auto fetch = [&](int k) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
#pragma unroll
      for (int i = 0; i < NE; i++) {
        if (packed) {
          raw[h][i] = reinterpret_cast<const float2 *>(s.map)[((int64_t)k * 4 + i) * N + n[h]];
          raw_w[h][i] = 0.f;
        } else {
          const int64_t e = (n[h] * s.K + k) * NE + i;
          raw[h][i] = reinterpret_cast<const float2 *>(s.map)[e];
          raw_w[h][i] = s.weighted ? s.iw[e] : 1.f;
        }
      }
      if constexpr (TWO) {
#pragma unroll
        for (int i = 0; i < 4; i++) raw[h][NE + i] = s.map2[((int64_t)k * 4 + i) * N + n[h]];
      }
    }
  };
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  unsigned off[2][NT];
  float wgt[2][NT];
  f32x4 v[2][NT];
  typename SplitWeights<NB>::u32x4 wv[SplitWeights<NB>::kPer];
  bool more = false;  // (wave-uniform) an entry beyond the first NE is in use
  auto resolve = [&]() __attribute__((always_inline)) {
    bool any = false;
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int i = 0; i < NT; i++) {
        if (packed || i >= NE) {
          off[h][i] = __builtin_bit_cast(unsigned, raw[h][i].x) * record;
          wgt[h][i] = live[h] ? raw[h][i].y * kSplitScale : 0.f;
        } else {
          PairTap<1> t;
          resolve_pairs<1, 1>(raw[h][i].x, raw[h][i].y, s.SH, s.SW, false,
                              live[h] ? raw_w[h][i < NE ? i : 0] * kSplitScale : 0.f, t);
          off[h][i] = t.off[0] * record;
          wgt[h][i] = t.wt[0];
        }
        off[h][i] += (unsigned)qc * 4u;
        if (i >= NE) any |= wgt[h][i] != 0.f;
      }
    if constexpr (TWO) more = __builtin_amdgcn_ballot_w64(any) != 0;
  };
  auto issue = [&](int k, int c) __attribute__((always_inline)) {
    const int so = __builtin_amdgcn_readfirstlane(c * (kGC * 4));
    auto load = [&](int i) __attribute__((always_inline)) {
#pragma unroll
      for (int h = 0; h < 2; h++)
        v[h][i] = __builtin_bit_cast(
            f32x4, __builtin_amdgcn_raw_buffer_load_b128(img, (int)off[h][i], so, 0));
    };
    wts.load(wbuf, __builtin_amdgcn_readfirstlane((unsigned)(k * chunks + c) * w_unit), wv);
#pragma unroll
    for (int i = 0; i < NE; i++) load(i);
    if constexpr (TWO) {
      if (more) {
#pragma unroll
        for (int i = NE; i < NT; i++) load(i);
      }
    }
  };

  fetch(0);
  resolve();
  fetch(min(1, s.K - 1));
  issue(0, 0);
  const int units = s.K * chunks;
  int k = 0, c = 0, buf = 0;
  for (int u = 0; u < units; u++) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
      f32x4 q;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        q[j] = wgt[h][0] * v[h][0][j];
#pragma unroll
        for (int i = 1; i < NE; i++) q[j] = __builtin_fmaf(wgt[h][i], v[h][i][j], q[j]);
      }
      if constexpr (TWO) {
        if (more) {
#pragma unroll
          for (int i = NE; i < NT; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) q[j] = __builtin_fmaf(wgt[h][i], v[h][i][j], q[j]);
        }
      }
      *reinterpret_cast<f32x4 *>(&Samples[qp + 16 * h][qc]) = q;
    }
    // (of this wave's own pixels: LDS serves a wave in order, and the fences, which cost nothing,
    // keep the compiler from moving a lane's reads ahead of what other lanes write)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    float sv[8];
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const f32x4 q = *reinterpret_cast<const f32x4 *>(&Samples[pe][lhi * 8 + 4 * j]);
#pragma unroll
      for (int e = 0; e < 4; e++) sv[4 * j + e] = q[e];
    }
    bf16x8 bq[3];
    split8(sv, bq);
    wts.store(Wt[buf], wv);
    __syncthreads();
    if (u + 1 < units) {
      if (++c == chunks) {
        c = 0;
        ++k;
        resolve();
        fetch(min(k + 1, s.K - 1));
      }
      issue(k, c);
    }
    bf16x8 a[NB][3];
    read_split_weights<NB>(Wt[buf], l31, lhi, a);
    split_products<NB>(a, bq, acc);
    buf ^= 1;
  }
  split_epilogue<NB, (NE == 4 && NB > 1 ? 2 : 1)>(s, acc, Bias, tile, b, o0, ei, ej, lhi);
}

}  // namespace

int launch_gather_split(const SplitArgs &a, int64_t tiles, bool cl, hipStream_t s) {
  // Blocks of 32 outputs a workgroup computes: a block of zeros costs as many matrix instructions
  // as one of weights, and its accumulators the registers of a fourth wave.  (Always two or four of
  // them, against this: 4 x 64 -> 32 channels onto 256 x 512, transposed, forward and backward 450 us, 413;
  // 3 x 24 -> 40 of 125 x 250, whose input gradient has 24, 257 and 253.  Three blocks keep the two waves
  // of four.)
  const int blocks = (a.O + 31) / 32;
  const int nb = blocks == 1 ? 1 : blocks == 3 ? 3 : a.Opad % (2 * kOT) == 0 ? 4 : 2;
  const int64_t by_outputs = (blocks + nb - 1) / nb;
  // Windows (gather_product_split_kernel) where the grid is three workgroups a CU and more - with fewer,
  // each waits out a group's taps and then its window, where the form in memory has its loads in flight
  // - and where two chunks of channels and more share the taps' work; not with four blocks of outputs,
  // whose matrix instructions hide the loads.  In memory and in windows: 8 x 64 -> 64 channels of 256 x 512, four
  // corners, 770 us and 669; 3 x 64 -> 64 of 128 x 256 95 and 84; 8 x 32 -> 96 of 128 x 256 156 and 147; 3 x 24 -> 40 of
  // 125 x 250, a training pass, 246 and 213; 4 x 64 -> 32 onto 256 x 512, transposed, 380 and 355.  Against
  // them: 4 x 32 -> 32 of 64 x 128 (256 workgroups) 31.3 and 34.4; 8 x 8 -> 3 onto 256 x 512, transposed, 159 and
  // 188; 4 x 16 -> 20 of 128 x 256 32 and 38; 2 x 40 -> 128 of 128 x 256, 5 x 5, 159 and 176.
  // One tap and one block of outputs have nothing else that would share the window (one tap, in windows and in memory:
  // 2 x 64 -> 3 of 256 x 512 39 and 28; 4 x 128 -> 1 97 and 66; 4 x 32 -> 32 57 and 40, of a random map, whose groups do not
  // fit and are the fewer at a time for it, 489 and 577).
  const bool window = tiles * by_outputs >= 768 && a.G > kGC && nb < 4 && (a.K > 1 || nb > 1);
  const dim3 grid((unsigned)tiles, (unsigned)by_outputs);
#define MCX_SPLIT(KERNEL, ...) \
  hipLaunchKernelGGL((KERNEL<__VA_ARGS__>), grid, dim3(kThreads), 0, s, a)
#define MCX_SPLIT_CL(...)                                                       \
  switch (nb) {                                                                 \
    case 1: MCX_SPLIT(gather_product_split_cl_kernel, __VA_ARGS__, 1); break;   \
    case 2: MCX_SPLIT(gather_product_split_cl_kernel, __VA_ARGS__, 2); break;   \
    case 3: MCX_SPLIT(gather_product_split_cl_kernel, __VA_ARGS__, 3); break;   \
    default: MCX_SPLIT(gather_product_split_cl_kernel, __VA_ARGS__, 4); break;  \
  }
#define MCX_SPLIT_PLANAR(NE, WINDOW)                                                   \
  switch (nb) {                                                                        \
    case 1: MCX_SPLIT(gather_product_split_kernel, NE, 1, WINDOW); break;              \
    case 2: MCX_SPLIT(gather_product_split_kernel, NE, 2, WINDOW); break;              \
    case 3: MCX_SPLIT(gather_product_split_kernel, NE, 3, WINDOW); break;              \
    default: MCX_SPLIT(gather_product_split_kernel, NE, 4, false); break;              \
  }
  if (cl) {
    if (a.map2) {
      MCX_SPLIT_CL(4, true)
    } else {
      switch (a.packed ? 4 : a.np) {
        case 1: MCX_SPLIT_CL(1, false) break;
        case 2: MCX_SPLIT_CL(2, false) break;
        case 3: MCX_SPLIT_CL(3, false) break;
        default: MCX_SPLIT_CL(4, false) break;
      }
    }
  } else if (!a.packed && a.ncorn == 1) {
    MCX_SPLIT_PLANAR(1, false)
  } else if (window) {
    MCX_SPLIT_PLANAR(4, true)
  } else {
    MCX_SPLIT_PLANAR(4, false)
  }
#undef MCX_SPLIT_CL
#undef MCX_SPLIT_PLANAR
#undef MCX_SPLIT
  MCX_HIP_CHECK_LAUNCH();
  return 0;
}

}  // namespace mcx
