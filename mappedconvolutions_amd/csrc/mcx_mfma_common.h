// What the matrix-core kernels share: operand types, the exact split of fp32 values into three
// bf16 parts (mcx_conv_split.hip says what it is for), and the order of workgroups over the chip.
#pragma once

#include "mcx_taps.h"

namespace mcx {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));

// acc + w.lo * word.lo + w.hi * word.hi (v_dot2_f32_bf16: products exact, fp32 sum)
__device__ inline float dot_bf16(unsigned word, unsigned w, float acc) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, word),
                                         __builtin_bit_cast(bf16x2, w), acc, false);
}

constexpr int kTilePx = 128;  // pixels of a tile
constexpr int kGC = 16;       // source channels per reduction chunk
constexpr int kOT = 64;       // outputs are padded to a multiple of this

// Factor of the weights and of the samples before they are split.
constexpr float kSplitScale = 16777216.f;  // 2^24
constexpr float kSplitUnscale = 1.f / (kSplitScale * kSplitScale);

// x = p[0] + p[1] + p[2] for 8 values: words of two bf16 each
__device__ inline void split8(const float *x, bf16x8 *p) {
  unsigned h[4], m[4], l[4];
  // {-1, 0} and {0, -1} from registers: as immediates the compiler renders both as the inline
  // constant -1.0, which the instruction takes for one and the same word.
  unsigned neg_lo = 0x0000bf80u, neg_hi = 0xbf800000u;
  asm("" : "+s"(neg_lo), "+s"(neg_hi));
#pragma unroll
  for (int j = 0; j < 4; j++) {
    // (a remainder is the dot product of the pair word with {-1, 0} or {0, -1} plus the value)
    h[j] = __builtin_bit_cast(unsigned,
                              __builtin_convertvector(floatx2{x[2 * j], x[2 * j + 1]}, bf16x2));
    const float r0 = dot_bf16(h[j], neg_lo, x[2 * j]);
    const float r1 = dot_bf16(h[j], neg_hi, x[2 * j + 1]);
    m[j] = __builtin_bit_cast(unsigned, __builtin_convertvector(floatx2{r0, r1}, bf16x2));
    const float q0 = dot_bf16(m[j], neg_lo, r0);
    const float q1 = dot_bf16(m[j], neg_hi, r1);
    l[j] = __builtin_bit_cast(unsigned, __builtin_convertvector(floatx2{q0, q1}, bf16x2));
  }
  p[0] = __builtin_bit_cast(bf16x8, make_uint4(h[0], h[1], h[2], h[3]));
  p[1] = __builtin_bit_cast(bf16x8, make_uint4(m[0], m[1], m[2], m[3]));
  p[2] = __builtin_bit_cast(bf16x8, make_uint4(l[0], l[1], l[2], l[3]));
}

// Whether a pair beyond the first two of a tap is in use anywhere in the map, from the pair
// mask: one word (at least 4 then), or `words` words of which any may say so (one per block
// of the launch that examined the map).  Called by whole waves.
__device__ inline bool later_pairs_in_use(const int *__restrict__ mask, int words) {
  if (words <= 1) return (unsigned)*mask >= (1u << 2);
  const int lane = threadIdx.x & 63;
  const unsigned v = (unsigned)mask[lane < words ? lane : 0];
  return __builtin_amdgcn_ballot_w64(v >= (1u << 2)) != 0;
}

// Workgroups are dealt round-robin to the 8 XCDs; give every XCD one contiguous
// run of tiles so that neighbouring tiles (which share source rows) share an L2.
__device__ inline int xcd_contiguous_tile(int wg, int total) {
  const int q = total >> 3, r = total & 7;
  const int xcd = wg & 7, slot = wg >> 3;
  return xcd * q + min(xcd, r) + slot;
}

inline size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

}  // namespace
}  // namespace mcx
