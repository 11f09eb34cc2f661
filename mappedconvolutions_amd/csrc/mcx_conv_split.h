// Interface of the fp32 gather-product on the bf16 matrix instructions (mcx_conv_split.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mcx {

struct SplitArgs {
  const float *src, *map, *iw;
  const float2 *map2;     // second-level entries of a transposed map, or NULL (channel-last only)
  const uint16_t *w;      // split weights, see pack_split_weight
  const float *bias;
  float *y;
  const float *addend;    // see gather_product_mfma_kernel, like the gates and masks below
  const int *gate, *pair_mask, *row_mask;
  int *nonfinite;         // a word per pixel tile
  int G, O, Opad, Gpad, SH, SW, OH, OW, K, np, ncorn, weighted, wrap, packed;
  int tiles_x, tiles_per_img, tw_shift, run_if_zero, mask_words;
};

// Channel (of G) that element j of half kg of chunk c stands for, or -1 (a weight of zero).
// Planar sources read the second half of a partial last chunk `rem - 8` channels after the
// first, so that no lane reads past the last channel (see split_upper_half).
__host__ __device__ inline int split_channel(int c, int kg, int j, int G, int planar) {
  const int g0 = c * 16, rem = G - g0;
  if (!planar || rem >= 16) return g0 + kg * 8 + j < G ? g0 + kg * 8 + j : -1;
  if (kg == 0) return j < rem ? g0 + j : -1;
  if (rem <= 8) return -1;
  return g0 + rem - 8 + j >= g0 + 8 ? g0 + rem - 8 + j : -1;
}

// tiles: of 128 pixels, over all images; cl: the source is channel-last.
int launch_gather_split(const SplitArgs &a, int64_t tiles, bool cl, hipStream_t s);

}  // namespace mcx
