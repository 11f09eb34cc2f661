// Interface of the weight gradient over runs of neighbouring pixels (mcx_conv_runs.hip).
#pragma once

#include "mcx_device.h"

namespace mcx {

// Words of `state`: [0] this path has done the work, [1] a sum is not finite, [2] pair mask for
// weight_grad_mfma_kernel (at least 4: corners of the lower row are in use), [3] the table of its taps
// is there.
constexpr int kRunStateWords = 64;

__device__ inline bool runs_done(const int *state) { return state[0] != 0 && state[1] == 0; }
__device__ inline bool runs_table(const int *state) { return state[3] != 0; }

// How the work is cut, from the sizes alone.
struct RunPlan {
  int st, cblocks, ablocks, passes, groups, tiles_per_img;
  int64_t total_tiles;
  int ranges, stat_words;
  size_t desc_bytes, wts_bytes;
  double us;  // of the kernel, about, where all groups are runs under one row of corners
  // What the groups that are no runs (448 each, 160 under one row of corners) and those fetched element
  // by element (56 and 10) may come to.  Less than zero: the general kernel is the faster one for every
  // map.
  int64_t limit;
};
RunPlan run_plan(int64_t B, int64_t A, int64_t G, int64_t GW, int64_t MH, int64_t MW, int64_t K);
bool runs_apply(int64_t B, int64_t A, int64_t G, int64_t GH, int64_t GW, int64_t MH, int64_t MW,
                int64_t K, int64_t P);
// Sets `limit` where the general kernel, and what goes with it, take general_us.  A workgroup waits for
// its slowest wave, and a wave for corners or elements fetched one by one: each hundredth of the
// groups that is no run costs a tenth of the time under one row of corners, a quarter under two (8 x 64 -> 64
// channels of 256 x 512, general kernel in brackets: no such groups 675 us (800), 1.6 % 763 (798), 3.1 % 853
// (810), 12 % 1260 (871); two rows 865 (974), 1.6 % 1094 (1001), 12 % 2207 (1151)), a group fetched
// element by element a sixteenth and an eighth of that.
void set_run_limit(RunPlan &p, int64_t K, double general_us);
// Bytes of the tables that resolve_runs fills, and their state words.
size_t run_table_bytes(const RunPlan &p);
int *run_state(const RunPlan &p, char *tables);
// What weight_grad_mfma_kernel reads where this path leaves a map of two-pair taps to it: the taps in
// the order of its tiles, [tile of an image][tap][pixel of the tile] two byte offsets in a plane and
// their two weights.  table NULL: taps of one corner.
struct TapTable {
  uint4 *table;
  int tiles_x, tw_shift, tiles;
};
int resolve_runs(const RunPlan &p, char *tables, const float *map, const float *iw, int64_t GH,
                 int64_t GW, int64_t MH, int64_t MW, int64_t K, int ncorn, int wrap, int weighted,
                 const TapTable &taps, hipStream_t stream);
// Per-range partial sums [ranges][K][G][A padded to 4]; sum_part (may be NULL): the same of the
// plain operand, [ranges][A].
int weight_grad_by_runs(const RunPlan &p, char *tables, const float *plain, const float *gath,
                        float *part, float *sum_part, int64_t A, int64_t G, int64_t GH, int64_t GW,
                        int64_t MH, int64_t MW, int64_t K, hipStream_t stream);

}  // namespace mcx
