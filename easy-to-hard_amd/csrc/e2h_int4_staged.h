// Decode-batch int4 matmul on staged activations: its arguments, and the launches of each group size (one translation unit each, e2h_int4_staged_g*.hip, so that
// they compile beside each other).
#pragma once

#include "e2h_common.h"
#include "e2h_staged.h"

namespace e2h {
namespace staged {

enum StagedEpilogue { kStPlain = 0, kStGate = 1, kStRope = 2, kStPartial = 3, kStArgmax = 4 };

struct StagedRope {
  const uint16_t *freqs;     // [>= S, D/2, 2] bf16 (cos, sin)
  uint16_t *q_out, *kc, *vc;
  const int64_t *input_pos;  // [1] on the device
  int H, Hkv, S, D;
};

struct StagedArgs {
  const uint8_t *frag;  // staged activations
  const float *sums;
  const uint32_t *wp, *sz, *wp2, *sz2;
  uint16_t *y;          // bf16 [M][N] (plain, gate; may be null for gate when only the staged result is wanted)
  float *partials;      // f32 [S][M][N] (partial)
  unsigned long long *cand;  // [column blocks][M] (arg-max): per row the best (value key << 32 | ~column) of the block's columns
  StagedOut out;        // gate: the result in staged form for the next linear (frag null: not wanted)
  int M, Mpad, N, K;
  int col_blocks;
  StagedRope rope;
};

struct Geometry {
  int t, slices, mt, halves, waves;  // weight tiles per workgroup, workgroups along K, row tiles per workgroup, workgroups along the rows, waves of a workgroup
};

// most weight tiles whose sums, words, pairs and operands fit a wave's 256 vector registers beside the group's products
constexpr int max_tiles(int G, int MT, bool gate) { return MT == 4 ? 6 : gate && G != 32 ? 12 : 8; }

// group size G: 32, 64 or 128
template <int G>
int launch_group(int epilogue, const StagedArgs &a, const Geometry &g, hipStream_t stream);

}  // namespace staged
}  // namespace e2h
