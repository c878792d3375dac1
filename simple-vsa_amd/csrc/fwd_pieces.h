// How many workgroups of the block-64 forward one launch takes (host code only,
// kept apart from fine_fwd.hip so that a host program can check it).
#pragma once

#include <stdint.h>

namespace vsa {

// Workgroups a CU holds at block 64 (two waves each): four at head dim 128, by
// registers (two waves a SIMD), eight at 64 (four waves a SIMD).
constexpr int fwd_wg_per_cu(int D) { return D == 64 ? 8 : 4; }

// Workgroups of one launch, of `grid` (a multiple of 8) in all.
//
// Workgroups of one head that start together walk their routes (ascending key
// blocks) roughly in step and find most K / V tiles in their XCD's L2; left to
// start as others end, they drift apart, and a head's K / V does not fit.  At
// block 64, which reads the most K / V per product, a long pass (ten times the
// workgroups the chip holds at once: the drift adds up) whose heads have
// several times the L2 of K / V and whose routes are long is therefore launched
// in pieces of the workgroups the chip holds (the last one takes the
// remainder).  Whole / in pieces on the op's own routes, head dim 128, top-k an
// eighth: 40 heads x 640 blocks 6.90 / 5.50 ms, 24 x 640 3.84 / 3.33, 16 x 640
// 2.45 / 2.27, 12 x 1280 8.60 / 6.64, 40 x 400 2.44 / 2.34; head dim 64, 24 x
// 1280 8.57 / 7.22.  On skewed routes, which share key blocks as they are, the
// lines keep it even (40 x 384 1.84 / 1.83 ms, 24 x 1280 with 48 of them 3.86 /
// 3.89, head dim 64 6.51 / 6.52); below them the pieces' ends cost what they
// bring: 12 x 624 1.49 / 1.53 ms, 24 x 320 822 / 829 us, skewed routes of 40 in
// 1280 3.44 / 3.52 ms, at head dim 64 of 100 in 800 2.47 / 2.60; so they do for
// padded rows (20 x 640 blocks of 27, with backward 5.55 / 5.62), at block 128
// (16 x 640 7.38 / 7.44) and at head dim 256 (8 x 640 2.66 / 2.70).
inline int fwd_piece(int D, int be, int rows, int grid, int64_t skv, int topk, int elem_bytes,
                     int cus) {
  constexpr int64_t kL2Bytes = 4 << 20;
  const int64_t kv_bytes = (D == 64 ? 5 : 3) * kL2Bytes;
  const int long_route = D == 64 ? 160 : 48;
  const int held = (cus * fwd_wg_per_cu(D) + 7) / 8 * 8;
  const bool pieces = be == 64 && D <= 128 && rows > be - 32 && topk >= long_route &&
                      2 * skv * D * elem_bytes >= kv_bytes && grid / 10 >= held;
  return pieces ? held : grid;
}

// Size of the launch that starts at workgroup `first`.
inline int fwd_launch(int grid, int first, int piece) {
  const int left = grid - first;
  return left - piece < piece ? left : piece;
}

}  // namespace vsa
