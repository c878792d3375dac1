// Launch sizes of the block-64 forward (host program, see test_fwd_pieces_host.py):
// arguments D, block, rows, tiles, skv, topk, element bytes, CUs; prints the size
// of each launch, or with D alone the workgroups a CU holds.
#include "fwd_pieces.h"

#include <cstdio>
#include <cstdlib>

int main(int argc, char** argv) {
  long long a[8] = {};
  for (int i = 1; i < argc && i <= 8; ++i) a[i - 1] = atoll(argv[i]);
  if (argc == 2) return printf("%d\n", vsa::fwd_wg_per_cu((int)a[0])) < 0;
  const int grid = (int)((a[3] + 7) / 8 * 8);
  const int piece = vsa::fwd_piece((int)a[0], (int)a[1], (int)a[2], grid, a[4], (int)a[5],
                                   (int)a[6], (int)a[7]);
  for (int first = 0, n; first < grid; first += n)
    printf("%d ", n = vsa::fwd_launch(grid, first, piece));
}
