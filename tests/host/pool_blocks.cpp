// What the pooling kernels load for a window, by the blocks that their launches choose (csrc/pool_blocks.h).
// Windows on stdin, one a line: kx ky.  One line out per window: loads and trips to memory of the average, of the maximum.
#include <stdio.h>

#include "../../pulp_nn_amd/csrc/pool_blocks.h"

static void say(int kx, int ky, int block)
{
  const PoolBlockSize s = pool_block_size(block);
  const long long trips = pool_block_trips(kx, ky, block);
  printf("%lld %lld ", trips * s.w * s.h, trips);
}

int main()
{
  int kx, ky;
  while (scanf("%d %d", &kx, &ky) == 2) {
    say(kx, ky, pool_avg_block(kx, ky));
    say(kx, ky, pool_max_block(kx, ky));
    puts("");
  }
  return 0;
}
