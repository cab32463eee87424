// How a pooling window is read: in blocks of so many columns and rows of taps, whose loads are issued together.  Plain C++: the launch
// chooses, the kernels have a loop for each, and a host program can count.
#pragma once

enum PoolBlock { PB_1x1, PB_2x1, PB_1x2, PB_2x2, PB_3x1, PB_1x3, PB_3x3, PB_4x1, PB_1x4, PB_5x1, PB_5x3, PB_4x4, PB_COUNT };
struct PoolBlockSize {
  int w, h;
};
inline PoolBlockSize pool_block_size(int block)
{
  static const PoolBlockSize sizes[PB_COUNT] = {{1, 1}, {2, 1}, {1, 2}, {2, 2}, {3, 1}, {1, 3}, {3, 3}, {4, 1}, {1, 4}, {5, 1}, {5, 3}, {4, 4}};
  return sizes[block];
}
inline long long pool_block_trips(int kx, int ky, int block)
{
  const PoolBlockSize s = pool_block_size(block);
  return (long long)((kx + s.w - 1) / s.w) * ((ky + s.h - 1) / s.h);
}

// The block with the least of loads and trips to memory, a trip counting as two loads (taps past the window's end are loaded, its last row or
// column once more).  Whole calls, blocks by the window's longer side / so: average 7x1 on 64 images of 28x28x256 38.2 / 18.8 us, 5x5 62.6 / 38.1,
// 7x1 stride 7x1 8.8 / 5.1, 28x1 stride 28x1 8.9 / 4.8.
inline int pool_avg_block(int kx, int ky)
{
  int best = PB_1x1;
  long long least = -1;
  for (int b = PB_COUNT - 1; b >= 0; b--) {
    const PoolBlockSize s = pool_block_size(b);
    const long long cost = pool_block_trips(kx, ky, b) * (s.w * s.h + 2);
    if (least >= 0 && cost >= least) continue;
    least = cost;
    best = b;
  }
  return best;
}

// The maximum, sixteen channels a tap: windows of up to 2x2 and of up to 3x3 as a whole, others in a row or a column with the fewest loads (trips
// between equals).  Rows of four or five and nine taps up to 3x3, whatever the window / so: 1x7 on 64 images of 28x28x256 26.3 / 13.7 us, 1x4 stride
// 1x4 7.8 / 3.9, 3x1 11.4 / 6.8.
inline int pool_max_block(int kx, int ky)
{
  if (kx <= 2 && ky <= 2) return PB_2x2;
  if (kx > 1 && ky > 1 && kx <= 3 && ky <= 3) return PB_3x3;
  int best = PB_4x1;
  const int others[] = {PB_5x1, PB_3x1, PB_1x4, PB_1x3};
  auto cost = [&](int b) { return pool_block_trips(kx, ky, b) * (pool_block_size(b).w * pool_block_size(b).h + 1); };
  for (const int b : others)
    if (cost(b) < cost(best)) best = b;
  return best;
}
