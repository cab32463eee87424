// Walks the waves' runs of pw_any_kernel on the host with the kernel's own arithmetic (csrc/pw_any_geom.h): every pixel in
// one run, no pixel counter past what an int holds, piece of a block's last pixels inside the block.  Layers on stdin, one a
// line: M N K bn_bytes cus.  One line out per layer: "ok RUNS", "no" (not taken by the kernel) or what is wrong.
#include <stdio.h>

#include <string>

#include "../../pulp_nn_amd/csrc/pw_any_geom.h"

static std::string check(long long M, int N, int K, int bn_bytes, int cus)
{
  PwAnyGeom g;
  int ks, np;
  if (!pw_any_shape(M, N, K, cus, bn_bytes, &g, &ks, &np)) return "no";
  const int nw = ks <= 2 ? 16 : 8;
  if (pw_any_lds(ks, np, nw, bn_bytes) > 160 * 1024 - 512) return "more LDS than a launch may ask for";
  if (64 * ks < K || 64 * np < g.NB || g.NB * g.nblk < N || N - (g.nblk - 1) * g.NB < 16 || (g.nblk > 1 && g.NB % 4)) return "blocks of channels";
  long long next = 0, runs = 0;
  for (int wg = 0; wg < g.nwg; wg++)
    for (int wave = 0; wave < nw; wave++) {
      int px, px_end;
      pw_any_run(g, wg, wave, nw, &px, &px_end);
      if (px >= px_end) continue;
      if (px != next) return "run starts at pixel " + std::to_string(px) + ", the one before ended at " + std::to_string(next);
      // the run's last step asks for the pixels of two steps ahead, and its counter goes one step past the end (steps of 32 in
      // pw_stream_kernel, which has the same limit)
      const long long last = px + (px_end - 1ll - px) / 16 * 16;
      if (last + 3 * 32 + 15 > 0x7fffffffll) return "pixel counter past an int: " + std::to_string(last);
      next = px_end;
      runs++;
    }
  if (next != M) return "pixels left out from " + std::to_string(next);
  return "ok " + std::to_string(runs);
}

int main()
{
  long long M;
  int N, K, bn_bytes, cus;
  while (scanf("%lld %d %d %d %d", &M, &N, &K, &bn_bytes, &cus) == 5) puts(check(M, N, K, bn_bytes, cus).c_str());
  return 0;
}
