// Walks the rows of dw_hwc_kernel on the host, with the kernel's own arithmetic (csrc/dw_hwc_geom.h), and reports loads of another
// byte than the one meant, LDS places outside a row or used twice, and output bytes written twice, to a wrong place or not at all.
// Layers on stdin, one a line: B CH H W Ho S cus.  One line out per layer: "ok ROWS", "no" (not taken) or what is wrong.
#include <stdio.h>
#include <stdlib.h>

#include <set>
#include <string>
#include <vector>

#include "../../pulp_nn_amd/csrc/dw_hwc_geom.h"

template <int W, int S>
static std::string check(const DwLayer &L, int cus)
{
  constexpr int NT = 64 / W, WO = W / S;
  DwhGeom g;
  if (!dwh_shape<W, S>(L, cus, &g)) return "no";
  const long long in_bytes = (long long)L.B * L.H * W * L.CH, out_bytes = (long long)L.B * L.Ho * WO * L.CH;
  if ((long long)g.lead + in_bytes != g.size || out_bytes != g.out_size || g.size >= DWH_OOB || g.out_size >= DWH_OOB) return "sizes of the buffers";
  std::set<int> places;
  for (int col = 0; col < W + 2; col++)
    for (int j = 0; j < NT; j++) {
      const int p = dwh_lds<W>(col, j);
      if (p < 0 || p + 16 > dwh_row_bytes<W>() || p % 16 || !places.insert(p).second) return "place in LDS";
    }
  const bool all = g.total <= 3000;
  std::vector<unsigned char> written(all ? out_bytes / 4 : 0);
  for (int i = 0; i < (all ? g.total : 400); i++) {
    const DwhItem it = dwh_item<NT>(g, all || i < 200 ? (unsigned)i : (unsigned)(g.total - 400 + i));
    if ((int)it.b >= L.B || it.c0 >= L.CH || it.oy0 >= L.Ho || it.rows <= 0) return "empty item";
    for (int ir = 0; ir < dwh_rows_in<S>(it) + 8; ir++) {
      const int iy = it.oy0 * S - 1 + ir;
      if (dwh_row_ok<S>(g, it, ir) != (iy >= 0 && iy < L.H && ir < (it.rows - 1) * S + 3)) return "rows that are fetched";
      if (!dwh_row_ok<S>(g, it, ir)) continue;
      for (int lane = 0; lane < 64; lane++) {
        const long long at = (long long)dwh_in_offset<W, S>(g, it, lane) + (long long)ir * W * L.CH - g.lead;
        const long long want = (((long long)it.b * L.H + iy) * W + lane / NT) * L.CH + it.c0 + 16 * (lane % NT);
        if (at != want || at < 0 || at + 16 > in_bytes) return "load at " + std::to_string(at) + " for " + std::to_string(want);
      }
    }
    for (int r = 0; r < it.rows + 4; r += W == 64 ? S : 1)
      for (int lane = 0; lane < 64; lane++)
        for (int x = 0; x < (NT == 1 ? 1 : WO / 16); x++) {
          if (!dwh_out_ok<W, S>(it, r, lane)) continue;
          // NT == 1: chunk `lane` of the rows from r on; else 4 * NT channels of pixel lane % 16 of strip x
          const int px = NT == 1 ? lane % WO : 16 * x + lane % 16, row = NT == 1 ? r + lane / WO : r, ch = NT == 1 ? 0 : 4 * NT * (lane / 16);
          const long long at = (long long)dwh_out_offset<W, S>(g, it, lane) + (long long)(r * WO + (NT == 1 ? 0 : 16 * x)) * L.CH;
          const long long want = (((long long)it.b * L.Ho + it.oy0 + row) * WO + px) * L.CH + it.c0 + ch;
          if (at != want || row >= it.rows || at + (NT == 1 ? 16 : 4 * NT) > out_bytes) return "store at " + std::to_string(at) + " for " + std::to_string(want);
          if (all)
            for (int d = 0; d < (NT == 1 ? 4 : NT); d++)
              if (written[at / 4 + d]++) return "output written twice";
        }
  }
  for (const unsigned char w : written)
    if (!w) return "output left out";
  return "ok " + std::to_string(g.R);
}

int main()
{
  char line[256];
  while (fgets(line, sizeof line, stdin)) {
    DwLayer L{};
    int s, cus;
    if (sscanf(line, "%d %d %d %d %d %d %d", &L.B, &L.CH, &L.H, &L.W, &L.Ho, &s, &cus) != 7) return 1;
    L.sx = L.sy = s;
    L.Wo = (L.W - 1) / s + 1;
    std::string said = "no";
    if (L.W == 64) said = s == 1 ? check<64, 1>(L, cus) : check<64, 2>(L, cus);
    else if (L.W == 32) said = s == 1 ? check<32, 1>(L, cus) : check<32, 2>(L, cus);
    else if (L.W == 16 && s == 1) said = check<16, 1>(L, cus);
    puts(said.c_str());
  }
}
