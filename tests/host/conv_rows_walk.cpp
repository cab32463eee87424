// Walks the fetches of conv_rows_kernel on the host, with the kernel's own arithmetic (csrc/conv_rows_geom.h): bytes outside the input,
// and filter rows whose bytes would not end up in place.
// Layers on stdin, one a line: B H W Ci kx ky pt pl sx sy Ho Wo N.  One line out per layer: "ok", "no" (not taken) or what is wrong.
#include <stdio.h>
#include <stdlib.h>

#include <string>
#include <vector>

#include "../../pulp_nn_amd/csrc/conv_rows_geom.h"

// the 16 bytes of a lane after its fetch, as byte offsets of the input (-1: nothing that counts)
typedef std::vector<int> Bytes;

static std::string check(const RowsGeom &g, unsigned m, const RowsWindow &w, const RowsWindow &first, int l16, int fy, bool row16, bool staged, int group_at)
{
  const int at = row16 ? first.at + rows_lane(g, l16, fy) : w.at + fy * g.W * g.Ci;
  const RowsKeep k = rows_keep(g, w, fy);
  const bool mend = !row16 || rows_edge(g, first);
  Bytes got(16, -1);
  if (mend && k.row && rows_near_end(g, at)) {
    const int from = rows_exact(g, at);
    if (from < 0 || from + 16 > g.total) return "exact fetch outside";
    for (int j = 0; j < 16; j++)
      if (j + at - from >= 0 && j + at - from < 16) got[j] = at + j;
  } else if (staged) {
    // piece by piece: chunk c of row fy holds bytes from rows_chunk_at on, at 16 * c
    const int base = (group_at & ~3);
    for (int j = 0; j < 16; j++) {
      const int place = at + j - base, c = place / 16;
      if (place < 0 || c >= rows_chunks(g)) return "outside the row in LDS";
      const int from = rows_chunk_at(g, group_at, c);
      if (from < 0 || from + 16 > g.total) return "piece outside";
      got[j] = from + place % 16;
    }
  } else {
    const int from = rows_fetch(g, at), more = rows_more(g, at), sh = at & 3;
    if (from < 0 || from + 16 > g.total || from % 4 || more < 0 || more + 4 > g.total || more % 4) return "fetch outside";
    for (int j = 0; j < 16; j++)
      if (j + sh < 16) got[j] = from + j + sh;
      else if (rows_long(g)) got[j] = more + j + sh - 16;
  }
  for (int j = 0; j < g.L; j++) {
    const int ix = w.ix + j / g.Ci, iy = w.iy + fy;
    const bool inside = fy < g.ky && iy >= 0 && iy < g.H && ix >= 0 && ix < g.W;
    const bool kept = mend ? k.row && j >= k.lo && j < k.hi : fy < g.ky;
    if (kept != inside) return "byte kept or cleared wrongly";
    if (inside && got[j] != at + j) return "byte " + std::to_string(j) + " of pixel " + std::to_string(m) + " row " + std::to_string(fy);
  }
  return "";
}

int main()
{
  char line[256];
  while (fgets(line, sizeof line, stdin)) {
    int B, H, W, Ci, kx, ky, pt, pl, sx, sy, Ho, Wo, N;
    if (sscanf(line, "%d %d %d %d %d %d %d %d %d %d %d %d %d", &B, &H, &W, &Ci, &kx, &ky, &pt, &pl, &sx, &sy, &Ho, &Wo, &N) != 13) return 1;
    RowsGeom g;
    std::string said = "ok";
    if (!rows_shape((const uint8_t *)4096, nullptr, nullptr, nullptr, (long long)B * Ho * Wo, N, H, W, Ci, Ho, Wo, kx, ky, pt, pl, sx, sy, 256, 1, &g)) said = "no";
    else
      for (int place = 0; place < 3 && said == "ok"; place++) {  // any, units of one row, groups of one row
        if ((place == 1 && Wo % 16) || (place == 2 && (Wo % 64 || rows_chunks(g) > 32))) continue;
        for (unsigned m = 0; m < (unsigned)g.M && said == "ok"; m++)
          for (int fy = 0; fy < 4; fy++) {
            const RowsWindow w = rows_window(g, m), group = rows_window(g, m / 64 * 64);
            RowsWindow first = rows_window(g, m / 16 * 16);
            if (place == 2) {
              const int u = m % 64 / 16;
              const RowsWindow f = {group.at + 16 * u * g.sx * g.Ci, group.iy, group.ix + 16 * u * g.sx};
              if (f.at != first.at || f.ix != first.ix) said = "unit";
              first = f;
            }
            const std::string bad = check(g, m, w, first, m % 16, fy, place > 0, place == 2, group.at + fy * g.W * g.Ci);
            if (!bad.empty()) {
              said = bad;
              break;
            }
          }
      }
    puts(said.c_str());
  }
}
