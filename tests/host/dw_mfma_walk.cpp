// Walks the tiles of dw_mfma_kernel on the host, with the kernel's own tile arithmetic (csrc/dw_mfma_geom.h), and reports
// loads that leave the input, LDS ranges that overlap, and output pixels that are written to a wrong place or not at all.
// Layers on stdin, one a line: B CH H W Ho Wo kx ky pt pl sx sy cus.  One line out per layer: "ok TILES", "no" (not
// taken by the kernel) or what is wrong.
#include <stdio.h>
#include <stdlib.h>

#include <string>
#include <vector>

#include "../../pulp_nn_amd/csrc/dw_mfma_geom.h"

static std::string wrong(const char *what, const DwmTile &t, long long a, long long b)
{
  char s[200];
  snprintf(s, sizeof s, "%s: image %u channel %d row %d column %d: %lld, %lld", what, t.b, t.c0, t.oy0, 16 * t.xg0, a, b);
  return s;
}

template <int CB>
static std::string check(const DwLayer &L, int cus)
{
  DwmGeom g;
  int nm;
  size_t lds;
  if (!dwm_shape<CB>(L, cus, &g, &nm, &lds)) return "no";
  const long long plane = (long long)L.H * L.W, bytes = (long long)L.B * L.CH * plane;
  if (lds > 65536) return "more LDS than a launch may ask for";
  if (g.in_bytes != bytes) return "size of the input: " + std::to_string(g.in_bytes) + " for " + std::to_string(bytes);
  // all tiles, or the first, the last and some between
  std::vector<unsigned> ids;
  const bool all = g.total <= 4096;
  for (int i = 0; i < (all ? g.total : 512); i++) ids.push_back(all ? i : i < 256 ? i : g.total - 512 + i);
  long long outputs = 0;
  for (const unsigned id : ids) {
    const DwmTile t = dwm_tile<CB>(g, id);
    if ((int)t.b >= L.B || t.c0 >= L.CH || t.rows <= 0 || t.wt <= 0 || t.ncb <= 0) return wrong("empty tile", t, t.rows, t.wt);
    const long long before = ((long long)t.b * L.CH + t.c0) * plane;
    const int iy0 = t.oy0 * g.sy - g.pt, x0 = 16 * t.xg0 * g.sx - g.pl;
    const bool edge = dwm_edge(g, t, before);
    const long long behind = g.in_bytes - before - 16;
    const int lo = (int)std::max(-before, -(1ll << 30)), hi = (int)std::min(behind, 0x7fffffffll);
    // Every load the staging makes: the passes over slots, the threads of a pass, the channels of a thread.  `seen`: slots and channels staged.
    // (Of the first and the last 48 tiles.)
    const int slots = id < 48u || id + 48u >= (unsigned)g.total ? g.NR * g.Q : 0, UN = DWM_LOADS;
    std::vector<unsigned char> seen(slots * t.ncb);
    if (g.nper > 256 || g.nper * g.cpar > 256 || g.cpar < 1) return wrong("threads of a pass", t, g.nper, g.cpar);
    for (int s0 = 0; s0 < slots; s0 += g.nper)
      for (int tid = 0; tid < 256; tid++) {
        const int cpi = (int)fastdiv((unsigned)tid, g.d_nper), slot = s0 + tid - cpi * g.nper, row = (int)fastdiv((unsigned)slot, g.d_q), q = slot - row * g.Q;
        const int iy = iy0 + row, x = x0 + 16 * q, base = dwm_load_base(g, iy, x), ch = dwm_thread_channel(CB, cpi, slot < slots);
        for (int cj = 0; cj < t.ncb; cj += UN * g.cpar)
          for (int u = 0; u < UN; u++) {
            const int c = cj + u * g.cpar;
            if (u != 0 && c >= t.ncb) break;
            const bool staged = ch < t.ncb - c;
            long long at;  // bytes from the tile's first plane
            if (edge) {
              at = std::min(std::max(std::min(cpi + c, t.ncb - 1) * (int)plane + base, lo), hi);
            } else {
              const unsigned off = dwm_buffer_off(dwm_buffer_first((int)plane, ch, cpi, base), dwm_buffer_last((int)plane, t.ncb, ch, cpi, base), (int)plane, c);
              if (off >= (unsigned long long)std::min(g.in_bytes - before + 64, 0x7fffffffll)) {  // out of range: zeros
                if (staged) return wrong("load of a channel out of range", t, cpi + c, off);
                continue;
              }
              at = (long long)off - 64;
            }
            if (before + at < 0 || before + at + 16 > bytes) return wrong("load outside the input", t, before + at, bytes);
            if (!staged) continue;
            const long long want = (long long)(cpi + c) * plane + base;  // the chunk that the slot is for
            for (int j = 0; j < 16; j++)
              if (iy >= 0 && iy < L.H && x + j >= 0 && x + j < L.W && (j + want - at < 0 || j + want - at > 15))
                return wrong("byte of the image not loaded", t, iy, x + j);
            seen[slot * t.ncb + cpi + c] = 1;  // (threads past the channels side by side stage some of them once more, alike)
          }
      }
    for (const unsigned char n : seen)
      if (!n) return wrong("not staged", t, slots, t.ncb);
    // 8 bytes of filter a lane, from the tensor's last 8 at the most (layers of fewer are read byte by byte)
    for (int wave = 0; wave < 4; wave++) {
      const int nq = CB == 16 ? 1 : (t.ncb + 15) / 16, cw = 4 * nq * wave, nrow = 4 * nq * g.ky;
      if (nrow * DWM_WROW + 8 > dwm_wpart(CB, g.ky)) return wrong("filter rows of a wave", t, nrow, g.ky);
      for (int r = 0; r < std::max(nrow, 64) && g.wt_bytes >= 8; r++) {
        const int want = dwm_filter_at(g, t, cw, r), at = std::min(want, g.wt_bytes - 8);
        if (at < 0) return wrong("load outside the filters", t, cw, r);
        if (cw + r / g.ky < t.ncb && r < nrow && (want != ((t.c0 + cw) * g.ky + r) * g.kx || want + g.kx > at + 8)) return wrong("filter row not loaded", t, cw, r);
      }
    }
    if (g.NR * g.pitch > g.CS || 16 * g.Q > g.pitch || CB * g.CS > g.w_off || g.w_off + 4 * dwm_wpart(CB, L.ky) > g.o_off ||
        g.o_off + (size_t)t.rows * t.wt * (CB + 4) > lds)
      return wrong("LDS ranges", t, g.o_off, (long long)lds);
    for (int p = 0; p < t.rows * t.wt; p++)
      if (dwm_out_row(g, t, p) * (L.Wo - t.wt) != (p / t.wt) * (L.Wo - t.wt)) return wrong("output pixel misplaced", t, p, dwm_out_row(g, t, p));
    outputs += (long long)t.rows * t.wt * t.ncb;
  }
  if (all && outputs != (long long)L.B * L.CH * L.Ho * L.Wo) return "outputs left out";
  return "ok " + std::to_string(g.total) + (CB == 64 && dwm_wide(L, g, cus) ? " wide" : "");
}

int main()
{
  DwLayer L = {};
  int cus;
  while (scanf("%d %d %d %d %d %d %d %d %d %d %d %d %d", &L.B, &L.CH, &L.H, &L.W, &L.Ho, &L.Wo, &L.kx, &L.ky, &L.pt, &L.pl, &L.sx, &L.sy, &cus) == 13) {
    std::string s = check<16>(L, cus);
    if (s.compare(0, 2, "ok") == 0 || s == "no") {
      const std::string s64 = (long long)L.Ho * L.Wo <= 64 ? check<64>(L, cus) : "no";
      if (s64.compare(0, 2, "ok") != 0 && s64 != "no") s = "64 channels: " + s64;
      else if (s64.find("wide") != std::string::npos) s = s64;
    }
    puts(s.c_str());
  }
  return 0;
}
