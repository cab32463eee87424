// Walks the tiles of dwpw_kernel and dwpw_chain_kernel on the host, with the kernels' own arithmetic (csrc/dwpw_geom.h): shapes that the
// entry points take but no tile fits, loads of another byte than the one meant or past an array, LDS places outside their range, activations that are
// left out or written twice, output pixels left out.
// Blocks on stdin, one a line: B C H W Co S chained bn_bytes cus.  One line out per block: "ok WAVES", "no" (refused) or what is wrong.
// A line "every": a tile for every shape that the entry points take, up to heights that only add tiles: the number of them.
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <string>
#include <vector>

#include "../../pulp_nn_amd/csrc/dwpw_geom.h"

// Loads whose range is checked by the lane's own offset: none may reach past its array, whatever the scalar offset adds.
static const char *loads(int C, int Co, int kp, int bn_bytes)
{
  for (int cf = 0; cf < Co / 16; cf++)
    for (int kt = 0; kt < (C + 63) / 64 + kp; kt++)
      for (int lane = 0; lane < 64; lane++) {
        const unsigned off = dwpw_w_lane(C, cf, lane, C <= 64);
        const DwPwWeight at = dwpw_w_slice(C, off, kt);
        const int row = lane >> 2, byte = 16 * ((lane & 3) ^ ((row >> 1) & 3)) + 64 * kt;
        if (at.off < (unsigned)(Co * C) ? byte >= C || (int)at.off + at.add != (16 * cf + row) * C + byte : byte < C || at.add) return "weights";
      }
  for (int form = 0; form < 8; form++) {
    const bool filter = form & 1, bias = form & 2, bn = form & 4;
    const DwPwPar at = dwpw_par(C, bn_bytes, filter);
    std::vector<int> seen[4] = {std::vector<int>(C), std::vector<int>(C * bn_bytes), std::vector<int>(C * bn_bytes), std::vector<int>(9 * C)};
    for (int to = 0; to < at.bytes; to += 1024) {
      const DwPwParPiece p = dwpw_par_piece(at, C, bn_bytes, bias, bn, to);
      for (int lane = 0; lane < 64; lane++) {
        if (16 * lane >= p.bytes) continue;
        for (int b = p.first + 16 * lane; b < p.first + 16 * lane + 16; b++)
          if (b >= (int)seen[p.array].size() || seen[p.array][b]++) return "parameters past their array";
      }
    }
    for (int array = 0; array < 4; array++)
      for (const int n : seen[array])
        if (n != (array == 0 ? bias : array == 3 ? filter : bn)) return "parameters left out";
  }
  return nullptr;
}

template <int W, int S>
static std::string check(int B, int C, int H, int Co, int chained, int bn_bytes, int cus)
{
  constexpr int WO = W / S;
  const int Ho = (H - 1) / S + 1;
  if (dwpw_refusal(B, C, W, Ho, WO, Co, S, chained ? 2 : 1, cus, bn_bytes)) return "no";
  DwPwTile g;
  if (!dwpw_shape(B, C, H, W, Ho, Co, S, chained, cus, bn_bytes, &g)) return "taken, but no tile fits";
  const int act_bytes = g.act_px * C, x_bytes = g.par_off - g.x_off, BM = g.act_px, KT = (C + 63) / 64;
  const int nblk = g.cf_per << g.lpxb, loading = chained ? g.waves : nblk < g.waves ? nblk : g.waves;  // blocks, waves with weights of their own
  if (g.lds > 160 * 1024 || g.x_off < act_bytes || (g.slabs - 1) * g.CS >= C || g.CS * g.slabs < C || (g.CS % 64 && C >= 64) || g.TR * WO > BM || BM > 64 << g.lpxb || BM % 16 ||
      g.TR % g.R || (g.whole && Ho % g.R) || (g.waves != 4 && g.waves != 8 && g.waves != 16) || (g.kp == 1 && C > 64) || (C < 64 && g.kp != 1) ||
      g.par_off + dwpw_par(C, bn_bytes, true).bytes > g.w_off || g.w_off + loading * g.kp * 1024 > g.lds || (g.cf_per << g.lsplit) * 16 < Co ||
      (chained && (g.lsplit || g.slabs != 1)))
    return "shape";
  // the multiply reads blocks of 64 pixels, also where there are fewer
  if ((C < 64 ? ((64 << g.lpxb) - 1) * C + C : (KT - 1) * 64 * g.act_px + ((64 << g.lpxb) - 1) * 64 + 64) > g.lds) return "operand past the LDS";
  if (const char *wrong = loads(C, Co < 128 ? Co : 128, g.kp, bn_bytes)) return wrong;
  const int cgs = g.CS / 16, ids[] = {0, g.tiles / 2, g.tiles - 1};
  long long outputs = 0;
  for (int t = 0; t < g.tiles; t++) outputs += dwpw_place<WO>(g, (unsigned)t).live;
  if (outputs != (long long)B * Ho * WO) return "output pixels: " + std::to_string(outputs);
  for (const int id : ids)
   for (int slab = 0; slab < g.slabs; slab += g.slabs > 1 ? g.slabs - 1 : 1) {
    const DwPwPlace at = dwpw_place<WO>(g, (unsigned)id);
    // input: every place of a pixel once, from the right byte
    std::vector<int> src(x_bytes / 16, -2);  // image pixel behind a 16-byte place: -1 padding
    const int chunks = dwpw_chunks<W>(g);
    for (int c = 0; c < chunks + 4096; c++) {
      const DwPwChunk k = dwpw_chunk<W, S>(g, at, c);
      if (c >= chunks) {
        if (k.off >= 0) return "load past the last chunk";
        continue;
      }
      if (k.lds < 0 || k.lds + 16 > x_bytes || k.lds % 16) return "input place";
      if (src[k.lds / 16] != -2) return "input place twice";
      src[k.lds / 16] = -1;
      if (k.off >= 0) {
        if (slab * g.CS + k.off % C >= C) continue;  // (past the last channel: nobody reads it)
        if (k.off + 16 > dwpw_rows_in(g) * W * C - slab * g.CS) return "input offset";
        const long long row = dwpw_first_row<S>(g, at) + k.off / C / W;
        if (row < 0 || row >= (long long)B * H) return "row outside the input";
        if (k.off % C != 16 * ((k.lds / 16) % (g.pitch / 16))) return "channel";
        src[k.lds / 16] = (int)(row * W + k.off / C % W);
      }
    }
    // depthwise stage: every activation of a real pixel once, from the rows and columns around it
    std::vector<unsigned char> act(act_bytes / 16);
    for (int it = 0; it < cgs * g.nst; it++) {
      const int st = (int)fastdiv((unsigned)it, g.d_n), cg = it - st * cgs, ch = slab * g.CS + 16 * cg;
      if (ch >= C) continue;
      for (int l16 = 0; l16 < 16; l16++)
        for (int kx = 0; kx < 3; kx++) {
          const DwPwLane n = dwpw_lane<W, S>(g, st, l16, kx);
          if (n.x < 0 || n.x + ((g.R - 1) * S + 3) * (W + 2) * g.pitch + 16 * cg + 16 > x_bytes) return "a strip's rows";  // (one row past the last)
          for (int r = 0; r < g.R; r++) {
            const int px = n.px + r * WO;
            if (px < 0 || px >= BM) return "pixel";
            const int p = dwpw_act(g, px, ch);
            if (p < 0 || p + 16 > act_bytes || p % 16) return "activation place";
            if (n.live && kx == 0 && act[p / 16]++) return "activation twice";
            if (!n.live || px >= at.live) continue;
            const int row = px / WO, y = g.whole ? row % Ho : at.oy0 + row, b = at.b0 + (g.whole ? row / Ho : 0), x = px % WO;
            for (int fy = 0; fy < 3; fy++) {
              const int iy = y * S - 1 + fy, ix = x * S - 1 + kx;
              const int want = iy >= 0 && iy < H && ix >= 0 && ix < W ? (b * H + iy) * W + ix : -1;
              if (src[(n.x + (r * S + fy) * (W + 2) * g.pitch + 16 * cg) / 16] != want) return "operand of another pixel";
            }
          }
        }
    }
    for (int px = 0; px < g.TR * WO; px++)
      for (int ch = slab * g.CS; ch < C && ch < (slab + 1) * g.CS; ch += 16)
        if (!act[dwpw_act(g, px, ch) / 16]) return "activation left out";
    if (chained)
      for (int px = 0; px < at.live; px++) {
        const int p = dwpw_next_x<W>(g, px);
        if (p < 0 || p + C > x_bytes || src[p / 16] != (at.b0 * H) * W + px) return "next block's input";
      }
  }
  return "ok " + std::to_string(g.waves) + (!chained && g.kp == 4 && dwpw_lean(g, cus) ? " lean" : "");
}

// every W, S, C and bn, heights up to three tiles of 256 pixels, and channels out and batches on both sides of every line
static std::string every()
{
  long long taken = 0;
  for (const int W : {64, 32, 16, 8, 4})
    for (int S = 1; S <= 2; S++)
      for (int C = 16; C <= 1024; C += C < 32 ? 16 : C < 64 ? 32 : 64)
        for (int H = 1; H <= 3 * 256 * S * S / W + 2; H++)
          for (const int Co : {16, 32, 48, 64, 96, 128, 192, 256, 320, 512, 1008, 1024, 2048, 4096})
            for (const int B : {1, 2, 3, 4, 15, 16, 60, 64, 128, 255, 256, 257, 512, 1000, 1024, 5000})
              for (int chained = 0; chained < (S == 1 && Co == 16 ? 2 : 1); chained++)
                for (const int bn : {4, 8})
                  for (const int cus : {64, 256}) {
                    const int Ho = (H - 1) / S + 1, co = chained ? C : Co;
                    if (dwpw_refusal(B, C, W, Ho, W / S, co, S, chained ? 2 : 1, cus, bn)) continue;
                    DwPwTile g;
                    taken++;
                    if (!chained && dwpw_small16(B, C, W, Ho, co, S, cus)) {  // dwpw16_kernel: items of two rows, constants of 1024 channels, 64 KB
                      const int split = dwpw16_split((B * Ho * 8 + DWPW16_PX - 1) / DWPW16_PX, co, cus);
                      if (Ho % 2 == 0 && C % 64 == 0 && ((co + 63) / 64 + split - 1) / split <= 16 && dwpw16_lds(C, co, split, bn) <= 65536) continue;
                    }
                    else if (dwpw_shape(B, C, H, W, Ho, co, S, chained, cus, bn, &g) && g.lds <= 160 * 1024) continue;
                    char what[256];
                    snprintf(what, sizeof what, "taken, but no tile fits: %d %d %d %d %d %d %d %d %d", B, C, H, W, co, S, chained, bn, cus);
                    return what;
                  }
  return std::to_string(taken);
}

int main()
{
  char line[256];
  while (fgets(line, sizeof line, stdin)) {
    if (!strncmp(line, "every", 5)) {
      puts(every().c_str());
      continue;
    }
    int B, C, H, W, Co, S, chained, bn, cus;
    if (sscanf(line, "%d %d %d %d %d %d %d %d %d", &B, &C, &H, &W, &Co, &S, &chained, &bn, &cus) != 9) return 1;
    std::string said = "no";
#define AT(w)                                                                 \
  if (W == w && S == 1) said = check<w, 1>(B, C, H, Co, chained, bn, cus);    \
  if (W == w && S == 2 && w > 4) said = check<w, w == 4 ? 1 : 2>(B, C, H, Co, chained, bn, cus);
    AT(64) AT(32) AT(16) AT(8) AT(4)
    puts(said.c_str());
    fflush(stdout);
  }
}
