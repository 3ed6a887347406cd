// Host-side export of comfyui_amd/csrc/tail_units.h for the CPU tests.
#include <cmath>

#include "../comfyui_amd/csrc/tail_units.h"
extern "C" void t_tail_unit(int swiglu, int item, int wave, int tile, int* out) {
  const G4TailUnit u = g4_tail_unit(swiglu != 0, item, wave, tile);
  out[0] = u.q; out[1] = u.w; out[2] = u.tt;
}
extern "C" int t_part_blocks(int rows, int w) { return g4_part_blocks(rows, w); }
extern "C" int t_place(int longs, int shorts, int light_rounds, int xcd, int slot, int i) {
  const G4Place p = g4_place(longs, shorts, light_rounds, xcd, slot, i);
  return p.tile < 0 ? -1 : p.tile * 2 + (p.is_short ? 1 : 0);
}
extern "C" int t_dealt(int end, int xcd) { return g4_dealt(end, xcd); }
extern "C" int t_likely_tiles(int rows, int n, int bm) { return g4_likely_tiles(rows, n, bm); }
extern "C" int t_cut_height(int bm, int rows, int n, int rows_static, int pd, int ps, int nt) { return g4_cut_height(bm, rows, n, rows_static, pd, ps, nt); }
extern "C" int t_mix(int rows, int style) { const S224Mix t = s224_mix(rows, style); return t.highs | t.lows << 16; }
extern "C" int t_s224_cost(int highs, int lows) { return s224_cost(highs, lows); }
