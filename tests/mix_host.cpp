// Host-side export of the choice of tiles in comfyui_amd/csrc/tail_units.h for the CPU tests.
#include <cmath>

#include "../comfyui_amd/csrc/tail_units.h"
extern "C" int t_price(int highs, int lows, int both, int shift) {
  const S224Tiles t = {highs, lows, both, 0};
  return s224_price(t, shift);
}
extern "C" int t_shift(int cols, int kbytes, int whole) { return s224_shift(cols, kbytes, whole); }
// The style that tile_mix takes for G groups of rows[g] rows and cols[g] columns, the last `fixed` of them static: experts' * 5 + static one's.
extern "C" int t_style(int G, int fixed, const int* rows, const int* cols, int kbytes) {
  int best = 0, whole = 0, style = 0, all = 0, shift = 0;
  for (int g = 0; g < G; ++g) all += cols[g];
  for (int c = 0; c < S224_STYLES * S224_STYLES; ++c) {
    S224Tiles t = {0, 0, 0, 0};
    for (int g = 0; g < G; ++g) s224_add(t, s224_mix(rows[g], g < G - fixed ? c / S224_STYLES : c % S224_STYLES), cols[g]);
    if (c == 0) shift = s224_shift(all, kbytes, t.highs);
    const int p = s224_price(t, shift);
    if (c == 0) whole = best = p;
    else if (p < best) { best = p; style = c; }
  }
  return s224_low_pays(best, whole) ? style : 0;
}
// The same for gate/up on 16-bit activations, one group of `rows` rows and `cols` columns (gemm4w.h: G4_LOW_COST, G4_LOW_ALONE).
extern "C" int t_style16(int rows, int cols, int alone) {
  int best = 0, whole = 0, style = 0;
  for (int c = 0; c < S224_STYLES; ++c) {
    S224Tiles t = {0, 0, 0, 0};
    s224_add(t, s224_mix(rows, c, 256), cols);
    const int p = s224_cost(t.highs, t.lows, 78 + alone * t.alone / (t.lows > 1 ? t.lows : 1));
    if (c == 0) whole = best = p;
    else if (p < best) { best = p; style = c; }
  }
  return s224_low_pays(best, whole, 24) ? style : 0;
}
