// How gemm4w_tail_kernel deals out the work of adding up a tail tile's parts (gemm4w.h), also for the host.
//
// A unit is what one wave does: the 16 rows that wave w of the GEMM has of token block tt (32 tt + 16 (w >> 1) on) by 32 of its 128
// features (gate/up: 32 of its 64 outputs). A block takes four units that follow each other; its XCD is its index mod 8. With few
// rows only the first token blocks of each tile have any, so a unit's place in its tile turns with the tile: else those
// blocks fall to a few XCDs. Token block in the low bits of the block's index -> so, Linear of 128 rows in bf16, us: by
// 2560 x 10240 (40 tiles) 10.5 -> 7.7; by 2048 x 2048 (8 tiles) 6.0 -> 6.0, but the GEMM in front, which writes the parts, 18.8 -> 15.4 (the
// lines that it overwrites are then held by all XCDs' caches).
#pragma once

#if defined(__HIPCC__)
#define HDMOE_TAIL_HD __host__ __device__ __forceinline__
#else
#define HDMOE_TAIL_HD static inline
#endif

struct G4TailUnit { int q, w, tt; };

// 128 units per tile, gate/up 64. item: the block's index within the tile.
HDMOE_TAIL_HD G4TailUnit g4_tail_unit(bool swiglu, int item, int wave, int tile) {
  const int unit = item * 4 + wave, bits = swiglu ? 1 : 2;
  const int at = ((unit >> bits) + (swiglu ? 10 : 5) * tile) & 31;   // by 5 blocks (a block holds two places of gate/up)
  return {unit & ((1 << bits) - 1), at & 3, at >> 2};
}

// Token blocks of which wave w of the GEMM has rows, in a tile of `rows`: those are what it leaves of a part. A Linear of up to 16 rows by
// 2560 x 10240 in bf16, whole blocks of 32 rows -> so: 17.3 -> 16.6 us (240 parts of 16 KiB instead of 32).
HDMOE_TAIL_HD int g4_part_blocks(int rows, int w) { return (rows - (w >> 1) * 16 + 31) >> 5; }

// Which tile is item i of a block (`slot` of XCD `xcd`, 32 blocks on each of 8): of `longs` tiles round by round over the blocks and
// `shorts` behind them (gemm4w.h, g4_two_lengths; 0 = tiles of one length). A last round of a few tiles is spread over the XCDs: consecutive
// blocks of it on the first ones, Linear of 80 tiles in fp8 34.2 us, so 30.2. tile < 0: none.
struct G4Place { bool is_short; int tile; };
HDMOE_TAIL_HD G4Place g4_place(int longs, int shorts, int light_rounds, int xcd, int slot, int i) {
  const int full = longs >> 8, left = longs & 255, share = (left + 7) >> 3;
  const int start = xcd * share < left ? xcd * share : left, heavies = left - start < share ? left - start : share;
  const bool heavy = slot < heavies;
  if (i < full) return {false, i * 256 + xcd * 32 + slot};
  if (heavy && i == full) return {false, full * 256 + start + slot};
  const int lights = 256 - left, j = i - full - (heavy ? 1 : 0);
  const int rank = xcd * 32 - start + slot - heavies;   // among the light blocks
  const int tile = heavy ? light_rounds * lights + j * 256 + lights + start + slot
                   : j < light_rounds ? j * lights + rank : light_rounds * lights + (j - light_rounds) * 256 + rank;
  return {true, tile < shorts ? tile : -1};
}

// Lists of tiles one behind the other, each dealt out to 8 XCDs in contiguous shares: the tiles in front of XCD `xcd`'s shares of all lists that
// end at tile `end` of the whole. Its share of the list from tile a to tile b starts at tile g4_dealt(b, xcd) - g4_dealt(a, xcd) of it. The
// shares of a list differ by at most one tile and so do the shares of all lists together; with each list cut in eighths by itself the odd tiles
// fell to the same XCDs, and a round of 250 parts of five groups left 33 to one of 32 blocks.
HDMOE_TAIL_HD int g4_dealt(int end, int xcd) { return (end >> 3) * xcd + ((end & 7) < xcd ? (end & 7) : xcd); }

// The m-tiles of bm rows that n segments of `rows` rows together are counted as: each a standard deviation above the mean, and no more than
// that many rows can make (four segments of 1024 rows: 7 of 256 rows, where each counted for itself would have two).
inline int g4_likely_tiles(int rows, int n, int bm) {
  const double mu = (double)rows / n;
  const int each = n * (((int)(mu + std::sqrt(mu)) + bm - 1) / bm), most = rows > n ? (rows - n) / bm + n : rows;
  return each < most ? each : most;
}

// The height of the tiles of a layer's down projection cut in pd / ps parts, `bm` or the next multiple of 32 with which n segments of `rows`
// rows together (g4_likely_tiles) and the shared expert's `rows_static` fit one round of 256 blocks (nt tiles along
// the features). Where it is not bm the device takes it if the segments' own tiles of bm rows are more than a round: the parts, and with them
// the bytes, are the same. fp8 layers of 4 experts in (2, 1) parts, 128-token tiles -> this, us, three experts above 256 rows (one
// input in seven at 512 tokens): 512 tokens 143 -> 135, 500 146 -> 133; fewer above 256 134.0 and 134.0, skewed 131.0 and 131.4. (Higher tiles whatever the
// segments: skewed 134.)
inline int g4_cut_height(int bm, int rows, int n, int rows_static, int pd, int ps, int nt) {
  while (bm < 256 && (g4_likely_tiles(rows, n, bm) * pd + (rows_static + bm - 1) / bm * ps) * nt > 256) bm += 32;
  return bm;
}

// The tiles of a segment on swiglu224_kernel (swiglu224.h): high ones of 224 rows, then low ones of 128. Styles: 0 high ones alone; 1 the last
// one low if its rows fit; 2 what is left after full ones in low ones; 3 the last full one's rows too; 4 low ones alone.
struct S224Mix { int highs, lows; };
HDMOE_TAIL_HD S224Mix s224_mix(int rows, int style, int high = 224) {
  const int full = (int)((unsigned)rows / (unsigned)high), rest = rows - full * high, all = full + (rest > 0 ? 1 : 0);
  const int keep = style == 0 || (style == 1 && rest > 128) ? all : style <= 2 ? full : style == 3 ? (full > 0 ? full - 1 : 0) : 0;
  const int left = rows - keep * high;
  return {keep, left > 0 ? (left + 127) >> 7 : 0};
}

// How the list of a launch is dealt out: highs in whole rounds of 256 blocks, what is left of them to as many blocks, lows to the other ones first
// (g4_place). What the longest block comes to, a high tile being S224_HIGH and a low one, 64 by its matrix instructions, 75. Beyond 16 rounds of
// high tiles there is nothing to gain.
constexpr int S224_HIGH = 100, S224_LOW = 75, S224_STYLES = 5, S224_TILES = 4096;
HDMOE_TAIL_HD int s224_cost(int highs, int lows, int low = S224_LOW) {
  const int full = highs >> 8, left = highs & 255, lights = 256 - left, light = full * S224_HIGH, heavy = light + (left > 0 ? S224_HIGH : 0);
  const int first = left > 0 ? 1 : 0, rest = lows - first * lights;
  if (rest <= 0) return heavy;
  const int q = rest >> 8, r = rest & 255;
  const int a = light + (first + q + (r > 0 ? 1 : 0)) * low, b = heavy + (left > 0 ? q + (r > lights ? 1 : 0) : 0) * low;
  return a > b ? a : b;
}

// The tiles of a launch; of the columns (tiles along the features): those with tiles of both heights, those with one low tile.
struct S224Tiles { int highs, lows, both, alone; };
HDMOE_TAIL_HD void s224_add(S224Tiles& t, const S224Mix& m, int cols) {
  t.highs += m.highs * cols;
  t.lows += m.lows * cols;
  t.both += m.highs > 0 && m.lows > 0 ? cols : 0;
  t.alone += m.lows == 1 ? cols : 0;
}
// The price of a choice of tiles. Low tiles behind high ones of the same columns read their weights again, and from memory where the launch's
// weights are more than about 100 MB: in 16ths of a hundredth of a high tile, 2 for such a column and 1 for a low tile (half of that where they
// are not), which is about 650 KB of weights at 6 TB/s; nothing from 8 rounds on where they stay in the memory-side cache (4 experts and a shared one,
// 4096 tokens, high tiles alone 475.5 and 475.4, this 469.8 and 471.4). Whole pass on this kernel, us, high tiles alone, lows where s224_cost alone gains,
// where this does (weights from memory): layers of 16 experts, 2048 tokens 424 480 424; 12 experts, 1600 321 362 323; 8 experts, 1100 233 251 234;
// width 4096, 950 332 350 335; 4 experts of 6912 and a shared one of 3584, 350 120 111 111, 500 139 138 130, 700 150 143 143, 1024 183 178 178; 6 experts,
// 950 211 209 203; dense branch, 32768 features, 768 rows 188 195 189; width 4096, 1300 rows 184 174 175; 1300 rows 87.3 85.0 85.5. Other tiles than
// high ones alone have to pay by a 32nd: the clock falls with the CUs that are busy (a 24th loses 1 % at 1300 and 2048 tokens).
HDMOE_TAIL_HD int s224_price(const S224Tiles& t, int shift) { return s224_cost(t.highs, t.lows) + ((2 * t.both + t.lows) >> shift); }
// whole: high tiles alone
HDMOE_TAIL_HD int s224_shift(int cols, int kbytes, int whole) {
  const long long bytes = (long long)cols * 256 * kbytes;
  return bytes <= (100ll << 20) ? 5 : bytes <= (200ll << 20) && whole >= 8 * 256 ? 8 : 4;
}
HDMOE_TAIL_HD bool s224_low_pays(int price, int whole, int margin = 32) { return price < whole - whole / margin; }
