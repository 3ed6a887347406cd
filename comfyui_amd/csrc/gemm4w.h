// Grouped GEMM with one wave per SIMD: the tile text of gen_gemm4w.py (tile of 256 weight rows by 256 tokens, or 128 to 224 in steps of
// 32 where fewer fill the rounds better; 4 waves, 512 registers each).
//
// Included by gemm.hip inside its unnamed namespace (uses GemmArgs, GemmGroup, swz, make_rsrc, lds_ptr_t). Same
// contraction, rounding points and LDS tile format as grouped_gemm_kernel; with bf16 activations weights may also be e4m3fn
// bytes (W8), converted to bf16 between LDS and the matrix cores.
//
// What bounds it: the matrix pipe at a clock that falls under it. Counters, MI355X: 24576 x 2048 x 8192 in fp16 has the pipe
// busy in 84 % of its cycles at 1.55 GHz (620 us); with e4m3fn weights, 8160 + 4080 rows by 2560, gate/up 77 % at 1.82 GHz and
// down 68 % at 1.88 GHz; with GELU 62 % at 1.59 GHz (the vector instructions of the activation and the stores in between); a
// last round with idle CUs (1024 tokens in bf16) 58 % at 1.93 GHz. No LDS bank conflicts, the address unit's queue full in 1 to
// 9 % of the wave cycles. A K step of a tile takes 1.36-1.5 us with every CU multiplying N(0,1) values and 0.95 us (the matrix pipe
// full) with most CUs idle. Against the 8-wave kernel with 32x32x16 MFMAs: half the fragment reads from LDS per product (128 x
// 128 per wave), the smaller MFMA (less energy), and no barrier that drains the pipe. bf16, M x N x K, 8-wave -> this kernel:
// 8192 x 8192 x 8192 917 -> 690 us, 16384 x 13824 x 2560 964 -> 805 us, 24576 x 2048 x 8192 654 -> 537 us (1.4-1.6 PFLOP/s).
// What the schedule hangs on: the 16 global->LDS loads of a wave and step are spread over the whole step (every 2 MFMAs: 730 us, every 6: 690 us at
// 8192^3; 4 waves times 16 lanes' worth of addresses each 16 cycles is all the address unit takes).
// GELU, 24576 x 8192 x 2048: 846 us in the 8-wave kernel's epilogue, 682 us hidden behind the next tile's K loop (560-585 us
// without activation; through the outputs themselves instead of a scratch buffer 732 us: the rows are written twice).
// fp8 (F8: e4m3fn activations and weights, no activation function): the same bytes and matrix cycles per K step as 16 bits, on
// v_mfma_f32_16x16x128_f8f6f4, whose fragments of a whole step (128 registers) are refilled quadrant by quadrant. M x N x K, 8-wave
// kernel with its assembly loop -> this one: 16384 x 13824 x 2560 511 -> 430 us (2.7 PFLOP/s), 16384 x 2560 x 6912 226 -> 213 us, 8192^3
// 374 -> 338 us, 16384^3 3076 -> 2637 us (3.3 PFLOP/s). One K step of one tile takes 0.88 us with few rows, a launch 8 us beside its steps.
#include "gemm4w_asm.inc"
#include "tail_units.h"

constexpr int G4_THREADS = 256;
constexpr int G4_BM = 256;                        // tokens per block tile
constexpr int G4_STAGE = 32768;
constexpr int G4_W_TILE = 65536;
constexpr int G4_TABLE = 131072;                  // LDS: [tok 0 | tok 1 | w 0 | w 1 | work item tables of the 4 waves | groups]
constexpr int G4_TABLE_ITEMS = 64;                // items a wave's lanes look up at a time
constexpr int G4_HEIGHTS = G4_TABLE + 4 * G4_TABLE_ITEMS * 16;   // 16 bytes per group, and 16 more (tile_mix)
constexpr int G4_SMEM = G4_HEIGHTS + (MAX_GROUPS + 1) * 16;
constexpr int G4_MIN_BLOCKS = 4;                  // least height of a tile, in token blocks of 32 rows
constexpr int G4_SCRATCH = 4 * 28 * 1024;         // GELU: bytes of scratch per block (28 pieces of 16 bytes per lane)
constexpr int G4_GELU_PAIRS = 16;                 // pairs of K steps a deferred activation needs to hide behind

// Gate/up on 16-bit activations ends its blocks' lists on low tiles of 128 rows as swiglu224.h does (tile_mix). A low one costs 78 of a whole one's
// 100, and with 16-bit weights 27 more where it is the only one of its segment: weights of more than the memory-side cache come from memory
// again for it alone (layer of 500 tokens, three experts a little over 256 rows: 202 -> 210 us without that). Up to 6 rounds of tiles; 3000
// tokens 593 -> 600 us. Tiles are as high as their rows need in any case. Before -> this, us: layers in bf16, 500 tokens 205 -> 197, 800 251 -> 244,
// 1000 285 -> 272, 1024 289 -> 283, 1500 370 -> 365; e4m3fn weights, 500 176 -> 166, 1000 264 -> 252, 1024 266 -> 255, 1800 404 -> 379; dense branch in bf16,
// 256 rows 98.7 -> 90.0, 400 101.9 -> 92.2, 1500 179 -> 170; e4m3fn weights 91.0 -> 77.9, 93.7 -> 78.6, 170 -> 157.
constexpr int G4_LOW_COST = 78, G4_LOW_ALONE = 27, G4_MIX_TILES = 6 * HDMOE_NUM_CU;
constexpr int G4_TAIL_MAX_PARTS = 12;
constexpr size_t G4_TAIL_BYTES = (size_t)HDMOE_NUM_CU * G4_BM * 256 * 4;  // fp32 sums of one tile per block

// Activations and weights: 16-bit alike, bf16 with e4m3fn weights that are converted, e4m3fn alike.
enum G4Type { G4_BF16, G4_F16, G4_W8, G4_F8 };
// Which 16 bytes of a K step's 128 go to the place of chunk c in LDS for v_mfma_f32_16x16x128_f8f6f4. Both fp8 matrix instructions add
// 16 products at a time to the fp32 sum (seen in what is lost beside a large product and its negative): the 16x16x128 one first the
// lower 16 bytes of every 16 lanes, then the upper ones; the 8-wave kernels' 32x32x64 the same way in its two groups of 32 bytes each,
// which takes the step's chunks as 0 2 1 3 4 6 5 7. In this order the sums are the same bit for bit; in ascending order one output in 1e4
// of operands with every exponent differed in a rounding. On the way into LDS it costs nothing; as an order of the reads it made
// bank conflicts (layer of 8192 tokens 836 -> 868 us).
__device__ __forceinline__ int f8_chunk(int c) { return (c & 4) | (c & 1) << 1 | (c >> 1 & 1); }

// What becomes of a tile's sums.
enum G4Epi { G4_PLAIN, G4_BIAS, G4_GELU, G4_SWIGLU, G4_PARTIAL };

typedef float v32f __attribute__((ext_vector_type(32)));
typedef int v32i __attribute__((ext_vector_type(32)));
typedef int v16i __attribute__((ext_vector_type(16)));

// positions in the context registers v[96:127] (gen_gemm4w.py)
enum { G4_TOK_ADDR = 0, G4_W_ADDR = 2, G4_TOK_VOFF = 4, G4_W_VOFF = 12, G4_OUT_VOFF = 20, G4_GATHER_VOFF = 22,
       G4_BIAS_VOFF = 23, G4_DEF_LD = 24, G4_DEF_ST = 25, G4_SCR_VOFF = 26 };

#define G4_A10(b) "a" #b "0", "a" #b "1", "a" #b "2", "a" #b "3", "a" #b "4", "a" #b "5", "a" #b "6", "a" #b "7", "a" #b "8", "a" #b "9"
#define G4_V10(b) "v" #b "0", "v" #b "1", "v" #b "2", "v" #b "3", "v" #b "4", "v" #b "5", "v" #b "6", "v" #b "7", "v" #b "8", "v" #b "9"
// what a tile's statement overwrites beside its operands: accumulators, slice 1 fragments, work registers, resources
#define G4_CLOBBER_V                                                                                                 \
  "memory", "scc", "v34", "v35", "v36", "v37", "v38", "v39", G4_V10(4), G4_V10(5), G4_V10(6), "v70",    \
      "v71", "v192", "v193", "v194", "v195", "v196", "v197", "v198", "v199", G4_V10(20), G4_V10(21), G4_V10(22),      \
      G4_V10(23), G4_V10(24), "v250", "v251", "v252", "v253", "v254", "v255"
#define G4_CLOBBER                                                                                                   \
  G4_CLOBBER_V, "s64", "s65", "s66", "s67", "s68", "s69", "s70", "s71", "s72", "s73", "s74", "s75", G4_A10(),         \
      G4_A10(1), G4_A10(2), G4_A10(3), G4_A10(4), G4_A10(5), G4_A10(6), G4_A10(7), G4_A10(8), G4_A10(9), G4_A10(10),  \
      G4_A10(11), G4_A10(12), G4_A10(13), G4_A10(14), G4_A10(15), G4_A10(16), G4_A10(17), G4_A10(18), G4_A10(19),     \
      G4_A10(20), G4_A10(21), G4_A10(22), G4_A10(23), G4_A10(24), "a250", "a251", "a252", "a253", "a254", "a255"

// A tile by its index inside a group of mtiles x ntiles: bands of GROUP_M m-tiles, a short remainder joins the last one.
__device__ __forceinline__ void g4_raster(int L, int mtiles, int ntiles, int& m, int& n) {
  const int nbands = max(1, (mtiles + GROUP_M / 2) / GROUP_M);
  const int band = min(tile_div(L, GROUP_M * ntiles), nbands - 1);
  const int first_m = band * GROUP_M;
  const int gm = band == nbands - 1 ? mtiles - first_m : GROUP_M;
  const int within = L - band * (GROUP_M * ntiles);
  n = tile_div(within, gm);
  m = first_m + within - n * gm;
}

// What is left when every block has had the same number of whole tiles (`rounds`): `tiles` of them, each cut along K into
// `parts` equal parts for blocks of their own; gemm4w_tail_kernel adds the parts up. parts = 1: not cut.
struct G4Tail { int rounds, tiles, parts; };

// Costs in units of one pair of K steps (2.0 us with most of the chip idle): a part takes its share of the pairs; leaving the
// fp32 parts and adding them up costs a second launch (9 us) and their bytes written and read again (256 KiB per part of
// a full tile, about 6 TB/s: 0.04 pairs). A cut has to pay by a seventh. With and without cuts: Hunyuan3D block of 128 tokens
// 260 and 326 us, 1000 tokens 313 and 335 us, 8192 tokens 1553 and 1587 us, bf16 layer of 400 tokens 188 and 211 us; the model is
// too hopeful near the line: bf16 layer of 1024 tokens 300 and 292 us. pairs: K step pairs of a tile; padding: rows that the
// tiles have beyond those of their segments, over all tiles.
// Both kernels of a launch work the plan out for themselves and have to agree, so it is integers throughout: costs in 25600ths
// of a pair (100ths, times the 256 rows of a tile).
__host__ __device__ inline G4Tail g4_plan_tail(int total, int blocks, int pairs, int min_pairs, int padding) {
  G4Tail t = {total / blocks, total % blocks, 1};
  if (t.tiles == 0) return t;
  const int fill = G4_BM - padding / total;   // rows of the average tile
  int best = 85 * G4_BM * pairs;
  for (int p = 2; p <= G4_TAIL_MAX_PARTS && p * t.tiles <= blocks && pairs / p >= min_pairs; ++p) {
    const int cost = 100 * G4_BM * ((pairs + p - 1) / p) + 450 * G4_BM + 4 * fill * (p * t.tiles);
    if (cost < best) { best = cost; t.parts = p; }
  }
  return t;
}

// The plan of a launch, from the segment sizes on the device; also its number of tiles.
template <G4Type TY, int FEAT>
__device__ __forceinline__ G4Tail g4_tail_of(const GemmArgs& args, const Segments& seg, int blocks) {
  int total = 0, padding = 0;
  for (int g = 0; g < args.G; ++g) {
    const int rows = seg.rows(g), nt = seg.ntiles(g, FEAT), mt = (rows + G4_BM - 1) / G4_BM;
    total += mt * nt;
    padding += (mt * G4_BM - rows) * nt;
  }
  if (args.tail == nullptr || total == 0) return {total / blocks, total % blocks, 1};
  return g4_plan_tail(total, blocks, seg.bytes(0) / (2 * BK), TY == G4_W8 ? 3 : 2, padding);
}

// Tiles of fewer rows, where the tiles left over are not cut. A segment of U blocks of 32 rows takes ceil(U / cap) m-tiles for a
// cap of 4 to 8 blocks, all as high as its blocks need (the last one may be lower). The groups follow each other from the highest
// tiles to the lowest and go round by round over the grid, so that a round takes what its first tile does.
// Costs as in g4_plan_tail, a pair of K steps of 8 blocks being 100 (a step costs a little beside its MFMAs: 13 us less for a round of
// 5 blocks of K = 2048, where 17 would be in proportion), and 150 for a tile's start and end. Lower tiles have to pay by a
// twelfth: the model takes a round with idle CUs for as long as a full one, but it has the higher clock. Whole tiles -> this: Linears in bf16,
// 700 x 2560 x 10240 48.8 -> 38.8 us (240 tiles of 4 blocks for 120), 1700 x 2560 x 2560 48.1 -> 38.1, 3300 x 2560 x 2560 49.2 -> 43.0; with
// e4m3fn weights 50.0 -> 37.4, 49.0 -> 36.8, 50.1 -> 42.3; Hunyuan3D block of 1250 tokens 367 -> 330, 1500 358 -> 348 (375 rows per expert:
// 3 rounds of 8 or of 6 to 7 blocks); in fp8, 8-wave kernel on 192-token tiles -> this, without the cast: 4480 x 2560 x 2560 31.6 -> 28.7, 2000 25.8 ->
// 21.8, 1000 22.0 -> 19.0, 2000 x 2560 x 10240 52.7 -> 46.9, 9000 x 2048 x 2048 44.0 -> 36.2, 193 x 4096 x 2560 28.4 -> 23.4; fp8 tiles are as
// high as their rows need without a cap too. Not for SWIGLU, whose two halves of the weights every further m-tile reads again (1300 tokens
// in bf16 361 -> 367 us, 1024 tokens 294 -> 298): it has whole tiles and low ones behind them (tile_mix). More than 24 rounds: one is not worth the search.
constexpr int G4_TILE_COST = 150, G4_CAP_ROUNDS = 24;
__host__ __device__ __forceinline__ int g4_div(int a, int b) {
#if defined(__HIP_DEVICE_COMPILE__)
  return tile_div(a, b);
#else
  return a / b;
#endif
}
struct G4Heights { int mt, height; };
__host__ __device__ __forceinline__ G4Heights g4_heights(int rows, int cap) {
  const int units = (rows + 31) >> 5, mt = g4_div(units + cap - 1, cap);
  return {mt, max(g4_div(units + mt - 1, max(mt, 1)), G4_MIN_BLOCKS)};
}

// What a cap comes to; rows(g), ntiles(g): the rows of group g, its tiles along the features.
template <class Rows, class Tiles>
__host__ __device__ __forceinline__ int g4_cap_cost(int G, int pairs, const Rows& rows, const Tiles& ntiles, int blocks, int cap) {
  constexpr int PAIR[5] = {58, 70, 80, 90, 100};
  int n[5] = {0, 0, 0, 0, 0};                  // tiles of each height
  for (int g = 0; g < G; ++g) {
    const int have = rows(g);
    if (have <= 0) continue;
    const G4Heights t = g4_heights(have, cap);
    const int tiles = t.mt * ntiles(g);
#pragma unroll
    for (int h = 0; h < 5; ++h) n[h] += t.height == h + G4_MIN_BLOCKS ? tiles : 0;
  }
  int cost = 0, at = 0;
#pragma unroll
  for (int h = 4; h >= 0; --h) {
    const int to = at + n[h];
    cost += ((to + blocks - 1) / blocks - (at + blocks - 1) / blocks) * (pairs * PAIR[h] + G4_TILE_COST);
    at = to;
  }
  return cost;
}

// Rounds of whole tiles that lower ones may replace, 0 = none.
__host__ __device__ __forceinline__ int g4_cap_rounds(const G4Tail& tail) {
  const int whole = tail.rounds + (tail.tiles > 0 ? 1 : 0);
  return tail.parts > 1 || whole > G4_CAP_ROUNDS ? 0 : whole;
}

// The cheapest cap if it is worth leaving `whole` rounds of whole tiles for, else 0. cost: of a cap.
template <class Cost>
__host__ __device__ __forceinline__ int g4_best_cap(int whole, int pairs, const Cost& cost) {
  const int old = whole * (100 * pairs + G4_TILE_COST);
  int best = 0, limit = old - old / 12;
#pragma unroll
  for (int cap = G4_BM / 32; cap >= G4_MIN_BLOCKS; --cap) {
    const int v = cost(cap);
    if (v < limit) { limit = v; best = cap; }
  }
  return best;
}

// On the device lane i works out cap 4 + i.
template <int FEAT>
__device__ __forceinline__ int g4_cap(const GemmArgs& args, const Segments& seg, const G4Tail& tail, int blocks, int lane) {
  const int whole = g4_cap_rounds(tail);
  if (whole == 0) return 0;
  const int mine = g4_cap_cost(args.G, seg.bytes(0) / (2 * BK), [&](int g) { return seg.rows(g); }, [&](int g) { return seg.ntiles(g, FEAT); }, blocks,
                               G4_MIN_BLOCKS + min(lane, 4));
  return g4_best_cap(whole, seg.bytes(0) / (2 * BK), [&](int cap) { return __builtin_amdgcn_readlane(mine, cap - G4_MIN_BLOCKS); });
}

// Tiles of two lengths (a layer's down projection: the experts' K and the shared expert's, args.spread). The long ones go round by round
// over the blocks; those without one in the last of these rounds (light blocks) take short ones first, as many rounds of them as fit beside a
// long one, and what is left goes round by round over all, light blocks first (g4_place). Groups are long or short by args.spread.
// The caps are those of the shortest longest block; others than whole tiles have to pay by a twelfth in fp8, an eighth in 16 bits (two rounds
// of 7 blocks and more, 90 % of the cost, take as long: the clock falls with the CUs that are busy). Layers of 4 experts with K = 6912 and a
// shared one with 3584, every XCD an eighth of every group -> this, us: fp8, 2600 tokens 319 -> 311, 3000 357 -> 344, 3500 405 -> 398, 4096 460 ->
// 450, 4500 517 -> 499, 5000 549 -> 534; e4m3fn weights in bf16, 2100 491 -> 438, 3000 616 -> 588, 4080 the same; bf16, 2100 520 -> 468, 3000
// 655 -> 637. With more than 448 long tiles the eighths are better or equal (fp8 8192 tokens 821 -> 826, 12000 1167 -> 1177).
struct G4Two { int cost, light_rounds; };
template <class Segs>
__host__ __device__ __forceinline__ G4Two g4_two_lengths(const Segs& seg, int G, int spread, int feat, int cap_long, int cap_short) {
  constexpr int PAIR[5] = {58, 70, 80, 90, 100}, BLOCKS = HDMOE_NUM_CU;
  int n[5] = {0, 0, 0, 0, 0}, shorts = 0, top = 0, pairs_long = 0, pairs_short = 0;
  for (int g = 0; g < G; ++g) {
    const bool is_short = seg.dynamic(g) == (spread < 0);
    (is_short ? pairs_short : pairs_long) = seg.bytes(g) / (2 * BK);
    const G4Heights t = g4_heights(seg.rows(g), is_short ? cap_short : cap_long);
    const int tiles = t.mt * seg.ntiles(g, feat);
    if (is_short) { shorts += tiles; top = max(top, t.mt > 0 ? t.height : 0); }
#pragma unroll
    for (int h = 0; h < 5; ++h) n[h] += !is_short && t.height == h + G4_MIN_BLOCKS ? tiles : 0;
  }
  int heavy = 0, last = 0, at = 0, each = G4_TILE_COST;
#pragma unroll
  for (int h = 4; h >= 0; --h) {
    const int to = at + n[h], started = (to + BLOCKS - 1) / BLOCKS - (at + BLOCKS - 1) / BLOCKS, tile = pairs_long * PAIR[h] + G4_TILE_COST;
    heavy += started * tile;
    last = started > 0 ? tile : last;
    each += top == h + G4_MIN_BLOCKS ? pairs_short * PAIR[h] : 0;
    at = to;
  }
  const int left = at % BLOCKS, lights = BLOCKS - left, light = left > 0 ? heavy - last : heavy;
  const int light_rounds = left > 0 ? g4_div(last, each) : 0;
  const int rest = shorts - light_rounds * lights;
  if (rest <= 0) return {heavy, light_rounds};
  const int q = rest / BLOCKS, r = rest % BLOCKS;
  return {max(light + (light_rounds + q + (r > 0 ? 1 : 0)) * each, heavy + (q + (r > lights ? 1 : 0)) * each), light_rounds};
}

// On the host, where the rows of a launch are known; -1: the device has to find it. On the device -> on the host, Linears in bf16, us: 700 rows
// by 2560 x 10240 38.5 -> 37.5, 1500 57.8 -> 57.1; 6000 by 2560 x 2560 (whole tiles) 57.8 -> 57.0.
inline int g4_host_cap(const GemmArgs& args, int feat, int min_pairs, int blocks) {
  int total = 0, padding = 0;
  for (int g = 0; g < args.G; ++g) {
    if (args.g[g].row_begin < 0) return -1;
    const int rows = args.g[g].row_end - args.g[g].row_begin, mt = (rows + G4_BM - 1) / G4_BM, nt = args.g[g].n_out / feat;
    total += mt * nt;
    padding += (mt * G4_BM - rows) * nt;
  }
  const int pairs = args.g[0].kbytes / (2 * BK);
  const G4Tail tail = args.tail == nullptr || total == 0 ? G4Tail{total / blocks, total % blocks, 1} : g4_plan_tail(total, blocks, pairs, min_pairs, padding);
  const int whole = g4_cap_rounds(tail);
  if (whole == 0) return 0;
  auto rows = [&](int g) { return args.g[g].row_end - args.g[g].row_begin; };
  return g4_best_cap(whole, pairs, [&](int cap) { return g4_cap_cost(args.G, pairs, rows, [&](int g) { return args.g[g].n_out / feat; }, blocks, cap); });
}

// High and low tiles of the segments (tail_units.h), lane g looking after group g: leaves [segment begin, end, high m-tiles | low ones << 16, tiles
// along the features] of each group and [rounds of high tiles, high tiles beyond, low tiles] behind them in `groups` (LDS, every wave the
// same) and says whether there are low ones. F8: tiles of swiglu224_kernel; W8: of gemm4w_kernel with one-byte weights. most: high tiles at which low
// ones are looked for.
template <bool F8, bool W8>
__device__ __forceinline__ bool tile_mix(const Segments& segs, int G, int lane, int high, int feat, int most, v4i* groups) {
  const int rows = segs.re - segs.rb, nt = (int)((unsigned)segs.n_out / (unsigned)feat), whole = s224_mix(rows, 0, high).highs * nt;
  int highs = 0, lows = 0, style = 0, cols = 0;
  for (int g = 0; g < G; ++g) {
    highs += __builtin_amdgcn_readlane(whole, g);
    cols += __builtin_amdgcn_readlane(nt, g);
  }
  if (highs <= most) {   // lane i: style i / 5 of the experts and i % 5 of the static group
    const int c = min(lane, S224_STYLES * S224_STYLES - 1), of_dyn = c * 13 >> 6, of_fix = c - 5 * of_dyn;
    S224Tiles tiles = {0, 0, 0, 0};
    for (int g = 0; g < G; ++g)
      s224_add(tiles, s224_mix(__builtin_amdgcn_readlane(rows, g), segs.dynamic(g) ? of_dyn : of_fix, high), __builtin_amdgcn_readlane(nt, g));
    int price;
    if constexpr (F8) price = s224_price(tiles, s224_shift(cols, segs.bytes(0), highs));
    else price = s224_cost(tiles.highs, tiles.lows, G4_LOW_COST + (W8 ? 0 : tile_div(G4_LOW_ALONE * tiles.alone, max(tiles.lows, 1))));
    const int mine = price << 5 | c;
    const int first = __builtin_amdgcn_readlane(mine, 0);
    int best = first;
#pragma unroll
    for (int k = 1; k < S224_STYLES * S224_STYLES; ++k) best = min(best, __builtin_amdgcn_readlane(mine, k));
    if (F8 ? s224_low_pays(best >> 5, first >> 5) : s224_low_pays(best >> 5, first >> 5, 24)) {
      const int pick = best & 31, pick_dyn = pick * 13 >> 6;
      style = segs.fixed >> lane & 1 ? pick - 5 * pick_dyn : pick_dyn;
      highs = __builtin_amdgcn_readlane(tiles.highs, pick);
      lows = __builtin_amdgcn_readlane(tiles.lows, pick);
    }
  }
  const S224Mix t = s224_mix(rows, style, high);
  v4i e = {segs.rb, segs.re, t.highs | t.lows << 16, nt};
  if (lane == MAX_GROUPS) e = v4i{highs / HDMOE_NUM_CU, highs % HDMOE_NUM_CU, lows, 0};
  if (lane <= MAX_GROUPS) groups[lane] = e;
  return lows > 0;
}
// Item i of a block's list: g < 0: none.
struct MixedTile { int g, row0, rows, n; bool low; };
__device__ __forceinline__ MixedTile mixed_tile(const v4i* groups, int G, int lane, int xcd, int slot, int i, int high) {
  constexpr int nslots = HDMOE_NUM_CU / HDMOE_NUM_XCD;
  const v4i mine = groups[min(lane, MAX_GROUPS)];
  const int rounds = __builtin_amdgcn_readlane(mine.x, MAX_GROUPS), left = __builtin_amdgcn_readlane(mine.y, MAX_GROUPS),
            lows = __builtin_amdgcn_readlane(mine.z, MAX_GROUPS);
  // whole rounds: an XCD's blocks take a contiguous eighth of the list
  const G4Place at = g4_place(left, lows, left > 0 ? 1 : 0, xcd, slot, i - rounds);
  const bool low = i >= rounds && at.is_short;
  int rem = i < rounds ? xcd * (rounds * nslots) + slot + i * nslots : low ? at.tile : rounds * HDMOE_NUM_CU + at.tile;
  int g_at = -1, mtiles = 1, ntiles = 1, L = 0, rb_at = 0, re_at = 0;
  for (int g = 0; g < G; ++g) {
    const int rb = __builtin_amdgcn_readlane(mine.x, g), re = __builtin_amdgcn_readlane(mine.y, g), mts = __builtin_amdgcn_readlane(mine.z, g),
              nt = __builtin_amdgcn_readlane(mine.w, g), mt = low ? mts >> 16 : mts & 0xffff;
    if (rem >= 0 && g_at < 0) {
      if (rem < mt * nt) { g_at = g; mtiles = mt; ntiles = nt; L = rem; rb_at = rb + (low ? (mts & 0xffff) * high : 0); re_at = re; }
      else rem -= mt * nt;
    }
  }
  MixedTile t = {g_at, 0, 0, 0, low};
  if (g_at >= 0) {
    int m;
    g4_raster(L, mtiles, ntiles, m, t.n);
    const int height = low ? 128 : high;
    t.row0 = rb_at + m * height;
    t.rows = min(re_at - t.row0, height);
  }
  return t;
}

template <G4Type TY, int EPI>
__global__ __launch_bounds__(G4_THREADS) __attribute__((amdgpu_waves_per_eu(1, 1))) void gemm4w_kernel(const GemmArgs args) {
#if defined(__HIP_DEVICE_COMPILE__)   // the host pass drops the stub of a kernel whose register operands it cannot parse
  constexpr bool F16 = TY == G4_F16, W8 = TY == G4_W8, F8 = TY == G4_F8;
  constexpr bool SWIGLU = EPI == G4_SWIGLU;
  constexpr bool HAS_BIAS = EPI == G4_BIAS || EPI == G4_GELU;
  constexpr int FEAT = SWIGLU ? 128 : 256;
  static_assert(!F8 || (EPI != G4_SWIGLU && EPI != G4_GELU), "fp8: plain contractions");
  constexpr int OUT_BYTES = EPI == G4_PARTIAL ? 4 : 2;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wq = wave & 1, wt = wave >> 1;
  auto sgpr = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  // A constant in a register of its own. The compiler otherwise takes constants out of the initial value of a register tuple,
  // spills the whole tuple and reloads it between the statements below without waiting for the parts that it does not use:
  // they would arrive while a statement has those registers in use.
  auto own = [](int v) { asm volatile("" : "+s"(v)); return v; };

  // ---- work items: as grouped_gemm_kernel's tiles --------------------------------------------------------------
  // A wave's lanes look its block's next 64 items up at once and leave them in LDS (one by one, the decoding is a serial
  // chain of integer divisions that the matrix cores would wait for at every tile).
  const Segments segs(args, lane);
  int plan_idx = 0;
  if (EPI == G4_PARTIAL && args.plan.n > 1) {
    int mt_dyn = 0, mt_static = 0;
    for (int g = 0; g < args.G; ++g) {
      int rb, re;
      segs.get(g, rb, re);
      (segs.dynamic(g) ? mt_dyn : mt_static) += (re - rb + args.plan.bm - 1) / args.plan.bm;
    }
    plan_idx = hdmoe_plan_pick(args.plan, mt_dyn, mt_static, segs.ntiles(0, FEAT));
  }
  int bm = EPI == G4_PARTIAL && F8 ? args.plan.bm : G4_BM;   // rows of a tile that is not capped
  if (EPI == G4_PARTIAL && F8 && args.plan.bm_else > 0) {    // (the plan has one entry)
    const int parts = segs.fixed >> lane & 1 ? args.plan.ps[0] : args.plan.pd[0];
    const int mine = tile_div(segs.re - segs.rb + bm - 1, bm) * (segs.n_out / FEAT) * parts;
    int tiles = 0;
    for (int g = 0; g < args.G; ++g) tiles += __builtin_amdgcn_readlane(mine, g);
    if (tiles > HDMOE_NUM_CU) bm = args.plan.bm_else;
  }
  auto parts_of = [&](int g) {
    return EPI != G4_PARTIAL ? 1 : segs.dynamic(g) ? args.plan.pd[plan_idx] : args.plan.ps[plan_idx];
  };
  // Whole rounds of tiles: each XCD (block ids congruent mod 8) takes a contiguous eighth of the tile list and its blocks
  // take consecutive tiles, so the CUs of an XCD share operand tiles in their L2. The remainder (tail): the parts of
  // one K range before those of the next, again consecutive inside an XCD. Groups of different K (`spread`) or cut by the
  // caller's plan: every XCD takes its eighth of every group, longest tiles first.
  const int xcd = blockIdx.x % HDMOE_NUM_XCD, slot = blockIdx.x / HDMOE_NUM_XCD;
  constexpr int nslots = HDMOE_NUM_CU / HDMOE_NUM_XCD;   // the grid is one block per CU
  const G4Tail tail = g4_tail_of<TY, FEAT>(args, segs, HDMOE_NUM_CU);
  int cap = 0, cap_short = 0, light_rounds = 0;
  if (EPI != G4_PARTIAL && !SWIGLU) {
    if (args.cap >= 0) {
      cap = args.cap;
    } else if (args.spread == 0) {
      cap = sgpr(g4_cap<FEAT>(args, segs, tail, HDMOE_NUM_CU, lane));
    } else {   // lane i works out caps 4 + i / 5 and 4 + i % 5
      const int c = min(lane, 24), c5 = c * 13 >> 6;
      const G4Two mine = g4_two_lengths(segs, args.G, args.spread, FEAT, G4_MIN_BLOCKS + c5, G4_MIN_BLOCKS + c - 5 * c5);
      int best = 24, limit = __builtin_amdgcn_readlane(mine.cost, 24);
      limit -= limit / (F8 ? 12 : 8);
#pragma unroll
      for (int k = 0; k < 24; ++k) {
        const int v = __builtin_amdgcn_readlane(mine.cost, k);
        if (v < limit) { limit = v; best = k; }
      }
      cap = sgpr(G4_MIN_BLOCKS + best / 5);
      cap_short = sgpr(G4_MIN_BLOCKS + best % 5);
      light_rounds = __builtin_amdgcn_readlane(mine.light_rounds, best);
    }
  }
  auto is_short = [&](int g) { return args.cap < 0 && args.spread != 0 && segs.dynamic(g) == (args.spread < 0); };
  // cap > 0: lane g looks up where group g comes among those of its length in the order of heights: [first tile, tiles, height, m-tiles]
  v4i* const heights = reinterpret_cast<v4i*>(smem + G4_HEIGHTS);
  if (cap > 0) {
    v4i e = {0, 0, 0, 0};
    for (int g = 0; g < args.G; ++g) {
      int rb, re;
      segs.get(g, rb, re);
      if (re > rb && lane == g) {
        const G4Heights t = g4_heights(re - rb, is_short(g) ? cap_short : cap);
        e = v4i{0, t.mt * segs.ntiles(g, FEAT), t.height, t.mt};
      }
    }
    for (int k = 0; k < args.G; ++k) {
      const int h = __builtin_amdgcn_readlane(e.z, k), tiles = __builtin_amdgcn_readlane(e.y, k);
      const bool other = args.cap < 0 && args.spread != 0 && segs.dynamic(k) != !(segs.fixed >> lane & 1);
      if (!other && (h > e.z || (h == e.z && k < lane))) e.x += tiles;
    }
    if (lane < args.G) heights[lane] = e;   // every wave the same
  }
  bool mixed = false;
  if constexpr (SWIGLU) {
    if (tail.parts == 1) mixed = tile_mix<false, W8>(segs, args.G, lane, G4_BM, FEAT, G4_MIX_TILES, heights);
  }
  v4i* const table = reinterpret_cast<v4i*>(smem + G4_TABLE) + wave * G4_TABLE_ITEMS;
  auto fill_table = [&](int base) {
    const int i = base + lane;
    if (SWIGLU && mixed) {
      const MixedTile t = mixed_tile(heights, args.G, lane, xcd, slot, i, G4_BM);
      v4i e = {-1, 0, 0, 0};
      if (t.g >= 0) e = v4i{t.g | t.rows << 16, t.row0, t.n, segs.bytes(0) / BK << 16};
      table[lane] = e;
      return;
    }
    if (cap > 0) {
      int longs = 0, shorts = 0;
      for (int g = 0; g < args.G; ++g) (is_short(g) ? shorts : longs) += sgpr(heights[g].y);
      const G4Place at = g4_place(longs, shorts, light_rounds, xcd, slot, i);
      const int L = at.tile;
      v4i e = {-1, 0, 0, 0};
      for (int g = 0; g < args.G; ++g) {
        const v4i t = heights[g];
        const int first = sgpr(t.x), tiles = sgpr(t.y), rows = sgpr(t.z) * 32, mtiles = sgpr(t.w);
        const int nt = segs.ntiles(g, FEAT), kt = segs.bytes(g) / BK;
        int rb, re, m, n;
        segs.get(g, rb, re);
        if (L < first || L >= first + tiles || is_short(g) != at.is_short) continue;
        g4_raster(L - first, mtiles, nt, m, n);
        const int row0 = rb + m * rows;
        e = v4i{g | min(re - row0, rows) << 16, row0, n, kt << 16};
      }
      table[lane] = e;
      return;
    }
    const bool eighths = EPI == G4_PARTIAL || args.spread != 0;   // every group cut in eighths
    int rem = slot + i * nslots, tail_part = 0, tail_slot = 0;
    bool some = true;
    if (!eighths) {
      if (i < tail.rounds) {
        rem = xcd * (tail.rounds * nslots) + slot + i * nslots;
      } else {
        const int units = tail.tiles * tail.parts, chunk = (units + HDMOE_NUM_XCD - 1) / HDMOE_NUM_XCD;
        const int w = xcd * chunk + slot;
        some = i == tail.rounds && slot < chunk && w < units;
        tail_part = some ? tile_div(w, tail.tiles) : 0;
        const int t = some ? w - tail_part * tail.tiles : 0;
        rem = tail.rounds * HDMOE_NUM_CU + t;
        tail_slot = tail.parts > 1 ? 1 + t * tail.parts + tail_part : 0;
      }
    }
    int g_at = -1, mtiles = 1, ntiles = 1, L = 0, rb_at = 0, re_at = 0, parts = 1, kt = 0, end = 0;
    for (int k = 0; k < args.G; ++k) {
      const int g = args.spread < 0 ? args.G - 1 - k : k;
      int rb, re;
      segs.get(g, rb, re);
      const int mt = EPI == G4_PARTIAL && F8 ? tile_div(re - rb + bm - 1, bm) : (re - rb + G4_BM - 1) / G4_BM, nt = segs.ntiles(g, FEAT), np = parts_of(g);
      const int from = end;
      end += mt * nt * np;
      const int lo = eighths ? g4_dealt(end, xcd) - g4_dealt(from, xcd) : 0;
      const int hi = eighths ? g4_dealt(end, xcd + 1) - g4_dealt(from, xcd + 1) : end - from;
      if (some && g_at < 0) {
        if (rem < hi - lo) { g_at = g; mtiles = mt; ntiles = nt; L = lo + rem; rb_at = rb; re_at = re; parts = np; kt = segs.bytes(g) / BK; }
        else rem -= hi - lo;
      }
    }
    v4i e = {-1, 0, 0, 0};
    if (g_at >= 0) {
      int part = EPI == G4_PARTIAL ? tile_div(L, mtiles * ntiles) : 0, m, n;
      g4_raster(L - part * (mtiles * ntiles), mtiles, ntiles, m, n);
      const int row0 = rb_at + m * bm;
      // parts start on a pair of K steps
      const int of = tail_slot > 0 ? tail.parts : parts, at = tail_slot > 0 ? tail_part : part;
      const int kt0 = at == 0 ? 0 : tile_div(kt / 2 * at, of) * 2, kt1 = at + 1 == of ? kt : tile_div(kt / 2 * (at + 1), of) * 2;
      e = v4i{g_at | part << 8 | min(re_at - row0, bm) << 16, row0, n | tail_slot << 16, kt0 | (kt1 - kt0) << 16};
    }
    table[lane] = e;
  };
  // an item as its four packed words (scalar registers are scarce here)
  struct Item {
    int x, y, z, w;
    __device__ __forceinline__ bool some() const { return x >= 0; }
    __device__ __forceinline__ int g() const { return x & 255; }
    __device__ __forceinline__ int part() const { return x >> 8 & 255; }
    __device__ __forceinline__ int rows_here() const { return x >> 16; }
    __device__ __forceinline__ int row0() const { return y; }
    __device__ __forceinline__ int n0() const { return (z & 0xffff) * FEAT; }
    __device__ __forceinline__ int slot() const { return z >> 16; }   // of a part of a tail tile, counted from 1
    __device__ __forceinline__ int kt0() const { return w & 0xffff; }
    __device__ __forceinline__ int nkt() const { return w >> 16; }
  };
  auto item = [&](int i) -> Item {
    if (i > 0 && i % G4_TABLE_ITEMS == 0) fill_table(i);
    const v4i e = table[i % G4_TABLE_ITEMS];
    return Item{sgpr(e.x), sgpr(e.y), sgpr(e.z), sgpr(e.w)};
  };

  fill_table(0);
  Item cur = item(0);
  if (!cur.some()) return;   // block-uniform: every wave of the block leaves together
  Item nxt = item(1), nx2 = nxt;
  if (nxt.some()) nx2 = item(2);

  // ---- addressing ---------------------------------------------------------------------------------------------
  // A wave-level global->LDS load moves 8 rows of 128 bytes: lane i lands in 16-byte chunk (i & 7) of row (i >> 3) and
  // fetches logical chunk (i & 7) ^ swz(row) (fp8: f8_chunk of it). Weight rows are placed so that the two 16-row MFMA tiles of a 32-row group
  // give a lane 8 consecutive features: row r of tile t holds weight row (r >> 2) * 8 + t * 4 + (r & 3) of the group.
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr_t)smem;
  int ld_row = wave * 8 + (lane >> 3);                 // row within a 32-row slab
  int ld_chunk = (lane & 7) ^ swz(ld_row);
  if constexpr (F8) ld_chunk = f8_chunk(ld_chunk);
  int ld_wrow = ((ld_row & 15) >> 2) * 8 + (ld_row >> 4) * 4 + (ld_row & 3);
  const int ldsw = sgpr((int)lds0 + wave * 1024);
  int ldswb = sgpr(ldsw + G4_W_TILE);
  const int fr_row = lane & 15, fr_grp = lane >> 4, fr_swz = swz(fr_row);

  v32i fa0, fb0, ctx;      // slice 0 fragments of the tile about to start; addresses
  v16i voff_nxt;           // row offsets of the next tile
  v8i gi;                  // row indices of the tile after it
#pragma unroll
  for (int i = 0; i < 32; ++i) ctx[i] = own(0);
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    ctx[G4_TOK_ADDR + ks] = (int)lds0 + (wt * 16 + fr_row) * 128 + ((ks * 4 + fr_grp) ^ fr_swz) * 16;
    ctx[G4_W_ADDR + ks] = (int)lds0 + G4_W_TILE + (wq * 128 + fr_row) * 128 +
                          (W8 ? ((ks * 2 + (fr_grp >> 1)) ^ fr_swz) * 16 + (fr_grp & 1) * 8 : ((ks * 4 + fr_grp) ^ fr_swz) * 16);
  }
  ctx[G4_BIAS_VOFF] = (wq * 128 + fr_grp * 8) * 2;
  ctx[G4_DEF_LD] = ctx[G4_SCR_VOFF] = wave * (G4_SCRATCH / 4) + lane * 16;
  ctx[G4_DEF_ST] = own((int)0x80000000u);
  struct Rsrc { uint64_t lo, hi; };
  auto rsrc64 = [&](const void* p, uint32_t bytes) -> Rsrc {
    const uint64_t a = reinterpret_cast<uint64_t>(p);
    const uint32_t a0 = sgpr((int)(uint32_t)a), a1 = sgpr((int)((uint32_t)(a >> 32) & 0xffffu)), b = sgpr((int)bytes);
    return {(uint64_t)a1 << 32 | a0, (uint64_t)0x00020000u << 32 | b};
  };
  auto rsrc4 = [&](const void* p, uint32_t bytes) -> v4i {
    const Rsrc r = rsrc64(p, bytes);
    return v4i{(int)(uint32_t)r.lo, (int)(uint32_t)(r.lo >> 32), (int)(uint32_t)r.hi, (int)(uint32_t)(r.hi >> 32)};
  };
  // the operands of an item's loads: resources of tokens and weights, the lane's row offsets (gi: its row indices where the
  // group gathers its tokens); rows past the end of the tile get an offset beyond the buffer and read as zeros
  struct Source { Rsrc a, b0, b1; };
  auto weight_voff = [&](int j, int wkb) { return ((SWIGLU ? (j >> 2) * 64 + (j & 1) * 32 : j * 32) + ld_wrow) * wkb + ld_chunk * 16; };
  auto set_source = [&](const Item& d, const v8i& rows, v16i& voff) -> Source {
    Source s = {{0, 0}, {0, 0}, {0, 0}};
    if (!d.some()) return s;   // no further item: the requests still go out, against empty buffers (zeros)
    const GemmGroup& gg = args.g[d.g()];
    const int kb = gg.kbytes, wkb = W8 ? kb >> 1 : kb;
    s.a = gg.gather != nullptr ? rsrc64(gg.a, (uint32_t)gg.a_rows * (uint32_t)kb)
                               : rsrc64(gg.a + (size_t)d.row0() * kb, (uint32_t)d.rows_here() * (uint32_t)kb);
    s.b0 = rsrc64(gg.b0 + (size_t)d.n0() * wkb, (uint32_t)FEAT * (uint32_t)wkb);
    s.b1 = SWIGLU ? rsrc64(gg.b1 + (size_t)d.n0() * wkb, (uint32_t)FEAT * (uint32_t)wkb) : s.b0;
    const bool by_list = gg.gather != nullptr;
    const int shift = by_list ? gg.gather_shift : 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int r = j * 32 + ld_row;
      const int row = by_list ? rows[j] >> shift : r;
      voff[j] = r < d.rows_here() ? row * kb + ld_chunk * 16 : (int)0x80000000u;
      voff[8 + j] = weight_voff(j, wkb);
    }
    return s;
  };
  auto load_rows = [&](const Item& d) -> v8i {
    v8i r;
#pragma unroll
    for (int j = 0; j < 8; ++j) r[j] = own(0);
    const int32_t* const list = args.g[d.g()].gather;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (list != nullptr && j * 32 + ld_row < d.rows_here()) r[j] = list[d.row0() + j * 32 + ld_row];
    return r;
  };
  auto w_start = [](const Item& d) { return W8 ? d.kt0() * (BK / 2) : d.kt0() * BK; };

  // ---- the block's first two K steps (w8: weights of two pairs) as a burst --------------------------------------
  // The first step's weights go out while the row indices are on their way, and the second step may still be when the first one starts (its
  // wait is step 0's own; w8: that one lets the last 8 requests be out, which are weights there as everywhere).
  Source src;
  {
    const GemmGroup& gg = args.g[cur.g()];
    const int kb = gg.kbytes, wkb = W8 ? kb >> 1 : kb;
    const v8i rows = load_rows(cur);
    gi = nxt.some() ? load_rows(nxt) : v8i{0, 0, 0, 0, 0, 0, 0, 0};
    asm volatile("" : : : "memory");   // (the wait below counts the requests behind the first step's: none may change places with them)
    const __amdgpu_buffer_rsrc_t pb0 = make_rsrc(gg.b0 + (size_t)cur.n0() * wkb, (uint32_t)FEAT * (uint32_t)wkb);
    const __amdgpu_buffer_rsrc_t pb1 = SWIGLU ? make_rsrc(gg.b1 + (size_t)cur.n0() * wkb, (uint32_t)FEAT * (uint32_t)wkb) : pb0;
    uint8_t* const base = smem + wave * 1024;
    auto weights = [&](int st) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        __builtin_amdgcn_raw_ptr_buffer_load_lds((j >> 1) & 1 ? pb1 : pb0, (lds_ptr_t)(base + st * G4_STAGE + G4_W_TILE + j * 4096), 16,
                                                 weight_voff(j, wkb), w_start(cur) + st * BK, 0, 0);
    };
    weights(0);
    src = set_source(cur, rows, voff_nxt);
#pragma unroll
    for (int j = 0; j < 16; ++j) ctx[G4_TOK_VOFF + j] = voff_nxt[j];
    const __amdgpu_buffer_rsrc_t pa = gg.gather != nullptr
        ? make_rsrc(gg.a, (uint32_t)gg.a_rows * (uint32_t)kb)
        : make_rsrc(gg.a + (size_t)cur.row0() * kb, (uint32_t)cur.rows_here() * (uint32_t)kb);
#pragma unroll
    for (int st = 0; st < 2; ++st) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(pa, (lds_ptr_t)(base + st * G4_STAGE + j * 4096), 16, ctx[G4_TOK_VOFF + j], (cur.kt0() + st) * BK, 0, 0);
      asm volatile("" : : : "memory");
    }
    weights(1);
  }
  asm volatile("s_waitcnt vmcnt(16)\n\ts_barrier" : : : "memory");
  if constexpr (W8) asm volatile(HDMOE_G4_FILL_W8 : "={v[128:159]}"(fa0), "={v[160:191]}"(fb0), "+{v[96:127]}"(ctx) : : G4_CLOBBER_V);
  else if constexpr (F8) asm volatile(HDMOE_G4_FILL_F8 : "={v[128:159]}"(fa0), "={v[160:191]}"(fb0), "+{v[96:127]}"(ctx) : : "memory");
  else asm volatile(HDMOE_G4_FILL : "={v[128:159]}"(fa0), "={v[160:191]}"(fb0), "+{v[96:127]}"(ctx) : : "memory");

  // per-tensor scales come through the scalar cache: a vector load would be waited for together with every global->LDS
  // request in flight (one in-order counter)
  typedef const __attribute__((address_space(4))) float* const_float_ptr;
  auto scale = [&](const float* p) -> int {
    return sgpr(__float_as_int(p != nullptr ? hdmoe_dev_round_bf16(*(const_float_ptr)(uintptr_t)p) : 1.0f));
  };
  auto scale8 = [&](const float* s_in, const float* s_w) -> int {   // fp8: scale_input * scale_weight
    return sgpr(__float_as_int((s_in != nullptr ? *(const_float_ptr)(uintptr_t)s_in : 1.0f) * *(const_float_ptr)(uintptr_t)s_w));
  };
  // GELU: the tile whose activation is still to be applied (none: an empty buffer)
  v4i dro = rsrc4(nullptr, 0);
  int dldo = own(0), dnt = own(0);
  bool deferred = false;
  const v4i scr = EPI == G4_GELU ? rsrc4(args.scratch + (size_t)blockIdx.x * G4_SCRATCH, G4_SCRATCH) : rsrc4(nullptr, 0);
  const int gk = sgpr(__float_as_int((F16 ? 1.0f : 2.0f) * 0.84932180f)), gp = sgpr(__float_as_int(0.3f / 0.84932180f));  // gen_gemm4w.py: k (2 k), 0.3 / k
#define G4_DRAIN(TEXT)                                                                                               \
  asm volatile(TEXT : "+{v[128:159]}"(fa0), "+{v[160:191]}"(fb0), "+{v[96:127]}"(ctx) : [dro] "s"(dro), [dldo] "s"(dldo), [dnt] "s"(dnt), [dd] "s"(dd), [scr] "s"(scr), [gk] "s"(gk), [gp] "s"(gp) : G4_CLOBBER_V)
  // Output offsets of the pieces: the second pair of K steps stores the first two of token block 1, so DEF_ST starts a step in
  // front of them, at the last two of block 0, and advances by dd = dldo - 128 and 128 in turn.
  auto drain = [&] {
    const int dd = sgpr(dldo - 128);
    if constexpr (EPI == G4_GELU && F16) G4_DRAIN(HDMOE_G4_DRAIN_F16);
    else if constexpr (EPI == G4_GELU) G4_DRAIN(HDMOE_G4_DRAIN_BF16);
  };

  for (int i = 0;; ++i) {
    const GemmGroup& gg = args.g[cur.g()];
    // keep what depends on them out of registers that would live across the statement below
    asm volatile("" : "+v"(ld_row), "+v"(ld_chunk), "+v"(ld_wrow));
    const Source nsrc = set_source(nxt, gi, voff_nxt);
    Item nx3 = nx2;
    if (nx2.some()) nx3 = item(i + 3);
    int n = sgpr(cur.nkt() >> 1), so = sgpr((cur.kt0() + 2) * BK), wso = sgpr(w_start(cur) + 2 * BK);
    const int nso = sgpr(nxt.kt0() * BK), nwso = sgpr(w_start(nxt));
    const int ldo = gg.n_out * OUT_BYTES, ldo32 = sgpr(32 * ldo);
    int slot_u;   // in a scalar register for certain (the compiler drops the builtin where it finds the value uniform)
    // (the wait state between a vector register's write and its readfirstlane, which the compiler does not add inside a statement)
    asm volatile("s_nop 1\n\tv_readfirstlane_b32 %0, %1" : "=s"(slot_u) : "v"(cur.slot()));
    const bool part = EPI != G4_PARTIAL && slot_u > 0;   // of a tail tile: raw sums go to the slot's 256 KiB
    const uint8_t* const out = EPI == G4_PARTIAL
        ? reinterpret_cast<const uint8_t*>(gg.pout + (size_t)cur.part() * (size_t)args.part_stride + (size_t)cur.row0() * gg.n_out)
        : gg.out + (size_t)cur.row0() * ldo;
    const v4i ro = part ? rsrc4(args.tail + (size_t)(slot_u - 1) * (G4_BM * 256), G4_BM * 256 * 4)
                        : rsrc4(out, (uint32_t)cur.rows_here() * (uint32_t)ldo);
    ctx[G4_OUT_VOFF] = part ? wave * 8192 + lane * 16
                            : (wt * 16 + fr_row) * ldo + (cur.n0() + wq * (FEAT / 2) + fr_grp * 8) * OUT_BYTES;
    const int part_s = part ? sgpr(g4_part_blocks(cur.rows_here(), wave)) + 1 : 0;
    // token blocks: as its rows need (whole 256-row texts for what is not cut: Hunyuan3D block of 128 tokens 215.7 us, so 202.5; 300 230.8, 218.3)
    const int nt = sgpr(F8 || cap > 0 || (EPI != G4_PARTIAL && !part) ? max((cur.rows_here() + 31) >> 5, G4_MIN_BLOCKS) : G4_BM / 32);
    // row indices of nx2 and this tile's biases are loaded inside the statement
    const int32_t* const list = nx2.some() ? args.g[nx2.g()].gather : nullptr;
    const v4i gr = rsrc4(list != nullptr ? list + nx2.row0() : nullptr, list != nullptr ? (uint32_t)nx2.rows_here() * 4u : 0u);
    ctx[G4_GATHER_VOFF] = ld_row * 4;
    const bool with_bias = HAS_BIAS && gg.bias != nullptr;
    const v4i br = rsrc4(with_bias ? gg.bias + cur.n0() : nullptr, with_bias ? 512u : 0u);
    const int sc = W8 ? scale(gg.sb0) : F8 && EPI != G4_PARTIAL ? scale8(gg.s_in, gg.sb0) : 0, su = W8 && SWIGLU ? scale(gg.sb1) : 0;
    if (EPI == G4_GELU && deferred && n < G4_GELU_PAIRS) {
      drain();
      dro = rsrc4(nullptr, 0);
      deferred = false;
    }
    int dn = sgpr(2 * dnt - 2), dd = sgpr(dldo - 128);
#define G4_TILE(TEXT)                                                                                                \
    asm volatile(TEXT : "+{v[128:159]}"(fa0), "+{v[160:191]}"(fb0), "+{v[96:127]}"(ctx), "={v[72:79]}"(gi),          \
                        [n] "+s"(n), [so] "+s"(so), [wso] "+s"(wso), [ldswb] "+s"(ldswb), [dn] "+s"(dn), [dd] "+s"(dd) \
                 : "{v[80:95]}"(voff_nxt), [r0] "s"(src.a.lo), [r1] "s"(src.a.hi), [r2] "s"(src.b0.lo),              \
                   [r3] "s"(src.b0.hi), [r4] "s"(src.b1.lo), [r5] "s"(src.b1.hi), [nr0] "s"(nsrc.a.lo), [nr1] "s"(nsrc.a.hi),             \
                   [nr2] "s"(nsrc.b0.lo), [nr3] "s"(nsrc.b0.hi), [nr4] "s"(nsrc.b1.lo), [nr5] "s"(nsrc.b1.hi),       \
                   [nso] "s"(nso), [nwso] "s"(nwso), [ldsw] "s"(ldsw), [ro] "s"(ro), [ldo32] "s"(ldo32),             \
                   [gr] "s"(gr), [br] "s"(br), [sc] "s"(sc), [su] "s"(su), [dro] "s"(dro), [dldo] "s"(dldo),         \
                   [scr] "s"(scr), [gk] "s"(gk), [gp] "s"(gp), [nt] "s"(nt), [part] "s"(part_s)                    \
                 : G4_CLOBBER)
    if constexpr (F8 && EPI == G4_BIAS) G4_TILE(HDMOE_G4_TILE_F8_BIAS);
    else if constexpr (F8 && EPI == G4_PARTIAL) G4_TILE(HDMOE_G4_TILE_F8_PARTIAL);
    else if constexpr (F8) G4_TILE(HDMOE_G4_TILE_F8);
    else if constexpr (EPI == G4_GELU && F16) G4_TILE(HDMOE_G4_TILE_F16_GELU);
    else if constexpr (EPI == G4_GELU) G4_TILE(HDMOE_G4_TILE_BF16_GELU);
    else if constexpr (EPI == G4_BIAS && F16) G4_TILE(HDMOE_G4_TILE_F16_BIAS);
    else if constexpr (EPI == G4_BIAS && W8) G4_TILE(HDMOE_G4_TILE_BF16_W8_BIAS);
    else if constexpr (EPI == G4_BIAS) G4_TILE(HDMOE_G4_TILE_BF16_BIAS);
    else if constexpr (EPI == G4_SWIGLU && W8) G4_TILE(HDMOE_G4_TILE_BF16_W8_SWIGLU);
    else if constexpr (EPI == G4_SWIGLU) G4_TILE(HDMOE_G4_TILE_BF16_SWIGLU);
    else if constexpr (EPI == G4_PARTIAL && W8) G4_TILE(HDMOE_G4_TILE_BF16_W8_PARTIAL);
    else if constexpr (EPI == G4_PARTIAL) G4_TILE(HDMOE_G4_TILE_BF16_PARTIAL);
    else if constexpr (W8) G4_TILE(HDMOE_G4_TILE_BF16_W8);
    else G4_TILE(HDMOE_G4_TILE_BF16);
    if (EPI == G4_GELU && !part) {
      dro = ro;
      dldo = ldo32;
      dnt = nt;
      deferred = true;
      ctx[G4_DEF_LD] = ctx[G4_SCR_VOFF];
      ctx[G4_DEF_ST] = ctx[G4_OUT_VOFF] + 128;
    }
    if (!nxt.some()) break;
    src = nsrc;
    cur = nxt;
    nxt = nx2;
    nx2 = nx3;
  }
  if (deferred) drain();
  __builtin_amdgcn_s_waitcnt(0x0f70);  // the empty requests of the last pair have come back before the LDS is given up
#endif
}

// Adds the parts of the tail tiles up (in order) and finishes them as the epilogues of gen_gemm4w.py do. One thread: one
// token, 8 consecutive features. Bound by the fp32 sums read (256 KiB per part).
template <G4Type TY, int EPI>
__global__ __launch_bounds__(256) void gemm4w_tail_kernel(const GemmArgs args, int blocks) {
  constexpr bool F16 = TY == G4_F16, W8 = TY == G4_W8;
  constexpr bool SWIGLU = EPI == G4_SWIGLU;
  constexpr int FEAT = SWIGLU ? 128 : 256;
  using Act = std::conditional_t<F16, HdmoeF16, HdmoeBf16>;
  const int lane = threadIdx.x & 63;
  const Segments seg(args, lane);
  const G4Tail tail = g4_tail_of<TY, FEAT>(args, seg, blocks);
  if (tail.parts <= 1) return;
  constexpr int PER_TILE = SWIGLU ? 16 : 32;   // blocks' worth of work of a tile
  for (int item = blockIdx.x; item < tail.tiles * PER_TILE; item += gridDim.x) {
    const int t = item / PER_TILE;
    int L = __builtin_amdgcn_readfirstlane(tail.rounds * blocks + t), g = 0, m = 0, n = 0, rb = 0, re = 0;
    for (; g < args.G; ++g) {
      seg.get(g, rb, re);
      const int mt = (re - rb + G4_BM - 1) / G4_BM, nt = seg.ntiles(g, FEAT);
      if (L < mt * nt) { g4_raster(L, mt, nt, m, n); break; }
      L -= mt * nt;
    }
    const GemmGroup& gg = args.g[g];
    const int row0 = rb + m * G4_BM, rows_here = min(re - row0, G4_BM);
    // the order of gen_gemm4w.py: MFMA tile (tt, ft) of wave w at (tt * 32 + w * 8 + ft) KiB; ft 2q and 2q + 1 hold the 8 features.
    const G4TailUnit mine = g4_tail_unit(SWIGLU, item % PER_TILE, threadIdx.x >> 6, t);
    const int q = mine.q, tt = mine.tt, w = mine.w;
    const int wq = w & 1, wt = w >> 1;
    const int row = tt * 32 + wt * 16 + (lane & 15);
    if (row >= rows_here) continue;
    const float* src = args.tail + (size_t)t * tail.parts * (G4_BM * 256) + (tt * 32 + w * 8 + q * 2) * 256 + lane * 4;
    constexpr int QUADS = SWIGLU ? 4 : 2;
    float4 s[QUADS];
#pragma unroll
    for (int i = 0; i < QUADS; ++i) s[i] = *reinterpret_cast<const float4*>(src + (i & 1) * 256 + (i >> 1) * 1024);
    for (int p = 1; p < tail.parts; ++p) {
      src += G4_BM * 256;
#pragma unroll
      for (int i = 0; i < QUADS; ++i) {
        const float4 v = *reinterpret_cast<const float4*>(src + (i & 1) * 256 + (i >> 1) * 1024);
        s[i].x += v.x; s[i].y += v.y; s[i].z += v.z; s[i].w += v.w;
      }
    }
    float v[8] = {s[0].x, s[0].y, s[0].z, s[0].w, s[1].x, s[1].y, s[1].z, s[1].w};
    const int feat = n * FEAT + wq * (FEAT / 2) + q * 32 + (lane >> 4) * 8;
    auto scale = [](const float* p) { return p != nullptr ? hdmoe_dev_round_bf16(*p) : 1.0f; };
    if constexpr (SWIGLU) {
      const float u[8] = {s[2].x, s[2].y, s[2].z, s[2].w, s[3].x, s[3].y, s[3].z, s[3].w};
      const float sg = W8 ? scale(gg.sb0) : 1.0f, su = W8 ? scale(gg.sb1) : 1.0f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float h1 = hdmoe_dev_round_bf16(v[i] * sg), h3 = hdmoe_dev_round_bf16(u[i] * su);
        v[i] = hdmoe_dev_round_bf16(h1 * __builtin_amdgcn_rcpf(1.0f + __expf(-h1))) * h3;
      }
    } else {
      const float sc = W8 ? scale(gg.sb0) : 1.0f;
      float b[8] = {0, 0, 0, 0, 0, 0, 0, 0};
      if (gg.bias != nullptr) {
        const uint4 bw = *reinterpret_cast<const uint4*>(gg.bias + feat);
        const uint32_t words[4] = {bw.x, bw.y, bw.z, bw.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) { b[2 * i] = Act::lo(words[i]); b[2 * i + 1] = Act::hi(words[i]); }
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        v[i] = W8 ? __builtin_fmaf(v[i], sc, b[i]) : v[i] + b[i];
        if constexpr (EPI == G4_GELU) {
          const float h = Act::round(v[i]);
          v[i] = 0.5f * h * (1.0f + erff(h * 0.70710678118654752440f));
        }
      }
    }
    uint4 o;
    o.x = Act::pack(v[0], v[1]); o.y = Act::pack(v[2], v[3]); o.z = Act::pack(v[4], v[5]); o.w = Act::pack(v[6], v[7]);
    *reinterpret_cast<uint4*>(gg.out + ((size_t)(row0 + row) * gg.n_out + feat) * 2) = o;
  }
}

// Whether the launch fits gemm4w_kernel: whole pairs of K steps in every part, at least two of them (w8: three). Operands may
// have any size: rows are addressed from the start of their tile; gathered ones, which are not, are under 2 GiB for every kernel.
// Biases are read 8 and 16 bytes at a time.
inline bool gemm4w_fits(const GemmArgs& args, bool w8) {
  if (args.G <= 0) return false;
  for (int g = 0; g < args.G; ++g) {
    const int pairs = args.g[g].kbytes / (2 * BK);
    int parts = 1;
    if (args.nparts > 1)
      for (int i = 0; i < args.plan.n; ++i) parts = max(parts, args.g[g].row_begin < 0 ? args.plan.pd[i] : args.plan.ps[i]);
    if (args.g[g].kbytes % (2 * BK) != 0 || pairs / parts < (w8 ? 3 : 2) || args.g[g].kbytes / BK > 0x7fff) return false;
    if ((reinterpret_cast<uintptr_t>(args.g[g].bias) & 7) != 0) return false;
  }
  return true;
}
