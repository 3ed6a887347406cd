// fp8 gate/up GEMM + SiLU*mul on 224-token tiles, the epilogue of a tile hidden behind the K loop of the next one.
//
// Included by gemm.hip inside its unnamed namespace, behind gemm4w.h (uses GemmArgs, GemmGroup, Segments, g4_raster, swz, make_rsrc).
//
// Same contraction, rounding points and LDS tile format as grouped_gemm_kernel<FP8_SWIGLU, TT>
// (/root/reference/comfy/ldm/hidream/model.py:238 behind /root/reference/comfy/ops.py:314-358) on the K loop of gemm4w.h's fp8 kernel.
// What decides the tile: a finished tile has to wait somewhere while the next one is multiplied, as 32 bits per output (w1 x and w3 x
// in bf16). Through a scratch buffer in global memory (256-token tiles) that costs more than hiding the activation gains; 224 tokens leave
// room for 22 of 28 pieces in registers (224 accumulators and 120 fragment registers are in use) and for 6 in LDS. 8192 tokens, 2560 x
// (4 x 6912 + 3584), us: 8-wave kernel on 320-token tiles 652; 256-token tiles through a scratch buffer 660, of which the buffer 117 and
// the hidden vector instructions 27; this kernel 577 (2.53 PFLOP/s; back to back inside a layer, on other cards, 533 to 540: 2.7). 4096
// tokens: 365 (4-wave kernel of swiglu4w.h) -> 302.
//
// Low tiles of 128 tokens end a block's list where that shortens the longest block (tail_units.h, s224_mix and s224_price): the last m-tile of a
// segment rarely has 224 rows, and with a few rounds of tiles the last round is rarely full. A low tile multiplies 4 instead of 7 blocks per
// wave and step and takes about 0.75 of the time (its weights are as many, and come once more; s224_price, with what it measured).
// What a tile needs of its group sits in LDS and the first requests go out without a wait behind one another. Beside the search for low tiles, which
// takes 0.7 us at the start of a launch, that keeps a launch without any as long as it was with one height and the fields read out of the arguments
// tile by tile (layer of 8192 tokens 852.2 us so, 853.5 now).
//
// Limits (the launcher takes another kernel otherwise): K the same for all groups, a multiple of 256 bytes and at least 2048, the
// consuming Linears all with a scale_input or all without, a gathered operand under 2 GiB.
#include "swiglu224_asm.inc"

constexpr int S224_BM = 224;                      // tokens per block tile
constexpr int S224_FEAT = 128;                    // features per block tile
constexpr int S224_TT = 7;                        // 16-token blocks of a wave
constexpr int S224_LOW_TT = 4;                    // in a low tile (gen_swiglu224.py)
constexpr int S224_TABLE = 131072;                // LDS: [tok 0 | tok 1 | w 0 | w 1 | work item tables | deferred pieces | groups]
constexpr int S224_STG = S224_TABLE + 4 * G4_TABLE_ITEMS * 16;
constexpr int S224_STG_WAVE = 6 * 1024;
constexpr int S224_GROUPS = S224_STG + 4 * S224_STG_WAVE;   // [segment begin, end, high m-tiles | low ones << 16, tiles along the features] of each group; [rounds of high tiles, high tiles beyond, low tiles]
constexpr int S224_RECORDS = S224_GROUPS + (MAX_GROUPS + 1) * 16;   // four of 16 bytes for each group
constexpr int S224_SMEM = S224_RECORDS + MAX_GROUPS * 64;
static_assert(S224_SMEM <= 160 * 1024, "a CU's LDS");

// positions in the context registers v[96:127] (gen_swiglu224.py)
enum { S224_TOK_ADDR = 0, S224_W_ADDR = 2, S224_TOK_VOFF = 4, S224_W_VOFF = 11, S224_NEXT = 12, S224_DEF_ST = 19, S224_GATHER_VOFF = 20, S224_STG_ADDR = 21,
       S224_GATHER_VOFF3 = 22, S224_GATHER_VOFF4 = 23 };

#define S224_CLOBBER_V                                                                                               \
  "memory", "scc", "v34", "v35", "v36", "v37", G4_V10(16), G4_V10(17), G4_V10(18), G4_V10(19), G4_V10(20), "v210", "v211", "v212", "v213", "v214", "v215"
#define S224_CLOBBER                                                                                                 \
  S224_CLOBBER_V, "s64", "s65", "s66", "s67", "s68", "s69", "s70", "s71", "s72", "s73", "s74", "s75", "s76", "s77", "s78", G4_A10(),   \
      G4_A10(1), G4_A10(2), G4_A10(3), G4_A10(4), G4_A10(5), G4_A10(6), G4_A10(7), G4_A10(8), G4_A10(9), G4_A10(10),  \
      G4_A10(11), G4_A10(12), G4_A10(13), G4_A10(14), G4_A10(15), G4_A10(16), G4_A10(17), G4_A10(18), G4_A10(19),     \
      G4_A10(20), G4_A10(21), "a220", "a221", "a222", "a223"

// CLAMP: the consuming Linears have no scale_input, their cast clamps to the fp8 range (two more vector instructions behind the MFMAs for
// two values). Whole pass of such a layer on the 8-wave kernel -> here, us: 400 tokens 139.5 -> 115.1, 700 171 -> 144, 1300 237 -> 193, 3000 385 -> 337,
// 4096 508 -> 444, 8192 918 -> 825.
template <bool CLAMP>
__global__ __launch_bounds__(G4_THREADS) __attribute__((amdgpu_waves_per_eu(1, 1))) void swiglu224_kernel(const GemmArgs args) {
#if defined(__HIP_DEVICE_COMPILE__)   // the host pass drops the stub of a kernel whose register operands it cannot parse
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wq = wave & 1, wt = wave >> 1;
  auto sgpr = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  auto own = [](int v) { asm volatile("" : "+s"(v)); return v; };   // as in gemm4w_kernel
  auto lane_now = [] {   // the lane's number, worked out here and not kept
    int v = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    asm volatile("" : "+v"(v));
    return v;
  };

  // ---- tiles: high ones, then low ones (tail_units.h) -------------------------------------------------------------
  // What a tile needs of its group sits in LDS, put there once, lane g looking after group g: out of the arguments a field at a time, and
  // then what the scales' pointers lead to, is a chain of eight waits between two tiles, with the matrix cores idle. All fields are asked for at
  // once, beside the segments; the scales are on their way while the block looks its tiles up.
  static_assert(offsetof(GemmGroup, gather) == 8 && offsetof(GemmGroup, gather_shift) == 16 && offsetof(GemmGroup, a_rows) == 20 && offsetof(GemmGroup, b0) == 24 &&
                offsetof(GemmGroup, b1) == 32 && offsetof(GemmGroup, sb0) == 40 && offsetof(GemmGroup, sb1) == 48 && offsetof(GemmGroup, s_in) == 56 &&
                offsetof(GemmGroup, s_in_b) == 64 && offsetof(GemmGroup, s_next) == 72 && offsetof(GemmGroup, out) == 80 && sizeof(GemmGroup) % 8 == 0, "the fields");
  typedef unsigned long long v2u __attribute__((ext_vector_type(2), aligned(8)));
  v2u field[6];
  {
    typedef const __attribute__((address_space(4))) v2u* const_v2u_ptr;
    const auto mine = (const __attribute__((address_space(4))) char*)__builtin_amdgcn_kernarg_segment_ptr() + offsetof(GemmArgs, g) + min(lane, args.G - 1) * sizeof(GemmGroup);
#pragma unroll
    for (int k = 0; k < 6; ++k) field[k] = *(const_v2u_ptr)(mine + 16 * k);
  }
  const Segments segs(args, lane);
  const int kb = segs.bytes(0);
  auto value = [](unsigned long long p, unsigned long long or_p) { return *(const __attribute__((address_space(1))) float*)(p != 0 ? p : or_p); };
  const float v_sb0 = value(field[2].y, 0), v_sb1 = value(field[3].x, 0), v_in = value(field[3].y, field[2].y),
              v_in_b = value(field[4].x != 0 ? field[4].x : field[3].y, field[2].y), v_next = CLAMP ? 0.0f : value(field[4].y, 0);
  const bool use_alt = args.alt.flag != nullptr && sgpr(*args.alt.flag) == 0;   // the alternative token operand (GemmArgs::alt)
  v4i* const records = reinterpret_cast<v4i*>(smem + S224_RECORDS);
  v4i* const groups = reinterpret_cast<v4i*>(smem + S224_GROUPS);
  tile_mix<true, false>(segs, args.G, lane, S224_BM, S224_FEAT, S224_TILES, groups);
  const int xcd = blockIdx.x % HDMOE_NUM_XCD, slot = blockIdx.x / HDMOE_NUM_XCD;
  v4i* const table = reinterpret_cast<v4i*>(smem + S224_TABLE) + wave * G4_TABLE_ITEMS;
  auto fill_table = [&](int base) {
    const int l = lane_now(), i = base + l;
    const MixedTile t = mixed_tile(groups, args.G, l, xcd, slot, i, S224_BM);
    v4i e = {-1, 0, 0, 0};
    if (t.g >= 0) e = v4i{t.g | (t.low ? 256 : 0) | t.rows << 16, t.row0, t.n, 0};
    table[l] = e;
  };
  struct Item {
    int x, row0, n;
    __device__ __forceinline__ bool some() const { return x >= 0; }
    __device__ __forceinline__ int g() const { return x & 255; }
    __device__ __forceinline__ int rows_here() const { return x >> 16; }
    __device__ __forceinline__ int n0() const { return n * S224_FEAT; }
    __device__ __forceinline__ bool low() const { return (x & 256) != 0; }
    __device__ __forceinline__ int half() const { return low() ? 16 * S224_LOW_TT : 16 * S224_TT; }   // rows of a wave
  };
  auto item = [&](int i) -> Item {
    if (i > 0 && i % G4_TABLE_ITEMS == 0) fill_table(i);
    const v4i e = table[i % G4_TABLE_ITEMS];
    return Item{sgpr(e.x), sgpr(e.y), sgpr(e.z)};
  };
  fill_table(0);
  Item cur = item(0);
  if (!cur.some()) return;   // block-uniform: every wave of the block leaves together
  Item nxt = item(1), nx2 = nxt;
  if (nxt.some()) nx2 = item(2);

  // ---- addressing ---------------------------------------------------------------------------------------------
  // As in gemm4w_kernel, but that four MFMA tiles of 64 weight rows give a lane 16 consecutive features: row r of tile t holds weight
  // row (r >> 2) * 16 + t * 4 + (r & 3).
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr_t)smem;
  int ld_row = wave * 8 + (lane >> 3);                 // row within a 32-row slab
  int ld_chunk = f8_chunk((lane & 7) ^ swz(ld_row));
  const int ldsw = sgpr((int)lds0 + wave * 1024);
  const int fr_row = lane & 15, fr_grp = lane >> 4, fr_swz = swz(fr_row);
  const int kb8 = sgpr(8 * kb), kb64 = sgpr(64 * kb), pairs = sgpr(kb / (2 * BK));

  v32i fa0, fb0, ctx, d0, d2;   // fragments of the tile about to start; addresses; deferred pieces
  v16i d1;
  v8i d3, gi;                   // gi: row indices of the tile after the next
#pragma unroll
  for (int i = 0; i < 32; ++i) { ctx[i] = own(0); d0[i] = own(0); d2[i] = own(0); }
#pragma unroll
  for (int i = 0; i < 16; ++i) d1[i] = own(0);
#pragma unroll
  for (int i = 0; i < 8; ++i) d3[i] = own(0);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    ctx[S224_TOK_ADDR + h] = (int)lds0 + (wt * (16 * S224_TT) + fr_row) * 128 + ((h * 4 + fr_grp) ^ fr_swz) * 16;
    ctx[S224_W_ADDR + h] = (int)lds0 + G4_W_TILE + (wq * 128 + fr_row) * 128 + ((h * 4 + fr_grp) ^ fr_swz) * 16;
  }
  ctx[S224_W_VOFF] = (((ld_row & 15) >> 2) * 16 + (ld_row >> 4) * 4 + (ld_row & 3)) * kb + ld_chunk * 16;
  ctx[S224_DEF_ST] = own((int)0x80000000u);
  ctx[S224_GATHER_VOFF] = ld_row * 4;
  ctx[S224_GATHER_VOFF3] = ctx[S224_GATHER_VOFF4] = own(0);
  ctx[S224_STG_ADDR] = (int)lds0 + S224_STG + wave * S224_STG_WAVE + lane * 16;

  auto addr64 = [&](uint64_t a) -> uint64_t {   // the first half of a buffer resource
    const uint32_t a0 = sgpr((int)(uint32_t)a), a1 = sgpr((int)((uint32_t)(a >> 32) & 0xffffu));
    return (uint64_t)a1 << 32 | a0;
  };
  auto pair64 = [&](int lo, int hi) -> uint64_t { return (uint64_t)((uint32_t)sgpr(hi) & 0xffffu) << 32 | (uint32_t)sgpr(lo); };
  auto size64 = [&](uint32_t bytes) -> uint64_t { return (uint64_t)0x00020000u << 32 | (uint32_t)sgpr((int)bytes); };
  auto rsrc4 = [&](uint64_t p, uint32_t bytes) -> v4i {
    const uint64_t a = addr64(p);
    return v4i{(int)(uint32_t)a, (int)(uint32_t)(a >> 32), sgpr((int)bytes), 0x00020000};
  };
  // The lane's row of token slab j: rows 0-111 of the token tile in LDS belong to one wave row and 112-223 to the other, which multiply the first
  // and the second half of a tile's rows. Beyond what they multiply, and past the end: none (r undefined).
  struct Row { int r; bool some; };
  auto slab_row = [](const Item& d, int j, int ld) -> Row {
    const int half = d.half(), first = min(half, d.rows_here()), second = min(half, d.rows_here() - half), q = j * 32 - 16 * S224_TT + ld;
    if (j < 3) return {j * 32 + ld, j * 32 + ld < first};
    if (j > 3) return {half + q, q < second};
    return {(q < 0 ? 16 * S224_TT : half) + q, q < (q < 0 ? first - 16 * S224_TT : second)};
  };
  // the operands of an item's loads; rows past the end of the tile get an offset beyond the buffer and read as zeros
  struct Source { uint64_t a, ah, b, c; };
  struct Record { v4i r0, r1, r2; };
  auto record = [&](const Item& d) -> Record {
    const v4i* const r = records + 4 * (d.some() ? d.g() : 0);
    return {r[0], r[1], r[2]};
  };
  auto set_source = [&](const Item& d, const Record& of, const v8i& rows, v8i& voff) -> Source {
    Source s = {0, size64(0), 0, 0};
    if (!d.some()) return s;   // no further item: the requests still go out, against empty buffers (zeros)
    const bool by_list = pair64(of.r1.x, of.r1.y) != 0;
    const int shift = sgpr(of.r0.w);
    s.a = pair64(of.r0.x, of.r0.y);
    if (!by_list) s.a += (uint64_t)(uint32_t)d.row0 * (uint32_t)kb;
    s.ah = size64(by_list ? (uint32_t)of.r0.z : (uint32_t)d.rows_here() * (uint32_t)kb);
    s.b = pair64(of.r1.z, of.r1.w) + (uint64_t)(uint32_t)d.n0() * (uint32_t)kb;
    s.c = pair64(of.r2.x, of.r2.y) + (uint64_t)(uint32_t)d.n0() * (uint32_t)kb;
#pragma unroll
    for (int j = 0; j < S224_TT; ++j) {
      const Row at = slab_row(d, j, ld_row);
      const int row = by_list ? rows[j] >> shift : at.r;
      voff[j] = at.some ? row * kb + ld_chunk * 16 : (int)0x80000000u;
    }
    return s;
  };
  auto list_of = [&](const Record& of) { return pair64(of.r1.x, of.r1.y); };
  // The lane's entries of an item's list, as the statement below asks for the next ones: none past the end, any for rows that no wave multiplies
  auto buffer = [](uint64_t p, uint32_t bytes) { return make_rsrc(reinterpret_cast<const void*>(p), bytes); };
  auto load_rows = [&](const Item& d, const Record& of) -> v8i {
    const uint64_t list = list_of(of);
    const __amdgpu_buffer_rsrc_t entries = buffer(list + (uint64_t)(uint32_t)d.row0 * 4u, list != 0 && d.some() ? (uint32_t)d.rows_here() * 4u : 0u);
    v8i r;
    r[7] = own(0);
#pragma unroll
    for (int j = 0; j < S224_TT; ++j) r[j] = (int)__builtin_amdgcn_raw_buffer_load_b32(entries, slab_row(d, j, ld_row).r * 4, 0, 0);
    return r;
  };

  // ---- the block's first two K steps as a burst, as in gemm4w_kernel --------------------------------------------
  v8i voff;
  Source src;
  {
    if (lane < args.G) {   // every wave the same
      v4i* const r = records + 4 * lane;
      auto lo = [](uint64_t v) { return (int)(uint32_t)v; };
      auto hi = [](uint64_t v) { return (int)(uint32_t)(v >> 32); };
      const bool alt = use_alt && field[0].y != 0;
      const uint64_t a = alt ? (uint64_t)args.alt.a : field[0].x;
      r[0] = v4i{lo(a), hi(a), (alt ? args.alt.rows : hi(field[1].x)) * kb, alt ? args.alt.shift : lo(field[1].x)};
      r[1] = v4i{lo(field[0].y), hi(field[0].y), lo(field[1].y), hi(field[1].y)};
      r[2] = v4i{lo(field[2].x), hi(field[2].x), lo(field[5].x), hi(field[5].x)};
    }
    const Record of = record(cur);
    const v8i rows = load_rows(cur, of);
    gi = load_rows(nxt, record(nxt));
    const __amdgpu_buffer_rsrc_t pb0 = buffer(pair64(of.r1.z, of.r1.w) + (uint64_t)(uint32_t)cur.n0() * (uint32_t)kb, (uint32_t)S224_FEAT * (uint32_t)kb);
    const __amdgpu_buffer_rsrc_t pb1 = buffer(pair64(of.r2.x, of.r2.y) + (uint64_t)(uint32_t)cur.n0() * (uint32_t)kb, (uint32_t)S224_FEAT * (uint32_t)kb);
    asm volatile("" : : : "memory");   // (the wait below counts the requests behind the first step's: none may change places with them)
    uint8_t* const base = smem + wave * 1024;
    auto weights = [&](int st) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        __builtin_amdgcn_raw_ptr_buffer_load_lds((j >> 1) & 1 ? pb1 : pb0, (lds_ptr_t)(base + st * G4_STAGE + G4_W_TILE + j * 4096), 16, ctx[S224_W_VOFF],
                                                 st * BK + (j >> 2) * kb64 + (j & 1) * kb8, 0, 0);
    };
    weights(0);
    src = set_source(cur, of, rows, voff);
#pragma unroll
    for (int j = 0; j < S224_TT; ++j) ctx[S224_TOK_VOFF + j] = voff[j];
    const __amdgpu_buffer_rsrc_t pa = buffer(src.a, (uint32_t)src.ah);
#pragma unroll
    for (int st = 0; st < 2; ++st) {
#pragma unroll
      for (int j = 0; j < S224_TT; ++j)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(pa, (lds_ptr_t)(base + st * G4_STAGE + j * 4096), 16, ctx[S224_TOK_VOFF + j], st * BK, 0, 0);
      asm volatile("" : : : "memory");
    }
    weights(1);
  }
  asm volatile("s_waitcnt vmcnt(15)\n\ts_barrier" : : : "memory");
  asm volatile(HDMOE_S224_FILL : "={v[128:159]}"(fa0), "={a[224:255]}"(fb0), "+{v[96:127]}"(ctx) : : "memory");

  if (lane < args.G) {
    const float s_in = field[3].y != 0 ? v_in : 1.0f, s_in_b = field[4].x != 0 || field[3].y != 0 ? v_in_b : 1.0f;
    records[4 * lane + 3] = v4i{segs.n_out, __float_as_int(s_in * v_sb0), __float_as_int(s_in_b * v_sb1),
                                __float_as_int(CLAMP ? 448.0f : hdmoe_dev_round_bf16(__fdiv_rn(1.0f, v_next)))};
  }
  // the tile whose activation is still to be applied (none: an empty buffer), its output pitch times 16 and its cast factor
  v4i dro = rsrc4(0, 0);
  int dldo = own(0), inv = own(0), text = 0;
  const uint64_t bh = size64((uint32_t)S224_FEAT * (uint32_t)kb);

  for (int i = 0;; ++i) {
    {   // nothing that depends on the lane lives across the statement below
      const int l = lane_now();
      ld_row = wave * 8 + (l >> 3);
      ld_chunk = f8_chunk((l & 7) ^ swz(ld_row));
    }
    const Source nsrc = set_source(nxt, record(nxt), gi, voff);
#pragma unroll
    for (int j = 0; j < S224_TT; ++j) ctx[S224_NEXT + j] = voff[j];
    Item nx3 = nx2;
    if (nx2.some()) nx3 = item(i + 3);
    const uint64_t list = nx2.some() ? list_of(record(nx2)) : 0;
    {   // entries of rows that no wave multiplies may be any
      const int half = nx2.half();
      ctx[S224_GATHER_VOFF3] = (ld_row < 16 ? 96 + ld_row : half + ld_row - 16) * 4;
      ctx[S224_GATHER_VOFF4] = (half + 16 + ld_row) * 4;
    }
    const v4i gr = rsrc4(list != 0 ? list + (uint64_t)(uint32_t)nx2.row0 * 4u : 0, list != 0 ? (uint32_t)nx2.rows_here() * 4u : 0u);
    const v4i last = records[4 * cur.g() + 3];
    const int sc = sgpr(last.y), su = sgpr(last.z);
    const int nbn = sgpr(nxt.some() ? S224_FEAT * kb : 0);
    int n = sgpr(pairs), so = sgpr(2 * BK);
    text = sgpr(!cur.low() ? 0 : i > 0 && text == 0 ? 1 : 2);
#define S224_TILE(TEXT) \
    asm volatile(TEXT \
                 : "+{v[128:159]}"(fa0), "+{a[224:255]}"(fb0), "+{v[96:127]}"(ctx), "+{v[38:69]}"(d0), "+{v[70:85]}"(d1), \
                   "+{v[216:247]}"(d2), "+{v[248:255]}"(d3), "={v[88:95]}"(gi), [n] "+s"(n), [so] "+s"(so) \
                 : [ra] "s"(src.a), [rah] "s"(src.ah), [rb] "s"(src.b), [rc] "s"(src.c), [rbh] "s"(bh), [na] "s"(nsrc.a), [nah] "s"(nsrc.ah), \
                   [nb] "s"(nsrc.b), [nc] "s"(nsrc.c), [nbn] "s"(nbn), [gr] "s"(gr), [dro] "s"(dro), [dldo] "s"(sgpr(dldo)), [inv] "s"(sgpr(inv)), \
                   [sc] "s"(sc), [su] "s"(su), [kb8] "s"(kb8), [kb64] "s"(kb64), [ldsw] "s"(ldsw), [text] "s"(text) \
                 : S224_CLOBBER)
    if constexpr (CLAMP) S224_TILE(HDMOE_S224_TILE_CLAMP);
    else S224_TILE(HDMOE_S224_TILE);
    const v4i r2 = records[4 * cur.g() + 2], r3 = records[4 * cur.g() + 3];
    const int ldo = sgpr(r3.x);   // one byte per feature
    dro = rsrc4(pair64(r2.z, r2.w) + (uint64_t)(uint32_t)cur.row0 * (uint32_t)ldo, (uint32_t)cur.rows_here() * (uint32_t)ldo);
    dldo = 16 * ldo;
    inv = r3.w;
    const int l = lane_now();
    ctx[S224_DEF_ST] = (wt * cur.half() + (l & 15)) * ldo + cur.n0() + wq * 64 + (l >> 4) * 16;
    if (!nxt.some()) break;
    src = nsrc;
    cur = nxt;
    nxt = nx2;
    nx2 = nx3;
  }
#define S224_DRAIN(TEXT) \
  asm volatile(TEXT \
               : "+{v[128:159]}"(fa0), "+{a[224:255]}"(fb0), "+{v[96:127]}"(ctx), "+{v[38:69]}"(d0), "+{v[70:85]}"(d1), "+{v[216:247]}"(d2), "+{v[248:255]}"(d3) \
               : [dro] "s"(dro), [dldo] "s"(sgpr(dldo)), [inv] "s"(sgpr(inv)), [text] "s"(sgpr(text)) : S224_CLOBBER_V)
  if constexpr (CLAMP) S224_DRAIN(HDMOE_S224_DRAIN_CLAMP);
  else S224_DRAIN(HDMOE_S224_DRAIN);
  __builtin_amdgcn_s_waitcnt(0x0f70);  // the empty requests of the last pair have come back before the LDS is given up
#endif
}

// Whether the launch fits swiglu224_kernel (see the limits above).
inline bool swiglu224_fits(const GemmArgs& args) {
  if (args.G <= 0 || args.nparts != 1) return false;
  const int kb = args.g[0].kbytes;
  if (kb % (2 * BK) != 0 || kb < 16 * BK) return false;
  for (int g = 0; g < args.G; ++g)
    if (args.g[g].kbytes != kb || (args.g[g].s_next == nullptr) != (args.g[0].s_next == nullptr) || args.g[g].n_out % S224_FEAT != 0) return false;
  return true;
}
