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
// Limits (the launcher takes another kernel otherwise): K the same for all groups, a multiple of 256 bytes and at least 2048, every
// group with a scale_input for the consuming Linear (no clamp form of the cast), a gathered operand under 2 GiB.
#include "swiglu224_asm.inc"

constexpr int S224_BM = 224;                      // tokens per block tile
constexpr int S224_FEAT = 128;                    // features per block tile
constexpr int S224_TT = 7;                        // 16-token blocks of a wave
constexpr int S224_TABLE = 131072;                // LDS: [tok 0 | tok 1 | w 0 | w 1 | work item tables | deferred pieces]
constexpr int S224_STG = S224_TABLE + 4 * G4_TABLE_ITEMS * 16;
constexpr int S224_STG_WAVE = 6 * 1024;
constexpr int S224_SMEM = S224_STG + 4 * S224_STG_WAVE;

// positions in the context registers v[96:127] (gen_swiglu224.py)
enum { S224_TOK_ADDR = 0, S224_W_ADDR = 2, S224_TOK_VOFF = 4, S224_W_VOFF = 11, S224_NEXT = 12, S224_DEF_ST = 19, S224_GATHER_VOFF = 20, S224_STG_ADDR = 21 };

#define S224_CLOBBER_V                                                                                               \
  "memory", "scc", "v34", "v35", "v36", "v37", G4_V10(16), G4_V10(17), G4_V10(18), G4_V10(19), G4_V10(20), "v210", "v211", "v212", "v213", "v214", "v215"
#define S224_CLOBBER                                                                                                 \
  S224_CLOBBER_V, "s64", "s65", "s66", "s67", "s68", "s69", "s70", "s71", "s72", "s73", "s74", "s75", "s76", "s77", "s78", G4_A10(),   \
      G4_A10(1), G4_A10(2), G4_A10(3), G4_A10(4), G4_A10(5), G4_A10(6), G4_A10(7), G4_A10(8), G4_A10(9), G4_A10(10),  \
      G4_A10(11), G4_A10(12), G4_A10(13), G4_A10(14), G4_A10(15), G4_A10(16), G4_A10(17), G4_A10(18), G4_A10(19),     \
      G4_A10(20), G4_A10(21), "a220", "a221", "a222", "a223"

__global__ __launch_bounds__(G4_THREADS) __attribute__((amdgpu_waves_per_eu(1, 1))) void swiglu224_kernel(const GemmArgs args) {
#if defined(__HIP_DEVICE_COMPILE__)   // the host pass drops the stub of a kernel whose register operands it cannot parse
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wq = wave & 1, wt = wave >> 1;
  auto sgpr = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  auto own = [](int v) { asm volatile("" : "+s"(v)); return v; };   // as in gemm4w_kernel

  // ---- tiles: as gemm4w_kernel's, whole rounds and what is left of them ---------------------------------------
  const Segments segs(args, lane);
  int total = 0;
  for (int g = 0; g < args.G; ++g) {
    int rb, re;
    segs.get(g, rb, re);
    total += (re - rb + S224_BM - 1) / S224_BM * segs.ntiles(g, S224_FEAT);
  }
  const int xcd = blockIdx.x % HDMOE_NUM_XCD, slot = blockIdx.x / HDMOE_NUM_XCD;
  constexpr int nslots = HDMOE_NUM_CU / HDMOE_NUM_XCD;   // the grid is one block per CU
  const int rounds = total / HDMOE_NUM_CU, left = total % HDMOE_NUM_CU, chunk = (left + HDMOE_NUM_XCD - 1) / HDMOE_NUM_XCD;
  v4i* const table = reinterpret_cast<v4i*>(smem + S224_TABLE) + wave * G4_TABLE_ITEMS;
  auto fill_table = [&](int base) {
    const int i = base + lane;
    const int w = xcd * chunk + slot;
    const bool some = i < rounds || (i == rounds && slot < chunk && w < left);
    int rem = i < rounds ? xcd * (rounds * nslots) + slot + i * nslots : rounds * HDMOE_NUM_CU + w;
    int g_at = -1, mtiles = 1, ntiles = 1, L = 0, rb_at = 0, re_at = 0;
    for (int g = 0; g < args.G; ++g) {
      int rb, re;
      segs.get(g, rb, re);
      const int mt = (re - rb + S224_BM - 1) / S224_BM, nt = segs.ntiles(g, S224_FEAT);
      if (some && g_at < 0) {
        if (rem < mt * nt) { g_at = g; mtiles = mt; ntiles = nt; L = rem; rb_at = rb; re_at = re; }
        else rem -= mt * nt;
      }
    }
    v4i e = {-1, 0, 0, 0};
    if (g_at >= 0) {
      int m, n;
      g4_raster(L, mtiles, ntiles, m, n);
      const int row0 = rb_at + m * S224_BM;
      e = v4i{g_at | min(re_at - row0, S224_BM) << 16, row0, n, 0};
    }
    table[lane] = e;
  };
  struct Item {
    int x, row0, n;
    __device__ __forceinline__ bool some() const { return x >= 0; }
    __device__ __forceinline__ int g() const { return x & 255; }
    __device__ __forceinline__ int rows_here() const { return x >> 16; }
    __device__ __forceinline__ int n0() const { return n * S224_FEAT; }
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
  const int kb = segs.bytes(0);
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
  ctx[S224_STG_ADDR] = (int)lds0 + S224_STG + wave * S224_STG_WAVE + lane * 16;

  auto addr64 = [&](const void* p) -> uint64_t {   // the first half of a buffer resource
    const uint64_t a = reinterpret_cast<uint64_t>(p);
    const uint32_t a0 = sgpr((int)(uint32_t)a), a1 = sgpr((int)((uint32_t)(a >> 32) & 0xffffu));
    return (uint64_t)a1 << 32 | a0;
  };
  auto size64 = [&](uint32_t bytes) -> uint64_t { return (uint64_t)0x00020000u << 32 | (uint32_t)sgpr((int)bytes); };
  auto rsrc4 = [&](const void* p, uint32_t bytes) -> v4i {
    const uint64_t a = addr64(p);
    return v4i{(int)(uint32_t)a, (int)(uint32_t)(a >> 32), sgpr((int)bytes), 0x00020000};
  };
  // the gathered token operand: as the groups describe it, or the alternative the flag selects (GemmArgs::alt)
  const bool use_alt = args.alt.flag != nullptr && sgpr(*args.alt.flag) == 0;
  // the operands of an item's loads; rows past the end of the tile get an offset beyond the buffer and read as zeros
  struct Source { uint64_t a, ah, b, c; };
  auto set_source = [&](const Item& d, const v8i& rows, v8i& voff) -> Source {
    Source s = {0, size64(0), 0, 0};
    if (!d.some()) return s;   // no further item: the requests still go out, against empty buffers (zeros)
    const GemmGroup& gg = args.g[d.g()];
    const bool by_list = gg.gather != nullptr;
    const int shift = by_list ? (use_alt ? args.alt.shift : gg.gather_shift) : 0;
    if (by_list) {
      s.a = addr64(use_alt ? args.alt.a : gg.a);
      s.ah = size64((uint32_t)(use_alt ? args.alt.rows : gg.a_rows) * (uint32_t)kb);
    } else {
      s.a = addr64(gg.a + (size_t)d.row0 * kb);
      s.ah = size64((uint32_t)d.rows_here() * (uint32_t)kb);
    }
    s.b = addr64(gg.b0 + (size_t)d.n0() * kb);
    s.c = addr64(gg.b1 + (size_t)d.n0() * kb);
#pragma unroll
    for (int j = 0; j < S224_TT; ++j) {
      const int r = j * 32 + ld_row;
      const int row = by_list ? rows[j] >> shift : r;
      voff[j] = r < d.rows_here() ? row * kb + ld_chunk * 16 : (int)0x80000000u;
    }
    return s;
  };
  auto load_rows = [&](const Item& d) -> v8i {
    v8i r;
#pragma unroll
    for (int j = 0; j < 8; ++j) r[j] = own(0);
    const int32_t* const list = args.g[d.g()].gather;
#pragma unroll
    for (int j = 0; j < S224_TT; ++j)
      if (list != nullptr && j * 32 + ld_row < d.rows_here()) r[j] = list[d.row0 + j * 32 + ld_row];
    return r;
  };

  // ---- the block's first two K steps as a burst, as in gemm4w_kernel --------------------------------------------
  v8i voff;
  Source src;
  {
    auto buffer = [](uint64_t lo, uint32_t bytes) { return make_rsrc(reinterpret_cast<const void*>(lo), bytes); };
    const GemmGroup& gg = args.g[cur.g()];
    const v8i rows = load_rows(cur);
    gi = nxt.some() ? load_rows(nxt) : v8i{0, 0, 0, 0, 0, 0, 0, 0};
    asm volatile("" : : : "memory");   // (the wait below counts the requests behind the first step's: none may change places with them)
    const __amdgpu_buffer_rsrc_t pb0 = make_rsrc(gg.b0 + (size_t)cur.n0() * kb, (uint32_t)S224_FEAT * (uint32_t)kb);
    const __amdgpu_buffer_rsrc_t pb1 = make_rsrc(gg.b1 + (size_t)cur.n0() * kb, (uint32_t)S224_FEAT * (uint32_t)kb);
    uint8_t* const base = smem + wave * 1024;
    auto weights = [&](int st) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        __builtin_amdgcn_raw_ptr_buffer_load_lds((j >> 1) & 1 ? pb1 : pb0, (lds_ptr_t)(base + st * G4_STAGE + G4_W_TILE + j * 4096), 16, ctx[S224_W_VOFF],
                                                 st * BK + (j >> 2) * kb64 + (j & 1) * kb8, 0, 0);
    };
    weights(0);
    src = set_source(cur, rows, voff);
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

  // per-tensor scales come through the scalar cache (gemm4w_kernel)
  typedef const __attribute__((address_space(4))) float* const_float_ptr;
  auto scalar_load = [](const float* p) -> float { return *(const_float_ptr)(uintptr_t)p; };
  // the tile whose activation is still to be applied (none: an empty buffer), its output pitch times 16 and its cast factor
  v4i dro = rsrc4(nullptr, 0);
  int dldo = own(0), inv = own(0);
  const uint64_t bh = size64((uint32_t)S224_FEAT * (uint32_t)kb);

  for (int i = 0;; ++i) {
    const GemmGroup& gg = args.g[cur.g()];
    asm volatile("" : "+v"(ld_row), "+v"(ld_chunk));   // keeps what depends on them out of registers that would live across the statement below
    const Source nsrc = set_source(nxt, gi, voff);
#pragma unroll
    for (int j = 0; j < S224_TT; ++j) ctx[S224_NEXT + j] = voff[j];
    Item nx3 = nx2;
    if (nx2.some()) nx3 = item(i + 3);
    const int32_t* const list = nx2.some() ? args.g[nx2.g()].gather : nullptr;
    const v4i gr = rsrc4(list != nullptr ? list + nx2.row0 : nullptr, list != nullptr ? (uint32_t)nx2.rows_here() * 4u : 0u);
    const float s_in = gg.s_in != nullptr ? scalar_load(gg.s_in) : 1.0f;
    const int sc = sgpr(__float_as_int(s_in * scalar_load(gg.sb0)));
    const int su = sgpr(__float_as_int((gg.s_in_b != nullptr ? scalar_load(gg.s_in_b) : s_in) * scalar_load(gg.sb1)));
    const int nbn = sgpr(nxt.some() ? S224_FEAT * kb : 0);
    int n = sgpr(pairs), so = sgpr(2 * BK);
    asm volatile(HDMOE_S224_TILE
                 : "+{v[128:159]}"(fa0), "+{a[224:255]}"(fb0), "+{v[96:127]}"(ctx), "+{v[38:69]}"(d0), "+{v[70:85]}"(d1),
                   "+{v[216:247]}"(d2), "+{v[248:255]}"(d3), "={v[88:95]}"(gi), [n] "+s"(n), [so] "+s"(so)
                 : [ra] "s"(src.a), [rah] "s"(src.ah), [rb] "s"(src.b), [rc] "s"(src.c), [rbh] "s"(bh), [na] "s"(nsrc.a), [nah] "s"(nsrc.ah),
                   [nb] "s"(nsrc.b), [nc] "s"(nsrc.c), [nbn] "s"(nbn), [gr] "s"(gr), [dro] "s"(dro), [dldo] "s"(sgpr(dldo)), [inv] "s"(sgpr(inv)),
                   [sc] "s"(sc), [su] "s"(su), [kb8] "s"(kb8), [kb64] "s"(kb64), [ldsw] "s"(ldsw)
                 : S224_CLOBBER);
    const int ldo = gg.n_out;   // one byte per feature
    dro = rsrc4(gg.out + (size_t)cur.row0 * ldo, (uint32_t)cur.rows_here() * (uint32_t)ldo);
    dldo = 16 * ldo;
    inv = __float_as_int(hdmoe_dev_round_bf16(__fdiv_rn(1.0f, scalar_load(gg.s_next))));
    ctx[S224_DEF_ST] = (wt * (16 * S224_TT) + fr_row) * ldo + cur.n0() + wq * 64 + fr_grp * 16;
    if (!nxt.some()) break;
    src = nsrc;
    cur = nxt;
    nxt = nx2;
    nx2 = nx3;
  }
  asm volatile(HDMOE_S224_DRAIN
               : "+{v[128:159]}"(fa0), "+{a[224:255]}"(fb0), "+{v[96:127]}"(ctx), "+{v[38:69]}"(d0), "+{v[70:85]}"(d1), "+{v[216:247]}"(d2), "+{v[248:255]}"(d3)
               : [dro] "s"(dro), [dldo] "s"(sgpr(dldo)), [inv] "s"(sgpr(inv)) : S224_CLOBBER_V);
  __builtin_amdgcn_s_waitcnt(0x0f70);  // the empty requests of the last pair have come back before the LDS is given up
#endif
}

// Whether the launch fits swiglu224_kernel (see the limits above).
inline bool swiglu224_fits(const GemmArgs& args) {
  if (args.G <= 0 || args.nparts != 1) return false;
  const int kb = args.g[0].kbytes;
  if (kb % (2 * BK) != 0 || kb < 16 * BK) return false;
  for (int g = 0; g < args.G; ++g)
    if (args.g[g].kbytes != kb || args.g[g].s_next == nullptr || args.g[g].n_out % S224_FEAT != 0) return false;
  return true;
}
