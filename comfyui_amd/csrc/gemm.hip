// Grouped "NT" GEMM on the gfx950 matrix cores for the expert feed-forwards:
//   out[r, n] = epilogue( sum_k a[r, k] * w_g[n, k] ),  r in the row segment of group g.
// Replaces the per-expert operations.Linear calls of FeedForwardSwiGLU.forward
// (/root/reference/comfy/ldm/hidream/model.py:237-238) as fp8_linear evaluates them
// (/root/reference/comfy/ops.py:345-348: fp8 x fp8 products, fp32 accumulation,
// * scale_input*scale_weight, rounded to bf16) or, for bf16 weights, as a bf16
// Linear does (ops.py:107-115).
//
// Both operands are K-contiguous, which is the layout the MFMA wants: a lane feeds
// 32 (fp8) or 16 (bf16) consecutive K bytes of one row. Weights take the MFMA "A"
// slot (rows of the 32x32 result = output features) and tokens the "B" slot (columns
// = tokens), so a lane ends up with 4 consecutive features of one token per
// accumulator quad; the packed quads are transposed through LDS and leave as
// 128-byte row pieces.
//
// Block = 512 threads = 8 waves (2 per SIMD), block tile 256 tokens x 256 weight rows,
// K step 128 bytes, 2 LDS stages of 64 KiB filled by buffer_load ... lds (global ->
// LDS without passing through registers). Wave (wq, wt) owns weight rows {wq*32..+32}
// of each 128-row half and tokens {wt*128..+128}: 2x4 MFMA tiles of 32x32, 128 fp32
// accumulators per lane. In SwiGLU mode the two 128-row halves of the weight tile are
// the SAME 128 hidden features of w1 (gate) and w3 (up), so silu(gate)*up is formed
// in registers and the [rows, 2H] intermediate never exists.
//
// LDS tile layout: row-major, 128 bytes per row, 16-byte chunks XOR-swizzled with
// f(row) = ((row>>1)&7) ^ ((row&1)<<2) so that the 16-byte MFMA fragment reads of 8
// or 16 consecutive rows hit distinct banks. The global->LDS path writes LDS linearly
// per lane, so the swizzle is applied to the global address each lane fetches.
//
// Groups: row segments come from the dispatch offsets on the device (no host sync).
// The grid is sized for the worst case; a block first decodes (group, m-tile, n-tile)
// from its index and exits if its index is past the real tile count. Block ids are
// remapped so that each XCD (ids congruent mod 8) walks a contiguous range of tiles,
// 4 m-tiles deep, and its L2 sees each operand tile reused by neighbouring blocks.
#include <atomic>
#include <cmath>
#include <cstdlib>
#include <mutex>
#include <type_traits>

#include "common.h"
#include "numfmt.h"
#include "tail_units.h"

namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

constexpr int BN = 256;        // weight rows per block tile
constexpr int BK = 128;        // K bytes per stage
constexpr int STAGES = 2;
// Tokens per block tile: 2 wave rows x TT MFMA tiles of 32 tokens. TT = 4 (256 tokens) everywhere; the fp8 kernels
// also exist with TT = 5 (320 tokens: 10 % fewer operand bytes per MAC and fewer tiles), which the launcher picks
// when its tile count fills the chip as well, and the fp8 Linear with TT = 3 (192 tokens), for row counts that leave CUs
// without a tile or a last round nearly empty (hdmoe_launch_linear_bias).
constexpr int MAX_SLABS = 5;  // 64-row slabs of the largest token tile (arrays of dependent size in lambda
                              // signatures make the host pass drop the kernel stubs)
template <int TT>
struct TileCfg {
  static constexpr int BM = 64 * TT;                      // tokens per block tile
  // dynamic LDS of a block; the 128-token tile (TT = 2) has room for a third stage
  static constexpr int SMEM = (TT == 2 ? 3 : STAGES) * (BM + 256) * 128;
};
constexpr int GROUP_M = 4;     // m-tiles per raster band
constexpr int NTHREADS = 512;
constexpr int MAX_GROUPS = HDMOE_MAX_EXPERTS + 1;

// F16_PLAIN_BIAS: fp16 activations, weights, bias and outputs (the dtype the Hunyuan3D block runs in where the device
// takes it); the bf16 kernel with the other 16-bit MFMA and the other rounding.
enum Mode { FP8_SWIGLU = 0, FP8_PLAIN = 1, BF16_SWIGLU = 2, BF16_PLAIN = 3, BF16_PLAIN_BIAS = 4, FP8_PLAIN_BIAS = 5,
            F16_PLAIN_BIAS = 6 };

struct GemmGroup {
  const uint8_t* a;     // activations; row indices below are relative to this base
  const int32_t* gather;  // NULL: row r of the group is row r of a; else it is row gather[r] >> gather_shift of a (a_rows rows)
  int gather_shift;       // 1: gather holds flat slots 2t+s and a has one row per token
  int a_rows;
  const uint8_t* b0;    // plain: W [N,K]; swiglu: w1 [H,K]
  const uint8_t* b1;    // swiglu: w3 [H,K]
  const float* sb0;     // scale_weight of b0 (fp8)
  const float* sb1;     // scale_weight of b1 (fp8, swiglu)
  const float* s_in;    // scale_input of this Linear (fp8), NULL = 1
  const float* s_in_b;  // swiglu: scale_input of the w3 Linear (its value may differ from w1's where both round to the
                        // same cast factor); NULL = s_in
  const float* s_next;  // scale_input of the Linear that consumes the output (fp8 swiglu), NULL = clamp rule
  uint8_t* out;         // [rows, n_out] in the element type of the mode
  int row_begin;        // >= 0: static segment [row_begin, row_end); < 0: offsets[dyn], offsets[dyn+1]
  int row_end;
  int dyn;
  const uint16_t* bias; // BF16_PLAIN_BIAS: bf16 [n_out] added before the output is rounded, NULL = none
  int act;              // BF16_PLAIN_BIAS: 0 = none, 1 = erf GELU on the rounded output
  int n_out;            // output features (H for swiglu, N for plain)
  int kbytes;           // bytes per row of a and of the weights
  float* pout;          // split K: row 0 of this group in part 0 of the fp32 partial sums, [parts][rows][n_out]
};

// What the lists of tiles are made of, group by group, packed for one load (Segments).
struct GemmSegment { int row_begin, row_end, n_out, kbytes; };

struct GemmArgs {
  GemmGroup g[MAX_GROUPS];
  const int32_t* offsets;  // segment bounds of the dynamic groups, n_offsets + 1 entries
  int n_offsets;
  int G;
  int spread;  // 0: one tile list cut in eighths; 1 / -1: every group cut in eighths, groups walked up / down
  // Split K (plain modes, few tiles): nparts > 1, and every tile of a group exists `parts` times (the entry of `plan`
  // that hdmoe_plan_pick returns for the segment sizes at hand; experts' and static groups are cut differently), part p
  // multiplying K steps [KT*p/parts, KT*(p+1)/parts) and leaving its raw fp32 sums in pout + p * part_stride; a second kernel adds the
  // parts up. 1 = off.
  int nparts;
  long long part_stride;  // floats between two parts
  HdmoeSplitPlan plan;    // split K only
  // Gathered groups only: where *alt.flag reads 0 on the device, their token operand is alt.a (alt.rows rows, row
  // gather[r] >> alt.shift) instead of what the groups say (the gate kernel of the layer picks the layout of the fp8
  // tokens from the scale values and leaves the flag). flag NULL = off.
  HdmoeAltOperand alt;
  HdmoeRoute route;       // grouped_gemm_kernel<FP8_SWIGLU, TT, LIGHT> only
  // gemm4w_kernel only
  uint8_t* scratch;       // with GELU: G4_SCRATCH bytes per block
  float* tail;            // room for the parts of tail tiles (G4_TAIL_BYTES), NULL = tiles are not cut
  GemmSegment seg[MAX_GROUPS] __attribute__((aligned(16)));   // filled in by the launch functions (fill_segments)
  int cap;                // height of the tiles in blocks of 32 rows at most, 0 = whole tiles, -1 = by the segments' sizes
};

// a / b for 0 <= a, 0 < b; the approximate quotient of a below 2^22 is at most one off
__device__ __forceinline__ int tile_div(int a, int b) {
  if (a >> 22) return a / b;
  const int q = (int)((float)a * __builtin_amdgcn_rcpf((float)b)), r = a - q * b;
  return q + (r >= b ? 1 : 0) - (r < 0 ? 1 : 0);
}

// The groups' segments, lane g holding those of group g (none beyond the last one; dynamic groups come first). Read by one vector
// load: a group at a time they arrive a line of the arguments at a time, each wait as long as memory's (0.5 us), and a launch of five groups
// had looked its first tile up 4 to 6.5 us after its start. Whole pass, us: layer of 64 tokens 80.2 -> 75.5, 256 103.9 -> 98.6, 1024 in
// bf16 313 -> 305, Hunyuan3D block of 1500 358 -> 347. (A word of every line of the arguments read at once by scalar loads: 64 tokens 78.0, and
// 1 us more for every launch of one group.)
struct Segments {
  int rb, re, n_out, kbytes;
  unsigned long long fixed;   // bit g: a static group (or none)
  __device__ __forceinline__ Segments(const GemmArgs& args, int lane) {
    typedef const __attribute__((address_space(4))) v4i* const_v4i_ptr;
    v4i s = {0, 0, 0, 0};
    if (lane < MAX_GROUPS) s = ((const_v4i_ptr)((const __attribute__((address_space(4))) char*)__builtin_amdgcn_kernarg_segment_ptr() + offsetof(GemmArgs, seg)))[lane];
    int from = 0, to = 0;
    if (args.offsets != nullptr && lane < args.n_offsets) { from = args.offsets[lane]; to = args.offsets[lane + 1]; }
    fixed = __ballot(s.x >= 0);
    rb = s.x >= 0 ? s.x : from;
    re = s.x >= 0 ? s.y : to;
    n_out = s.z;
    kbytes = s.w;
  }
  __device__ __forceinline__ void get(int g, int& begin, int& end) const {
    begin = __builtin_amdgcn_readlane(rb, g);
    end = __builtin_amdgcn_readlane(re, g);
  }
  // (arithmetic behind the read: lane g may be switched off where these are called, and then forms nothing)
  __device__ __forceinline__ int rows(int g) const { return __builtin_amdgcn_readlane(re, g) - __builtin_amdgcn_readlane(rb, g); }
  __device__ __forceinline__ int ntiles(int g, int feat) const { return (int)((unsigned)__builtin_amdgcn_readlane(n_out, g) / (unsigned)feat); }
  __device__ __forceinline__ int bytes(int g) const { return __builtin_amdgcn_readlane(kbytes, g); }
  __device__ __forceinline__ bool dynamic(int g) const { return !(fixed >> g & 1); }
};

__device__ __forceinline__ int swz(int row) { return ((row >> 1) & 7) ^ ((row & 1) << 2); }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}

typedef __attribute__((address_space(3))) void* lds_ptr_t;

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// ---- fp8 K loop in assembly ---------------------------------------------------------------------
// The fragment registers of the fp8 K loop are fixed and its slices are written in assembly: the schedule below
// depends on every fragment being refilled in place right after its last use and on the global->LDS loads of the
// next step being issued one at a time between the MFMAs (the register allocator rotates fragment registers
// and then spills loop-invariant addresses, and a burst of loads behind the barrier keeps both waves of a SIMD
// in the vector-memory issue queue while the matrix pipe runs dry).
//   weight fragments  fb0 v[200:207]  fb1 v[208:215]        token fragments  fa(t) v[216+8t : 223+8t]
// One slice (64 K bytes) = part A (weight half 0 against every token block) + part B (weight half 1). LDS
// requests in flight at the start of a slice, oldest first: fb0, fa0 .. fa(TT-1), fb1 (two ds_read_b128 each);
// LDS returns in order, so part A waits with lgkmcnt(2*(TT-t)) in front of MFMA t. Part B refills fb0 first,
// then fa(t) behind the MFMA that last reads it, then fb1: every fragment is requested TT or more MFMAs (320+
// cycles of matrix pipe) before its first use. The global->LDS loads count on vmcnt, not lgkmcnt.
#define HDMOE_FB0 "v[200:207]"
#define HDMOE_FB1 "v[208:215]"
#define HDMOE_FA0 "v[216:223]"
#define HDMOE_FA1 "v[224:231]"
#define HDMOE_FA2 "v[232:239]"
#define HDMOE_FA3 "v[240:247]"
#define HDMOE_FA4 "v[248:255]"
#define HDMOE_MF(C, A, B) "v_mfma_f32_32x32x64_f8f6f4 %[" C "], " A ", " B ", %[" C "]\n"
// fragment reads: operands w0/w1 (weights) and t0/t1 (tokens) are the lane's two 16-byte halves of the slice read,
// ob / oa the byte offset of the stage read from
#define HDMOE_RD(LO, HI, A0, A1, OFF) \
  "ds_read_b128 " LO ", %[" A0 "] offset:" OFF "\nds_read_b128 " HI ", %[" A1 "] offset:" OFF "\n"
#define HDMOE_RD_FB0 HDMOE_RD("v[200:203]", "v[204:207]", "w0", "w1", "%[ob]")
#define HDMOE_RD_FB1 HDMOE_RD("v[208:211]", "v[212:215]", "w0", "w1", "%[ob]+16384")
#define HDMOE_RD_FA0 HDMOE_RD("v[216:219]", "v[220:223]", "t0", "t1", "%[oa]")
#define HDMOE_RD_FA1 HDMOE_RD("v[224:227]", "v[228:231]", "t0", "t1", "%[oa]+4096")
#define HDMOE_RD_FA2 HDMOE_RD("v[232:235]", "v[236:239]", "t0", "t1", "%[oa]+8192")
#define HDMOE_RD_FA3 HDMOE_RD("v[240:243]", "v[244:247]", "t0", "t1", "%[oa]+12288")
#define HDMOE_RD_FA4 HDMOE_RD("v[248:251]", "v[252:255]", "t0", "t1", "%[oa]+16384")
// one global->LDS load of 8 rows x 128 bytes per wave: M0 = LDS address of the wave's rows (ldsd: the wave's
// offset inside a 64-row slab, IMM: stage and slab), vector offset = the lane's row and chunk, scalar offset = K
#define HDMOE_LD(RS, VO, IMM) \
  "s_add_u32 m0, %[ldsd], " IMM "\ns_nop 0\nbuffer_load_dwordx4 %[" VO "], %[" RS "], %[so] offen lds\n"
#define HDMOE_LDW0 HDMOE_LD("rb0", "vb0", "%[wd]")
#define HDMOE_LDW1 HDMOE_LD("rb0", "vb1", "%[wd]+8192")
#define HDMOE_LDW2 HDMOE_LD("rb1", "vb0", "%[wd]+16384")
#define HDMOE_LDW3 HDMOE_LD("rb1", "vb1", "%[wd]+24576")
#define HDMOE_LDT0 HDMOE_LD("ra", "va0", "%[td]")
#define HDMOE_LDT1 HDMOE_LD("ra", "va1", "%[td]+8192")
#define HDMOE_LDT2 HDMOE_LD("ra", "va2", "%[td]+16384")
#define HDMOE_LDT3 HDMOE_LD("ra", "va3", "%[td]+24576")
#define HDMOE_LDT4 HDMOE_LD("ra", "va4", "%[td]+32768")
#define HDMOE_NONE ""
// part A; L0..L4: what follows each MFMA (a token load of the next step, or nothing)
#define HDMOE_PART_A4(L0, L1, L2, L3)                                                      \
  "s_waitcnt lgkmcnt(8)\n" HDMOE_MF("c0", HDMOE_FB0, HDMOE_FA0) L0                         \
  "s_waitcnt lgkmcnt(6)\n" HDMOE_MF("c1", HDMOE_FB0, HDMOE_FA1) L1                         \
  "s_waitcnt lgkmcnt(4)\n" HDMOE_MF("c2", HDMOE_FB0, HDMOE_FA2) L2                         \
  "s_waitcnt lgkmcnt(2)\n" HDMOE_MF("c3", HDMOE_FB0, HDMOE_FA3) L3
#define HDMOE_PART_A5(L0, L1, L2, L3, L4)                                                  \
  "s_waitcnt lgkmcnt(10)\n" HDMOE_MF("c0", HDMOE_FB0, HDMOE_FA0) L0                        \
  "s_waitcnt lgkmcnt(8)\n" HDMOE_MF("c1", HDMOE_FB0, HDMOE_FA1) L1                         \
  "s_waitcnt lgkmcnt(6)\n" HDMOE_MF("c2", HDMOE_FB0, HDMOE_FA2) L2                         \
  "s_waitcnt lgkmcnt(4)\n" HDMOE_MF("c3", HDMOE_FB0, HDMOE_FA3) L3                         \
  "s_waitcnt lgkmcnt(2)\n" HDMOE_MF("c4", HDMOE_FB0, HDMOE_FA4) L4
#define HDMOE_PART_A3(L0, L1, L2)                                                          \
  "s_waitcnt lgkmcnt(6)\n" HDMOE_MF("c0", HDMOE_FB0, HDMOE_FA0) L0                         \
  "s_waitcnt lgkmcnt(4)\n" HDMOE_MF("c1", HDMOE_FB0, HDMOE_FA1) L1                         \
  "s_waitcnt lgkmcnt(2)\n" HDMOE_MF("c2", HDMOE_FB0, HDMOE_FA2) L2
#define HDMOE_PART_A3_PLAIN HDMOE_PART_A3(HDMOE_NONE, HDMOE_NONE, HDMOE_NONE)
#define HDMOE_PART_A3_LOADS HDMOE_PART_A3(HDMOE_LDT0, HDMOE_LDT1, HDMOE_LDT2)
#define HDMOE_PART_A4_PLAIN HDMOE_PART_A4(HDMOE_NONE, HDMOE_NONE, HDMOE_NONE, HDMOE_NONE)
#define HDMOE_PART_A5_PLAIN HDMOE_PART_A5(HDMOE_NONE, HDMOE_NONE, HDMOE_NONE, HDMOE_NONE, HDMOE_NONE)
#define HDMOE_PART_A4_LOADS HDMOE_PART_A4(HDMOE_LDT0, HDMOE_LDT1, HDMOE_LDT2, HDMOE_LDT3)
#define HDMOE_PART_A5_LOADS HDMOE_PART_A5(HDMOE_LDT0, HDMOE_LDT1, HDMOE_LDT2, HDMOE_LDT3, HDMOE_LDT4)
// part B with the refills for the next slice; L0..L3: a weight load of the step after the next, or nothing
#define HDMOE_PART_B4(L0, L1, L2, L3)                                                            \
  HDMOE_RD_FB0 "s_waitcnt lgkmcnt(2)\n" HDMOE_MF("d0", HDMOE_FB1, HDMOE_FA0) HDMOE_RD_FA0 L0     \
  HDMOE_MF("d1", HDMOE_FB1, HDMOE_FA1) HDMOE_RD_FA1 L1                                           \
  HDMOE_MF("d2", HDMOE_FB1, HDMOE_FA2) HDMOE_RD_FA2 L2                                           \
  HDMOE_MF("d3", HDMOE_FB1, HDMOE_FA3) HDMOE_RD_FA3 HDMOE_RD_FB1 L3
#define HDMOE_PART_B5(L0, L1, L2, L3)                                                            \
  HDMOE_RD_FB0 "s_waitcnt lgkmcnt(2)\n" HDMOE_MF("d0", HDMOE_FB1, HDMOE_FA0) HDMOE_RD_FA0 L0     \
  HDMOE_MF("d1", HDMOE_FB1, HDMOE_FA1) HDMOE_RD_FA1 L1                                           \
  HDMOE_MF("d2", HDMOE_FB1, HDMOE_FA2) HDMOE_RD_FA2 L2                                           \
  HDMOE_MF("d3", HDMOE_FB1, HDMOE_FA3) HDMOE_RD_FA3 L3                                           \
  HDMOE_MF("d4", HDMOE_FB1, HDMOE_FA4) HDMOE_RD_FA4 HDMOE_RD_FB1
#define HDMOE_PART_B3(L0, L1, L2, L3)                                                            \
  HDMOE_RD_FB0 "s_waitcnt lgkmcnt(2)\n" HDMOE_MF("d0", HDMOE_FB1, HDMOE_FA0) HDMOE_RD_FA0 L0     \
  HDMOE_MF("d1", HDMOE_FB1, HDMOE_FA1) HDMOE_RD_FA1 L1                                           \
  HDMOE_MF("d2", HDMOE_FB1, HDMOE_FA2) HDMOE_RD_FA2 HDMOE_RD_FB1 L2 L3
#define HDMOE_PART_B3_PLAIN HDMOE_PART_B3(HDMOE_NONE, HDMOE_NONE, HDMOE_NONE, HDMOE_NONE)
#define HDMOE_PART_B3_LOADS HDMOE_PART_B3(HDMOE_LDW0, HDMOE_LDW1, HDMOE_LDW2, HDMOE_LDW3)
#define HDMOE_PART_B4_PLAIN HDMOE_PART_B4(HDMOE_NONE, HDMOE_NONE, HDMOE_NONE, HDMOE_NONE)
#define HDMOE_PART_B5_PLAIN HDMOE_PART_B5(HDMOE_NONE, HDMOE_NONE, HDMOE_NONE, HDMOE_NONE)
#define HDMOE_PART_B4_LOADS HDMOE_PART_B4(HDMOE_LDW0, HDMOE_LDW1, HDMOE_LDW2, HDMOE_LDW3)
#define HDMOE_PART_B5_LOADS HDMOE_PART_B5(HDMOE_LDW0, HDMOE_LDW1, HDMOE_LDW2, HDMOE_LDW3)
// part B of the last slice of a tile: no refills; the trailing wait states cover the distance the hardware wants
// between the last MFMA and the first VALU read of an accumulator (the compiler cannot see into the block)
#define HDMOE_PART_B3_LAST                                                                                  \
  "s_waitcnt lgkmcnt(0)\n" HDMOE_MF("d0", HDMOE_FB1, HDMOE_FA0) HDMOE_MF("d1", HDMOE_FB1, HDMOE_FA1)        \
  HDMOE_MF("d2", HDMOE_FB1, HDMOE_FA2) "s_nop 15\ns_nop 7\n"
#define HDMOE_PART_B4_LAST                                                                                  \
  "s_waitcnt lgkmcnt(0)\n" HDMOE_MF("d0", HDMOE_FB1, HDMOE_FA0) HDMOE_MF("d1", HDMOE_FB1, HDMOE_FA1)        \
  HDMOE_MF("d2", HDMOE_FB1, HDMOE_FA2) HDMOE_MF("d3", HDMOE_FB1, HDMOE_FA3) "s_nop 15\ns_nop 7\n"
#define HDMOE_PART_B5_LAST                                                                                  \
  "s_waitcnt lgkmcnt(0)\n" HDMOE_MF("d0", HDMOE_FB1, HDMOE_FA0) HDMOE_MF("d1", HDMOE_FB1, HDMOE_FA1)        \
  HDMOE_MF("d2", HDMOE_FB1, HDMOE_FA2) HDMOE_MF("d3", HDMOE_FB1, HDMOE_FA3)                                 \
  HDMOE_MF("d4", HDMOE_FB1, HDMOE_FA4) "s_nop 15\ns_nop 7\n"
// Two forms of a part in one block, chosen by the wave-uniform operand fl, so that the accumulators pass through the
// same statement either way (a branch around separate statements makes the compiler copy and spill them).
#define HDMOE_SELECT(IF_SET, IF_CLEAR) \
  "s_cmp_lg_u32 %[fl], 0\ns_cbranch_scc0 1f\n" IF_SET "s_branch 2f\n1:\n" IF_CLEAR "2:\n"
// the first fragments of a tile, in the order the waits of part A assume
#define HDMOE_FILL3 HDMOE_RD_FB0 HDMOE_RD_FA0 HDMOE_RD_FA1 HDMOE_RD_FA2 HDMOE_RD_FB1
#define HDMOE_FILL4 HDMOE_RD_FB0 HDMOE_RD_FA0 HDMOE_RD_FA1 HDMOE_RD_FA2 HDMOE_RD_FA3 HDMOE_RD_FB1
#define HDMOE_FILL5 HDMOE_RD_FB0 HDMOE_RD_FA0 HDMOE_RD_FA1 HDMOE_RD_FA2 HDMOE_RD_FA3 HDMOE_RD_FA4 HDMOE_RD_FB1

// LIGHT (fp8 only): the K loop is the compiler-scheduled one of the 16-bit modes, which skips the 32-token blocks of a
// tile that hold no rows, instead of the assembly loop, which multiplies padding like rows. For launches whose tiles are
// mostly padding (few tokens per segment).
template <int MODE, int TT, bool LIGHT = false>
__global__ __launch_bounds__(NTHREADS) void grouped_gemm_kernel(const GemmArgs args) {
  constexpr bool FP8 = (MODE == FP8_SWIGLU || MODE == FP8_PLAIN || MODE == FP8_PLAIN_BIAS);
  constexpr bool SWIGLU = (MODE == FP8_SWIGLU || MODE == BF16_SWIGLU);
  constexpr bool BIAS = (MODE == BF16_PLAIN_BIAS || MODE == FP8_PLAIN_BIAS || MODE == F16_PLAIN_BIAS);  // Linear with bias and optional GELU
  constexpr bool F16 = MODE == F16_PLAIN_BIAS;
  using Act = std::conditional_t<F16, HdmoeF16, HdmoeBf16>;  // element format of activations, bias and outputs
  constexpr int WAVE_TOK = 32 * TT;        // tokens per wave row
  constexpr int BM = 2 * WAVE_TOK;         // tokens per block tile
  constexpr int A_SLABS = BM / 64;         // 64-row slabs of the token tile
  constexpr int A_BYTES = BM * BK;         // token tile of one K step in LDS; the weight tile follows it
  constexpr int STAGE_BYTES = (BM + BN) * BK;
  constexpr int FEAT_PER_TILE = SWIGLU ? BN / 2 : BN;  // output features per block tile
  // LDS layout of the two stages. bf16: stage after stage, [A0 | B0 | A1 | B1]. fp8: [A0 | A1 | B0 | B1], so that
  // every fragment read of the K loop is one of eight per-lane base addresses plus an immediate below 64 KiB.
  constexpr int B_BYTES = BN * BK;
  constexpr int A_OFF1 = FP8 ? A_BYTES : STAGE_BYTES;
  constexpr int B_OFF0 = FP8 ? 2 * A_BYTES : A_BYTES;
  constexpr int B_OFF1 = FP8 ? 2 * A_BYTES + B_BYTES : STAGE_BYTES + A_BYTES;
  // RING3 (the light form on the 128-token tile; split K only): three stages [A | B] one after the other, K steps
  // requested two ahead. With few rows a K step lasts as long as its loads take to arrive, not as long as its MFMAs.
  constexpr bool RING3 = LIGHT && TT == 2;
  static_assert(!RING3 || !BIAS, "the three-stage ring is built for the feed-forward contractions");
  static_assert(TT != 3 || (FP8 && !LIGHT), "the 192-token tile exists only with the fp8 assembly loop");
  static_assert(TT != 2 || RING3, "the 128-token tile exists only with the three-stage ring");
  auto a_off = [](int stage) { return RING3 ? stage * STAGE_BYTES : (stage ? A_OFF1 : 0); };
  auto b_off = [](int stage) { return RING3 ? stage * STAGE_BYTES + A_BYTES : (stage ? B_OFF1 : B_OFF0); };
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  if constexpr (RING3 && !SWIGLU) {
    if (args.nparts <= 1) return;  // its plain epilogue is the partial-sum store only (kernel argument: uniform)
  }

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform by construction
  const int wq = wave & 3, wt = wave >> 2;

  // ---- tile enumeration (persistent blocks) ----------------------------------------------
  // (the 320-token tile has no registers for them: a group at a time out of the arguments there)
  constexpr bool LANES = TT != 5;
  [[maybe_unused]] auto segs = [&] {
    if constexpr (LANES) return Segments(args, lane);
    else return 0;
  }();
  [[maybe_unused]] int off_lane = 0;
  if constexpr (!LANES) {
    if (args.offsets != nullptr && lane <= args.n_offsets) off_lane = args.offsets[lane];
  }
  // Few slots: the dispatch happens here (the counting sort of dispatch_scatter_kernel, one slot per thread), while a launch of its own takes
  // as long as its latencies; the row indices then come out of LDS. Layer of 64 tokens 75.4 -> 73.0 us, 256 97.9 -> 95.7.
  constexpr bool ROUTES = MODE == FP8_SWIGLU && LIGHT;
  [[maybe_unused]] int32_t* const lds_perm = reinterpret_cast<int32_t*>(smem + TileCfg<TT>::SMEM);
  if constexpr (ROUTES) {
    if (args.route.idx != nullptr) {
      int32_t* const wave_cnt = lds_perm + HDMOE_ROUTE_SLOTS;   // [8][16]
      const int E = args.route.E;
      int e = tid < args.route.n ? args.route.idx[tid] : -1;
      if (e >= E) e = -1;   // never index a table with a bad id
      int rank = 0, mine = 0;
      for (int q = 0; q < E; ++q) {
        const unsigned long long m = __ballot(e == q);
        if (e == q) rank = __popcll(m & ((1ull << lane) - 1ull));
        if (lane == q) mine = __popcll(m);
      }
      if (lane < E) wave_cnt[wave * HDMOE_MAX_EXPERTS + lane] = mine;
      __syncthreads();
      int total = 0, before = 0, start = 0;   // lane q: of expert q
      if (lane < E) {
#pragma unroll
        for (int w = 0; w < NTHREADS / 64; ++w) {
          const int v = wave_cnt[w * HDMOE_MAX_EXPERTS + lane];
          total += v;
          before += w < wave ? v : 0;
        }
      }
      for (int q = 0; q < E; ++q) start += lane > q ? __builtin_amdgcn_readlane(total, q) : 0;
      const int pos = __shfl(start + before, e < 0 ? 0 : e, 64) + rank;
      if (e >= 0) lds_perm[pos] = tid;
      if (blockIdx.x == 0) {
        if (e >= 0) {
          args.route.perm[pos] = tid;
          args.route.inv_perm[tid] = pos;
        }
        if (tid < E) {
          args.route.counts[tid] = total;
          args.route.offsets[tid] = start;
          if (tid == E - 1) args.route.offsets[E] = start + total;
        }
      }
      if (!(segs.fixed >> lane & 1)) { segs.rb = start; segs.re = start + total; }
      __syncthreads();
    }
  }
  auto seg = [&](const GemmGroup& gg, [[maybe_unused]] int g, int& rb, int& re) {
    if constexpr (LANES) segs.get(g, rb, re);
    else if (gg.row_begin >= 0) { rb = gg.row_begin; re = gg.row_end; }
    else { rb = __builtin_amdgcn_readlane(off_lane, gg.dyn); re = __builtin_amdgcn_readlane(off_lane, gg.dyn + 1); }
  };
  auto dynamic = [&](int g) -> bool {
    if constexpr (LANES) return segs.dynamic(g);
    else return args.g[g].row_begin < 0;
  };
  auto ntiles_of = [&](int g) -> int {
    if constexpr (LANES) return segs.ntiles(g, FEAT_PER_TILE);
    else return args.g[g].n_out / FEAT_PER_TILE;
  };
  // the gathered token operand: as the groups describe it, or the alternative the flag selects
  const bool use_alt = args.alt.flag != nullptr && __builtin_amdgcn_readfirstlane(*args.alt.flag) == 0;
  auto gathered_a = [&](const GemmGroup& gg) { return use_alt ? args.alt.a : gg.a; };
  auto gathered_rows = [&](const GemmGroup& gg) { return use_alt ? args.alt.rows : gg.a_rows; };
  auto gathered_shift = [&](const GemmGroup& gg) { return use_alt ? args.alt.shift : gg.gather_shift; };
  // split K: which cut of the plan runs (a function of the segment sizes; the kernel that adds the parts up makes the
  // same choice)
  int plan_idx = 0;
  if (args.nparts > 1 && args.plan.n > 1) {
    int mt_dyn = 0, mt_static = 0;
    for (int g = 0; g < args.G; ++g) {
      int rb, re;
      seg(args.g[g], g, rb, re);
      const int mt = (re - rb + args.plan.bm - 1) / args.plan.bm;  // the plan's own tile height: the other kernel's count
      if (dynamic(g)) mt_dyn += mt;
      else mt_static += mt;
    }
    plan_idx = hdmoe_plan_pick(args.plan, mt_dyn, mt_static, ntiles_of(0));
  }
  const int parts_dyn = args.nparts > 1 ? args.plan.pd[plan_idx] : 1, parts_static = args.nparts > 1 ? args.plan.ps[plan_idx] : 1;
  auto parts_of = [&](int g) { return dynamic(g) ? parts_dyn : parts_static; };
  int total = 0;
  for (int g = 0; g < args.G; ++g) {
    int rb, re;
    seg(args.g[g], g, rb, re);
    total += ((re - rb + BM - 1) / BM) * ntiles_of(g) * parts_of(g);
  }
  // Each XCD (block ids congruent mod 8) walks one contiguous eighth of the tile list and its blocks take
  // consecutive tiles, so the CUs of an XCD share operand tiles in their L2.
  const int per_xcd = (total + HDMOE_NUM_XCD - 1) / HDMOE_NUM_XCD;
  const int xcd = blockIdx.x % HDMOE_NUM_XCD, slot = blockIdx.x / HDMOE_NUM_XCD;
  const int nslots = gridDim.x / HDMOE_NUM_XCD;

  auto div = [](int a, int b) { return LANES ? tile_div(a, b) : a / b; };
  struct Tile { int g, row0, rows_here, n0, kbytes, part, kt0, nkt; };
  auto decode = [&](int i) -> Tile {
    Tile d = {-1, 0, 0, 0, 0, 0, 0, 0};
    int in_xcd = slot + i * nslots;
    int L = 0, g = 0, rb = 0, re = 0, mtiles = 0, ntiles = 0;
    if (args.spread != 0) {
      // Groups whose tiles differ in length (the K of the shared expert's down projection is about half the
      // routed experts'): every XCD takes its eighth of every group, longest tiles first, so each block gets
      // the same mix and the blocks end together.
      int k = 0, end = 0;
      for (; k < args.G; ++k) {
        g = args.spread > 0 ? k : args.G - 1 - k;
        seg(args.g[g], g, rb, re);
        mtiles = (re - rb + BM - 1) / BM;
        ntiles = ntiles_of(g);
        const int from = end;
        end += mtiles * ntiles * parts_of(g);
        const int lo = g4_dealt(end, xcd) - g4_dealt(from, xcd), hi = g4_dealt(end, xcd + 1) - g4_dealt(from, xcd + 1);
        if (in_xcd < hi - lo) { L = lo + in_xcd; break; }
        in_xcd -= hi - lo;
      }
      if (k >= args.G) return d;
    } else {
      L = xcd * per_xcd + in_xcd;
      if (in_xcd >= per_xcd || L >= total) return d;
      for (; g < args.G; ++g) {
        seg(args.g[g], g, rb, re);
        mtiles = (re - rb + BM - 1) / BM;
        ntiles = ntiles_of(g);
        const int tiles = mtiles * ntiles * parts_of(g);
        if (L < tiles) break;
        L -= tiles;
      }
      if (g >= args.G) return d;
    }
    // split K: the parts of a group one after the other (tiles of one part share operand slices, parts do not)
    const int part = div(L, mtiles * ntiles);
    L -= part * (mtiles * ntiles);
    // bands of GROUP_M m-tiles; a short remainder joins the last band, so that the cheap partial m-tile at the
    // end of a segment is interleaved with full ones instead of forming a run of its own
    const int nbands = max(1, (mtiles + GROUP_M / 2) / GROUP_M);
    const int band = min(div(L, GROUP_M * ntiles), nbands - 1);
    const int first_m = band * GROUP_M;
    const int gm = band == nbands - 1 ? mtiles - first_m : GROUP_M;
    const int within = L - band * (GROUP_M * ntiles);
    const int n = div(within, gm);
    d.g = g;
    d.row0 = rb + (first_m + within - n * gm) * BM;
    d.rows_here = min(re - d.row0, BM);
    d.n0 = n * FEAT_PER_TILE;
    if constexpr (LANES) d.kbytes = segs.bytes(g);
    else d.kbytes = args.g[g].kbytes;
    const int ktf = d.kbytes / BK;
    d.part = part;
    d.kt0 = div(ktf * part, parts_of(g));
    d.nkt = div(ktf * (part + 1), parts_of(g)) - d.kt0;
    return d;
  };

  // ---- global -> LDS addressing --------------------------------------------------
  // One wave-level load moves 8 rows x 128 bytes. Lane i lands in LDS chunk (i&7) of row (i>>3) and therefore
  // fetches logical chunk (i&7) ^ f(row). Rows past the segment end are outside the buffer range and read as
  // zero: the row part of the address sits in the VGPR offset, the only one that is range-checked; the K
  // position goes through the scalar offset.
  const int ld_row = wave * 8 + (lane >> 3);                 // row within a 64-row slab
  const int ld_chunk = (lane & 7) ^ swz(ld_row);
  const int ld_lds = wave * 8 * BK;                          // + slab*64*BK

  // source of the tile being loaded (buffer resources are kept as plain locals: the opaque resource type
  // cannot be a struct member)
  //
  // Weight rows of the tile. SwiGLU: LDS half h (128 rows) holds rows n0..n0+127 of w1 (h=0) / w3 (h=1).
  // Plain: wave column wq multiplies LDS rows wq*32..+32 of both halves, and its 64 output features should be
  // contiguous in memory, so LDS row (h, wq, i) holds weight row n0 + wq*64 + h*32 + i.
  __amdgpu_buffer_rsrc_t src_a = make_rsrc(nullptr, 0), src_b0 = src_a, src_b1 = src_a;
  int src_voff[MAX_SLABS] = {};
  int src_voff_b[2] = {0, 0};
  // Row indices of a gathered token operand: loaded one tile ahead (load_gather), consumed by set_src.
  auto load_gather = [&](const Tile& d, int (&gi)[MAX_SLABS]) {
    const GemmGroup& gg = args.g[d.g];
#pragma unroll
    for (int j = 0; j < A_SLABS; ++j) {
      const int r = j * 64 + ld_row;
      if constexpr (ROUTES) {
        if (args.route.idx != nullptr) {
          gi[j] = (gg.gather != nullptr && r < d.rows_here) ? (lds_perm[d.row0 + r] >> gathered_shift(gg)) : -1;
          continue;
        }
      }
      gi[j] = (gg.gather != nullptr && r < d.rows_here) ? (gg.gather[d.row0 + r] >> gathered_shift(gg)) : -1;
    }
  };
  // the same three resources as plain descriptor words, for the loads issued from the assembly blocks
  [[maybe_unused]] v4i ra4 = {0, 0, 0, 0}, rb04 = ra4, rb14 = ra4;
  auto raw_rsrc = [](const void* p, uint32_t bytes) -> v4i {
    const uint64_t a = reinterpret_cast<uint64_t>(p);
    v4i r;
    r.x = (int)(uint32_t)a; r.y = (int)(uint32_t)((a >> 32) & 0xffffu); r.z = (int)bytes; r.w = 0x00020000;
    return r;
  };
  int k_base = 0;  // K byte offset of step 0 of the tile being loaded (split K)
  auto set_src = [&](const Tile& d, const int (&gi)[MAX_SLABS]) {
    const GemmGroup& gg = args.g[d.g];
    k_base = d.kt0 * BK;
    if constexpr (FP8) {
      if (gg.gather != nullptr) ra4 = raw_rsrc(gathered_a(gg), (uint32_t)gathered_rows(gg) * (uint32_t)d.kbytes);
      else ra4 = raw_rsrc(gg.a + (size_t)d.row0 * d.kbytes, (uint32_t)d.rows_here * (uint32_t)d.kbytes);
      const uint32_t wrows = SWIGLU ? BN / 2 : BN - 32;
      rb04 = raw_rsrc(gg.b0 + (size_t)d.n0 * d.kbytes, wrows * (uint32_t)d.kbytes);
      rb14 = raw_rsrc(SWIGLU ? gg.b1 + (size_t)d.n0 * d.kbytes : gg.b0 + (size_t)(d.n0 + 32) * d.kbytes,
                      wrows * (uint32_t)d.kbytes);
    }
    if (gg.gather != nullptr) {
      // rows past the segment end get an offset beyond the buffer and read as zero
      src_a = make_rsrc(gathered_a(gg), (uint32_t)gathered_rows(gg) * (uint32_t)d.kbytes);
#pragma unroll
      for (int j = 0; j < A_SLABS; ++j) src_voff[j] = gi[j] >= 0 ? gi[j] * d.kbytes + ld_chunk * 16 : (int)0x80000000u;
    } else {
      src_a = make_rsrc(gg.a + (size_t)d.row0 * d.kbytes, (uint32_t)d.rows_here * (uint32_t)d.kbytes);
#pragma unroll
      for (int j = 0; j < A_SLABS; ++j) src_voff[j] = (j * 64 + ld_row) * d.kbytes + ld_chunk * 16;
    }
    const uint8_t* b_half0 = gg.b0 + (size_t)d.n0 * d.kbytes;
    const uint8_t* b_half1 = SWIGLU ? gg.b1 + (size_t)d.n0 * d.kbytes : gg.b0 + (size_t)(d.n0 + 32) * d.kbytes;
    const uint32_t b_rows = SWIGLU ? BN / 2 : BN - 32;
    src_b0 = make_rsrc(b_half0, b_rows * (uint32_t)d.kbytes);
    src_b1 = make_rsrc(b_half1, b_rows * (uint32_t)d.kbytes);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int r = j * 64 + ld_row;  // row within the 128-row LDS half
      src_voff_b[j] = (SWIGLU ? r : (r >> 5) * 64 + (r & 31)) * d.kbytes + ld_chunk * 16;
    }
  };
  // K steps of the tile being loaded; a step at or past it (padding) is fetched as zeros. Step 0 of a tile is
  // requested before the tile becomes current, so the count is never below 1.
  int kt_real = 1;
  auto issue_loads = [&](int stage, int kt) {
    uint8_t* sa = smem + a_off(stage);
    uint8_t* sb = smem + b_off(stage);
    const int k0 = k_base + kt * BK;
    const __amdgpu_buffer_rsrc_t empty = make_rsrc(nullptr, 0);
    const bool pad = kt >= kt_real;
    const __amdgpu_buffer_rsrc_t ra = pad ? empty : src_a, rb0 = pad ? empty : src_b0, rb1 = pad ? empty : src_b1;
#pragma unroll
    for (int j = 0; j < A_SLABS; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr_t)(sa + ld_lds + j * 64 * BK), 16, src_voff[j], k0, 0, 0);
#pragma unroll
    for (int j = 0; j < 2; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb0, (lds_ptr_t)(sb + ld_lds + j * 64 * BK), 16, src_voff_b[j], k0, 0, 0);
#pragma unroll
    for (int j = 0; j < 2; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb1, (lds_ptr_t)(sb + ld_lds + (j + 2) * 64 * BK), 16, src_voff_b[j], k0, 0, 0);
  };

  // ---- LDS -> MFMA fragment addressing -------------------------------------------
  // Operand tile of 32 rows: lane l reads row (l&31); its K sub-block is (l>>5).
  const int fr_row = lane & 31;
  const int fr_grp = lane >> 5;
  const int fr_swz = swz(fr_row);  // tile origins are multiples of 32 rows, so f() only sees fr_row
  const int a_base = (wt * WAVE_TOK + fr_row) * BK;          // token operand within its stage, + tt*32*BK
  const int b_base = (wq * 32 + fr_row) * BK;                // weight operand within its stage, + ft*128*BK

  v16f acc[2][TT];
  // n_tt: how many of this wave's four 32-token blocks hold rows of the tile (4 except in the last, partial
  // m-tile of a segment); the others are neither read from LDS nor multiplied.
  [[maybe_unused]] auto compute = [&](int stage, auto full_c, int n_tt) {
    constexpr bool FULL = decltype(full_c)::value;
    const uint8_t* sa = smem + a_off(stage) + a_base;
    const uint8_t* sb = smem + b_off(stage) + b_base;
    if constexpr (!FP8) {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const int c0 = ((ks * 2 + fr_grp) ^ fr_swz) * 16;
        using frag_t = std::conditional_t<F16, v8h, v8bf>;
        frag_t fa[TT], fb[2];
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) {
          if (!FULL && tt >= n_tt) continue;
          fa[tt] = *reinterpret_cast<const frag_t*>(sa + tt * 32 * BK + c0);
        }
        if (!FULL && n_tt == 0) continue;
#pragma unroll
        for (int ft = 0; ft < 2; ++ft)
          fb[ft] = *reinterpret_cast<const frag_t*>(sb + ft * 128 * BK + c0);
#pragma unroll
        for (int ft = 0; ft < 2; ++ft)
#pragma unroll
          for (int tt = 0; tt < TT; ++tt) {
            if (!FULL && tt >= n_tt) continue;
            if constexpr (F16) acc[ft][tt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[ft], fa[tt], acc[ft][tt], 0, 0, 0);
            else acc[ft][tt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[ft], fa[tt], acc[ft][tt], 0, 0, 0);
          }
      }
    } else {
      // fp8: the fragments, MFMA and order over K of the assembly loop below (slice 0 then slice 1 of a step into the
      // same accumulator), scheduled by the compiler
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const int c0 = ((ks * 4 + fr_grp * 2) ^ fr_swz) * 16;
        auto frag = [&](const uint8_t* p) {
          const v4i lo = *reinterpret_cast<const v4i*>(p + c0), hi = *reinterpret_cast<const v4i*>(p + (c0 ^ 16));
          const v8i f = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
          return f;
        };
        v8i fa[TT], fb[2];
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) {
          if (!FULL && tt >= n_tt) continue;
          fa[tt] = frag(sa + tt * 32 * BK);
        }
        if (!FULL && n_tt == 0) continue;
#pragma unroll
        for (int ft = 0; ft < 2; ++ft) fb[ft] = frag(sb + ft * 128 * BK);
#pragma unroll
        for (int ft = 0; ft < 2; ++ft)
#pragma unroll
          for (int tt = 0; tt < TT; ++tt) {
            if (!FULL && tt >= n_tt) continue;
            acc[ft][tt] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fb[ft], fa[tt], acc[ft][tt], 0, 0, 0, 0, 0, 0);
          }
      }
    }
  };

  // ---- fp8: software-pipelined K loop in assembly (macros above the kernel) --------------------------------
  [[maybe_unused]] v8i fb0, fb1, fa0, fa1, fa2, fa3, fa4;
  [[maybe_unused]] uint32_t tok_addr[2][2], w_addr[2][2];  // LDS byte address of this lane's reads, [slice][16-byte half]
  if constexpr (FP8) {
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_ptr_t)smem;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int c = (((ks * 4 + fr_grp * 2) ^ fr_swz) * 16) ^ (h * 16);
        tok_addr[ks][h] = lds0 + a_base + c;
        w_addr[ks][h] = lds0 + B_OFF0 + b_base + c;
      }
  }
#define HDMOE_FRAGS3 "+{v[200:207]}"(fb0), "+{v[208:215]}"(fb1), "+{v[216:223]}"(fa0), "+{v[224:231]}"(fa1), "+{v[232:239]}"(fa2)
#define HDMOE_FRAGS3_OUT "={v[200:207]}"(fb0), "={v[208:215]}"(fb1), "={v[216:223]}"(fa0), "={v[224:231]}"(fa1), "={v[232:239]}"(fa2)
#define HDMOE_ACC_A3 [c0] "+v"(acc[0][0]), [c1] "+v"(acc[0][1]), [c2] "+v"(acc[0][2])
#define HDMOE_ACC_B3 [d0] "+v"(acc[1][0]), [d1] "+v"(acc[1][1]), [d2] "+v"(acc[1][2])
#define HDMOE_FRAGS4                                                                                           \
  "+{v[200:207]}"(fb0), "+{v[208:215]}"(fb1), "+{v[216:223]}"(fa0), "+{v[224:231]}"(fa1), "+{v[232:239]}"(fa2), \
      "+{v[240:247]}"(fa3)
#define HDMOE_FRAGS5 HDMOE_FRAGS4, "+{v[248:255]}"(fa4)
#define HDMOE_FRAGS4_OUT                                                                                       \
  "={v[200:207]}"(fb0), "={v[208:215]}"(fb1), "={v[216:223]}"(fa0), "={v[224:231]}"(fa1), "={v[232:239]}"(fa2), \
      "={v[240:247]}"(fa3)
#define HDMOE_FRAGS5_OUT HDMOE_FRAGS4_OUT, "={v[248:255]}"(fa4)
#define HDMOE_ACC_A4 [c0] "+v"(acc[0][0]), [c1] "+v"(acc[0][1]), [c2] "+v"(acc[0][2]), [c3] "+v"(acc[0][3])
#define HDMOE_ACC_B4 [d0] "+v"(acc[1][0]), [d1] "+v"(acc[1][1]), [d2] "+v"(acc[1][2]), [d3] "+v"(acc[1][3])
#define HDMOE_ACC_A5 HDMOE_ACC_A4, [c4] "+v"(acc[0][TT - 1])
#define HDMOE_ACC_B5 HDMOE_ACC_B4, [d4] "+v"(acc[1][TT - 1])
  // fragment reads of slice KS out of stage SS
#define HDMOE_SRC(KS, SS)                                                                                      \
  [w0] "v"(w_addr[KS][0]), [w1] "v"(w_addr[KS][1]), [t0] "v"(tok_addr[KS][0]), [t1] "v"(tok_addr[KS][1]),      \
      [oa] "i"((SS) * A_BYTES), [ob] "i"((SS) * B_BYTES)
  // token loads into stage TS: resource, the lane offsets of the slabs, K offset, the wave's LDS offset
#define HDMOE_TOK_LOADS(TS)                                                                                    \
  [fl] "s"(fl), [ra] "s"(ra), [so] "s"(so), [ldsd] "s"(lds_wave), [td] "i"((TS) ? A_OFF1 : 0),                 \
      [va0] "v"(src_voff[0]), [va1] "v"(src_voff[1]), [va2] "v"(src_voff[2]), [va3] "v"(src_voff[A_SLABS > 3 ? 3 : 2]), \
      [va4] "v"(src_voff[A_SLABS - 1])
  // weight loads into stage WS
#define HDMOE_W_LOADS(WS)                                                                                      \
  [fl] "s"(fl), [rb0] "s"(rb0), [rb1] "s"(rb1), [so] "s"(so), [ldsd] "s"(lds_wave),                            \
      [wd] "i"((WS) ? B_OFF1 : B_OFF0), [vb0] "v"(src_voff_b[0]), [vb1] "v"(src_voff_b[1])
  [[maybe_unused]] uint32_t lds_wave = 0;  // LDS address of this wave's rows inside a 64-row slab of stage 0's token tile
  if constexpr (FP8) lds_wave = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_ptr_t)smem + ld_lds);
  // the tile's first fragments: slice 0 of stage 0
  [[maybe_unused]] auto fp8_fill = [&] {
    if constexpr (FP8 && TT == 5) asm volatile(HDMOE_FILL5 : HDMOE_FRAGS5_OUT : HDMOE_SRC(0, 0) : "memory");
    else if constexpr (FP8 && TT == 3) asm volatile(HDMOE_FILL3 : HDMOE_FRAGS3_OUT : HDMOE_SRC(0, 0) : "memory");
    else if constexpr (FP8) asm volatile(HDMOE_FILL4 : HDMOE_FRAGS4_OUT : HDMOE_SRC(0, 0) : "memory");
  };
  [[maybe_unused]] auto fp8_a = [&] {
    if constexpr (FP8 && TT == 5) asm volatile(HDMOE_PART_A5_PLAIN : HDMOE_ACC_A5, HDMOE_FRAGS5 : : "memory");
    else if constexpr (FP8 && TT == 3) asm volatile(HDMOE_PART_A3_PLAIN : HDMOE_ACC_A3, HDMOE_FRAGS3 : : "memory");
    else if constexpr (FP8) asm volatile(HDMOE_PART_A4_PLAIN : HDMOE_ACC_A4, HDMOE_FRAGS4 : : "memory");
  };
  // part A that, if fl is set, also requests the token rows of K offset so into stage TS, one load behind each MFMA
#define HDMOE_DEF_PART_A_LOADS(NAME, TS)                                                                        \
  [[maybe_unused]] auto NAME = [&](int fl, v4i ra, int so) {                                                    \
    if constexpr (FP8 && TT == 5)                                                                               \
      asm volatile(HDMOE_SELECT(HDMOE_PART_A5_LOADS, HDMOE_PART_A5_PLAIN)                                       \
                   : HDMOE_ACC_A5, HDMOE_FRAGS5 : HDMOE_TOK_LOADS(TS) : "memory", "scc");                       \
    else if constexpr (FP8 && TT == 3)                                                                          \
      asm volatile(HDMOE_SELECT(HDMOE_PART_A3_LOADS, HDMOE_PART_A3_PLAIN)                                       \
                   : HDMOE_ACC_A3, HDMOE_FRAGS3 : HDMOE_TOK_LOADS(TS) : "memory", "scc");                       \
    else if constexpr (FP8)                                                                                     \
      asm volatile(HDMOE_SELECT(HDMOE_PART_A4_LOADS, HDMOE_PART_A4_PLAIN)                                       \
                   : HDMOE_ACC_A4, HDMOE_FRAGS4 : HDMOE_TOK_LOADS(TS) : "memory", "scc");                       \
  }
  HDMOE_DEF_PART_A_LOADS(fp8_a_loads_to0, 0);
  HDMOE_DEF_PART_A_LOADS(fp8_a_loads_to1, 1);
  // part B with the refills from slice KS of stage SS
#define HDMOE_DEF_PART_B(NAME, SS, KS)                                                                          \
  [[maybe_unused]] auto NAME = [&] {                                                                            \
    if constexpr (FP8 && TT == 5)                                                                               \
      asm volatile(HDMOE_PART_B5_PLAIN : HDMOE_ACC_B5, HDMOE_FRAGS5 : HDMOE_SRC(KS, SS) : "memory");            \
    else if constexpr (FP8 && TT == 3)                                                                          \
      asm volatile(HDMOE_PART_B3_PLAIN : HDMOE_ACC_B3, HDMOE_FRAGS3 : HDMOE_SRC(KS, SS) : "memory");            \
    else if constexpr (FP8)                                                                                     \
      asm volatile(HDMOE_PART_B4_PLAIN : HDMOE_ACC_B4, HDMOE_FRAGS4 : HDMOE_SRC(KS, SS) : "memory");            \
  }
  HDMOE_DEF_PART_B(fp8_b_s0k1, 0, 1);
  HDMOE_DEF_PART_B(fp8_b_s1k1, 1, 1);
  // second slice of an even step: refills from slice 0 of stage 1; if fl is set, the weight rows of K offset so
  // go into stage 0
  [[maybe_unused]] auto fp8_b_even = [&](int fl, v4i rb0, v4i rb1, int so) {
    if constexpr (FP8 && TT == 5)
      asm volatile(HDMOE_SELECT(HDMOE_PART_B5_LOADS, HDMOE_PART_B5_PLAIN)
                   : HDMOE_ACC_B5, HDMOE_FRAGS5 : HDMOE_SRC(0, 1), HDMOE_W_LOADS(0) : "memory", "scc");
    else if constexpr (FP8 && TT == 3)
      asm volatile(HDMOE_SELECT(HDMOE_PART_B3_LOADS, HDMOE_PART_B3_PLAIN)
                   : HDMOE_ACC_B3, HDMOE_FRAGS3 : HDMOE_SRC(0, 1), HDMOE_W_LOADS(0) : "memory", "scc");
    else if constexpr (FP8)
      asm volatile(HDMOE_SELECT(HDMOE_PART_B4_LOADS, HDMOE_PART_B4_PLAIN)
                   : HDMOE_ACC_B4, HDMOE_FRAGS4 : HDMOE_SRC(0, 1), HDMOE_W_LOADS(0) : "memory", "scc");
  };
  // second slice of an odd step: if fl is set (another pair of steps follows), refills from slice 0 of stage 0 and
  // the weight rows of K offset so go into stage 1; else it is the last slice of the tile
  [[maybe_unused]] auto fp8_b_odd = [&](int fl, v4i rb0, v4i rb1, int so) {
    if constexpr (FP8 && TT == 5)
      asm volatile(HDMOE_SELECT(HDMOE_PART_B5_LOADS, HDMOE_PART_B5_LAST)
                   : HDMOE_ACC_B5, HDMOE_FRAGS5 : HDMOE_SRC(0, 0), HDMOE_W_LOADS(1) : "memory", "scc");
    else if constexpr (FP8 && TT == 3)
      asm volatile(HDMOE_SELECT(HDMOE_PART_B3_LOADS, HDMOE_PART_B3_LAST)
                   : HDMOE_ACC_B3, HDMOE_FRAGS3 : HDMOE_SRC(0, 0), HDMOE_W_LOADS(1) : "memory", "scc");
    else if constexpr (FP8)
      asm volatile(HDMOE_SELECT(HDMOE_PART_B4_LOADS, HDMOE_PART_B4_LAST)
                   : HDMOE_ACC_B4, HDMOE_FRAGS4 : HDMOE_SRC(0, 0), HDMOE_W_LOADS(1) : "memory", "scc");
  };

  // ---- epilogue ----------------------------------------------------------------------
  // acc[ft][tt][i]: feature = (i>>2)*8 + (lane>>5)*4 + (i&3) within the 32-row MFMA tile (ft = weight half),
  // token = lane&31 within the 32-token MFMA tile: a lane owns 4 consecutive features of one token, and one store
  // instruction issued from that layout would touch 32 different rows with 8 or 16 bytes each. The packed values
  // therefore go through LDS (stage 1, free once the K loop is over) and leave as 16 bytes per lane, 8 lanes to
  // a 128-byte row piece. Staging rows are 128 bytes (256 for bf16 SwiGLU) with the 16-byte chunk index XORed
  // with (token & 7). Stores go through a buffer resource covering exactly the valid rows of the tile: rows past
  // the segment end are dropped by the range check.
  const int tok32 = lane & 31;
  const int hi32 = lane >> 5;
  // Staging room for the outputs once the K loop is over: whatever is not stage 0 (which takes the next tile's
  // first K step meanwhile). fp8: the token tile of stage 1 (BM x 128 bytes: exactly the SwiGLU tile) and the
  // weight tile of stage 1; bf16: stage 1 as a whole.
  // (three-stage ring: the token tile of stage 2; the next tile's first two K steps go to stages 0 and 1 meanwhile)
  uint8_t* const stg = smem + (RING3 ? 2 * STAGE_BYTES : FP8 ? A_OFF1 : STAGE_BYTES);
  auto wave_sync = [] {
    // orders this wave's LDS writes before its LDS reads of other lanes' data (LDS executes a wave's requests
    // in order; this only stops the compiler from moving them)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  // Per-tile epilogue factors. They are loaded before the K loop: a load issued after the next tile's
  // global->LDS requests would make the epilogue wait for those as well (one in-order counter).
  float ep_a = 1.0f, ep_b = 1.0f, ep_next = 1.0f;
  u32x2 ep_bias[2][4];  // BIAS: the 2 x 4 feature quads of this lane, 4 bf16 each
  auto load_scales = [&](const Tile& d) {
    if constexpr (BIAS) {
      const GemmGroup& gg = args.g[d.g];
#pragma unroll
      for (int ft = 0; ft < 2; ++ft)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          u32x2 z = {0u, 0u};
          if (gg.bias != nullptr)
            z = *reinterpret_cast<const u32x2*>(gg.bias + d.n0 + wq * 64 + ft * 32 + q * 8 + (lane >> 5) * 4);
          ep_bias[ft][q] = z;
        }
    }
    if constexpr (FP8) {
      const GemmGroup& gg = args.g[d.g];
      const float s_in = gg.s_in ? *gg.s_in : 1.0f;
      ep_a = s_in * *gg.sb0;
      if constexpr (SWIGLU) {
        ep_b = (gg.s_in_b ? *gg.s_in_b : s_in) * *gg.sb1;
        ep_next = gg.s_next ? hdmoe_dev_round_bf16(__fdiv_rn(1.0f, *gg.s_next)) : -1.0f;
      }
    }
  };
  auto round2_bf16 = [](float& a, float& b) {
    const uint32_t p = hdmoe_dev_pack_bf16(a, b);
    a = __uint_as_float(p << 16);
    b = __uint_as_float(p & 0xffff0000u);
  };
  auto epilogue = [&](const Tile& d) {
    const GemmGroup& gg = args.g[d.g];
    if constexpr (SWIGLU) {
      const float sg = ep_a, su = ep_b, inv_next = ep_next;
      constexpr int EB = FP8 ? 1 : 2;
      constexpr int ROWB = (BN / 2) * EB;  // bytes of one staged token row: the tile's 128 features
      const int ldo = gg.n_out * EB;
      const __amdgpu_buffer_rsrc_t ro = make_rsrc(gg.out + (size_t)d.row0 * ldo, (uint32_t)d.rows_here * (uint32_t)ldo);
      // The cast in front of the w2 Linear (ops.py:337-343) has three forms, fixed per tile: clamp to +-448 when
      // that Linear has no scale_input, nothing when 1/scale_input is 1, else multiply and round. The choice is
      // made once, outside the element loop.
      // bf16 with the 320-token tile: 320 rows of 256 bytes are more than stage 1 holds, so the tile is staged and
      // stored in two passes, the first three 32-token blocks of either wave row, then the last two.
      constexpr bool TWO_PASS = !FP8 && TT == 5;
      auto swiglu_tile = [&](auto next_mode, auto pass_c) {
        constexpr int NEXT = decltype(next_mode)::value;  // 0 clamp, 1 unit scale, 2 general scale
        constexpr int PASS = decltype(pass_c)::value;     // -1: all blocks in one go; 0, 1: the passes of TWO_PASS
        constexpr int TT0 = PASS == 1 ? 3 : 0, TT1 = PASS == 0 ? 3 : TT;
#pragma unroll
        for (int tt = TT0; tt < TT1; ++tt) {
          const int tok = PASS < 0 ? wt * WAVE_TOK + tt * 32 + tok32 : wt * ((TT1 - TT0) * 32) + (tt - TT0) * 32 + tok32;
          uint8_t* const row = stg + tok * ROWB;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            float m[4];
            uint32_t pm[2];  // the same four values as packed bf16 pairs (fp8 cast without unpacking them again)
#pragma unroll
            for (int i = 0; i < 4; i += 2) {
              // two elements at a time: one packed conversion rounds both to bf16
              float h1a = acc[0][tt][q * 4 + i] * sg, h1b = acc[0][tt][q * 4 + i + 1] * sg;   // w1(x)
              float h3a = acc[1][tt][q * 4 + i] * su, h3b = acc[1][tt][q * 4 + i + 1] * su;   // w3(x)
              round2_bf16(h1a, h1b);
              round2_bf16(h3a, h3b);
              float sa = h1a * __builtin_amdgcn_rcpf(1.0f + __expf(-h1a));                     // silu(.)
              float sb = h1b * __builtin_amdgcn_rcpf(1.0f + __expf(-h1b));
              round2_bf16(sa, sb);
              float ma = sa * h3a, mb = sb * h3b;                                              // silu(.) * w3(x)
              if constexpr (FP8 && NEXT == 1) {
                pm[i / 2] = hdmoe_dev_pack_bf16(ma, mb);  // the rounding to bf16; cast from the packed pair below
              } else {
                round2_bf16(ma, mb);
              }
              if constexpr (FP8 && NEXT == 2) {
                ma *= inv_next;
                mb *= inv_next;
                pm[i / 2] = hdmoe_dev_pack_bf16(ma, mb);
              }
              if constexpr (FP8 && NEXT == 0) {
                ma = ma < -448.0f ? -448.0f : (ma > 448.0f ? 448.0f : ma);
                mb = mb < -448.0f ? -448.0f : (mb > 448.0f ? 448.0f : mb);
              }
              m[i] = ma;
              m[i + 1] = mb;
            }
            const int byte = (wq * 32 + q * 8 + hi32 * 4) * EB;  // position of the 4 features in the staged row
            uint8_t* const dst = row + ((((byte >> 4) ^ (tok32 & 7)) << 4) | (byte & 15));
            if constexpr (FP8 && NEXT != 0) {
              *reinterpret_cast<uint32_t*>(dst) = hdmoe_dev_pack4_e4m3fn_bf16(pm[0], pm[1]);
            } else if constexpr (FP8) {
              *reinterpret_cast<uint32_t*>(dst) = hdmoe_dev_pack4_e4m3fn(m[0], m[1], m[2], m[3]);
            } else {
              u32x2 pk;
              pk.x = hdmoe_dev_pack_bf16(m[0], m[1]);
              pk.y = hdmoe_dev_pack_bf16(m[2], m[3]);
              *reinterpret_cast<u32x2*>(dst) = pk;
            }
          }
        }
      };
      constexpr int LANES_PER_ROW = ROWB / 16;
      constexpr int ROWS_PER_PASS = 64 / LANES_PER_ROW;
      const int c = lane % LANES_PER_ROW;
      constexpr std::integral_constant<int, -1> all_blocks{};
      if constexpr (TWO_PASS) {
        auto store_pass = [&](auto pass_c) {
          constexpr int PASS = decltype(pass_c)::value;
          constexpr int TT0 = PASS == 1 ? 3 : 0, NTT = PASS == 0 ? 3 : TT - 3;
          swiglu_tile(std::integral_constant<int, 1>{}, pass_c);
          __syncthreads();  // this pass's 2 x NTT x 32 rows are staged
#pragma unroll
          for (int p = 0; p < (NTT * 8) / ROWS_PER_PASS; ++p) {
            const int rl = wave * (NTT * 8) + p * ROWS_PER_PASS + lane / LANES_PER_ROW;    // staged row
            const int r = (rl / (NTT * 32)) * WAVE_TOK + TT0 * 32 + rl % (NTT * 32);        // row of the tile
            const v4i v = *reinterpret_cast<const v4i*>(stg + rl * ROWB + ((c ^ (rl & 7)) << 4));
            __builtin_amdgcn_raw_buffer_store_b128(v, ro, r * ldo + d.n0 * EB + c * 16, 0, 0);
          }
        };
        store_pass(std::integral_constant<int, 0>{});
        __syncthreads();  // everyone has read the first pass's rows
        store_pass(std::integral_constant<int, 1>{});
      } else {
        if constexpr (FP8) {
          const int next = __builtin_amdgcn_readfirstlane(inv_next < 0.0f ? 0 : (inv_next == 1.0f ? 1 : 2));
          if (next == 0) swiglu_tile(std::integral_constant<int, 0>{}, all_blocks);
          else if (next == 1) swiglu_tile(std::integral_constant<int, 1>{}, all_blocks);
          else swiglu_tile(std::integral_constant<int, 2>{}, all_blocks);
        } else {
          swiglu_tile(std::integral_constant<int, 1>{}, all_blocks);
        }
        __syncthreads();  // the tile's 256 x 128 outputs are staged
#pragma unroll
        for (int p = 0; p < (BM / 8) / ROWS_PER_PASS; ++p) {
          const int r = wave * (BM / 8) + p * ROWS_PER_PASS + lane / LANES_PER_ROW;
          const v4i v = *reinterpret_cast<const v4i*>(stg + r * ROWB + ((c ^ (r & 7)) << 4));
          __builtin_amdgcn_raw_buffer_store_b128(v, ro, r * ldo + d.n0 * EB + c * 16, 0, 0);
        }
      }
    } else {
      if constexpr (!BIAS) {
        if (args.nparts > 1) {
          // split K: this part's raw fp32 sums; scale and rounding happen where the parts are added up. A lane holds
          // four consecutive features of a token per accumulator quad: one 16-byte store each.
          const int ldp = gg.n_out * 4;
          float* const pb = gg.pout + (size_t)d.part * (size_t)args.part_stride + (size_t)d.row0 * gg.n_out;
          const __amdgpu_buffer_rsrc_t rp = make_rsrc(pb, (uint32_t)d.rows_here * (uint32_t)ldp);
#pragma unroll
          for (int tt = 0; tt < TT; ++tt)
#pragma unroll
            for (int ft = 0; ft < 2; ++ft)
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                v4i v;
                v.x = __float_as_int(acc[ft][tt][q * 4 + 0]);
                v.y = __float_as_int(acc[ft][tt][q * 4 + 1]);
                v.z = __float_as_int(acc[ft][tt][q * 4 + 2]);
                v.w = __float_as_int(acc[ft][tt][q * 4 + 3]);
                __builtin_amdgcn_raw_buffer_store_b128(
                    v, rp, (wt * WAVE_TOK + tt * 32 + tok32) * ldp + (d.n0 + wq * 64 + ft * 32 + q * 8 + hi32 * 4) * 4, 0, 0);
              }
          return;
        }
      }
      const float sc = ep_a;
      const int ldo = gg.n_out * 2;
      const __amdgpu_buffer_rsrc_t ro = make_rsrc(gg.out + (size_t)d.row0 * ldo, (uint32_t)d.rows_here * (uint32_t)ldo);
      // each wave stages its own 32 tokens x 64 features (128 bytes per token) at a time, two buffers in turn (TT = 3: one;
      // stage 1's token tile is too small for four waves' two, and the next tile's first step is on its way into stage 0)
      uint8_t* const mine = TT == 3 ? smem + B_OFF1 + wave * 4096
                            : FP8 ? (wave < 4 ? smem + A_OFF1 + wave * 8192 : smem + B_OFF1 + (wave - 4) * 8192)
                                : stg + wave * 8192;
      const int rd_row = lane >> 3, rd_c = lane & 7;
#pragma unroll
      for (int tt = 0; tt < TT; ++tt) {
        uint8_t* const buf = mine + (TT == 3 ? 0 : tt & 1) * 4096;
        wave_sync();  // the reads of two rounds ago (TT = 3: of the last one) are ahead of these writes
#pragma unroll
        for (int ft = 0; ft < 2; ++ft) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            u32x2 pk;
            if constexpr (BIAS) {
              // F.linear with bias: bf16(acc + bias); then F.gelu (erf form) of that bf16 tensor, rounded again
              // (/root/reference/comfy/ldm/hunyuan3dv2_1/hunyuandit.py:14-26, 44-50). fp8: the scaled-mm epilogue
              // bf16(acc * scale_input * scale_weight + bias) of fp8_linear (/root/reference/comfy/ops.py:345-346).
              const u32x2 bq = ep_bias[ft][q];
              float v[4] = {acc[ft][tt][q * 4 + 0], acc[ft][tt][q * 4 + 1], acc[ft][tt][q * 4 + 2], acc[ft][tt][q * 4 + 3]};
              {
                // product rounded to fp32 before the bias is added (no fused multiply-add), the order the CPU
                // checker and torch's own scaled matrix multiply on the CPU use
#pragma clang fp contract(off)
                if constexpr (FP8) {
#pragma unroll
                  for (int i = 0; i < 4; ++i) v[i] = v[i] * sc;
                }
                v[0] = v[0] + Act::lo(bq.x);
                v[1] = v[1] + Act::hi(bq.x);
                v[2] = v[2] + Act::lo(bq.y);
                v[3] = v[3] + Act::hi(bq.y);
              }
              if (gg.act == 1) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                  const float h = Act::round(v[i]);
                  v[i] = 0.5f * h * (1.0f + erff(h * 0.70710678118654752440f));
                }
              }
              pk.x = Act::pack(v[0], v[1]);
              pk.y = Act::pack(v[2], v[3]);
            } else {
              pk.x = hdmoe_dev_pack_bf16(acc[ft][tt][q * 4 + 0] * sc, acc[ft][tt][q * 4 + 1] * sc);
              pk.y = hdmoe_dev_pack_bf16(acc[ft][tt][q * 4 + 2] * sc, acc[ft][tt][q * 4 + 3] * sc);
            }
            *reinterpret_cast<u32x2*>(buf + tok32 * 128 + (((ft * 4 + q) ^ (tok32 & 7)) << 4) + hi32 * 8) = pk;
          }
        }
        wave_sync();
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const int r = p * 8 + rd_row;
          const v4i v = *reinterpret_cast<const v4i*>(buf + r * 128 + ((rd_c ^ rd_row) << 4));
          __builtin_amdgcn_raw_buffer_store_b128(v, ro, (wt * WAVE_TOK + tt * 32 + r) * ldo + (d.n0 + wq * 64) * 2 + rd_c * 16, 0, 0);
        }
      }
    }
  };

  // ---- persistent loop over this block's tiles ------------------------------------------------------
  // Per tile: K steps of 128 bytes through two LDS stages, one barrier per step (the loads of step kt+1 fly
  // while step kt is multiplied). The first K step of the NEXT tile is requested before the epilogue of the
  // current one, so its latency hides behind the stores.
  Tile cur = decode(0);
  if (cur.g < 0) return;
  int gi_cur[MAX_SLABS], gi_nxt[MAX_SLABS];
#pragma unroll
  for (int j = 0; j < A_SLABS; ++j) gi_nxt[j] = -1;
  load_gather(cur, gi_cur);
  set_src(cur, gi_cur);
  kt_real = cur.nkt;
  issue_loads(0, 0);
  if constexpr (RING3) {
    if (cur.nkt > 1) issue_loads(1, 1);
  }
  for (int i = 0; cur.g >= 0; ++i) {
    const int KT = cur.nkt;
    kt_real = KT;
    load_scales(cur);
    const Tile nxt = decode(i + 1);
    if (nxt.g >= 0) load_gather(nxt, gi_nxt);  // lands during the K loop
#pragma unroll
    for (int a2 = 0; a2 < 2; ++a2)
#pragma unroll
      for (int b2 = 0; b2 < TT; ++b2)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[a2][b2][r] = 0.0f;
    // fp8: two K steps per trip, the first out of stage 0, the second out of stage 1. The barrier of a step (the
    // loads of the next step have landed for everyone, everyone has read this stage) sits between the two parts
    // of the second slice, in front of the first refill from the other stage, with TT MFMAs still to issue behind
    // it: they cover the barrier skew and the LDS latency of the first new fragments. Rows past the end of a
    // partial tile are read as zeros and multiplied like the others.
    [[maybe_unused]] auto k_loop_fp8 = [&] {
      // An odd number of steps is padded with one whose loads come from an empty buffer (zeros).
      const int KTP = (KT + 1) & ~1;
      auto sgpr = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
      auto rsrc4 = [&](const v4i& r, bool real) -> v4i {  // the resource, or an empty one (every load returns zeros)
        v4i o;
        o.x = sgpr(r.x); o.y = sgpr(r.y); o.z = sgpr(real ? r.z : 0); o.w = sgpr(r.w);
        return o;
      };
      __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's part of the first stage has landed
      __syncthreads();
      issue_loads(1, 1);                   // step 1 as a burst; from step 2 on the loads sit between the MFMAs
      fp8_fill();
      for (int kt = 0; kt < KTP; kt += 2) {
        const int more = sgpr(kt + 2 < KTP ? 1 : 0);
        // step kt out of stage 0. Its first slice requests the token rows of step kt + 1 into stage 1 (the weight
        // rows of that step went out in the second slice of step kt - 1; step 1 was requested above).
        fp8_a_loads_to1(sgpr(kt > 0 ? 1 : 0), rsrc4(ra4, kt + 1 < KT), sgpr(k_base + (kt + 1) * BK));
        fp8_b_s0k1();
        fp8_a();
        __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0): my loads of step kt + 1, my reads of stage 0
        __syncthreads();
        fp8_b_even(more, rsrc4(rb04, true), rsrc4(rb14, true), sgpr(k_base + (kt + 2) * BK));  // weights of step kt + 2 -> stage 0
        // step kt + 1 out of stage 1
        fp8_a_loads_to0(more, rsrc4(ra4, true), sgpr(k_base + (kt + 2) * BK));                 // tokens of step kt + 2 -> stage 0
        fp8_b_s1k1();
        fp8_a();
        if (more) {
          __builtin_amdgcn_s_waitcnt(0x0070);
          __syncthreads();
        }
        fp8_b_odd(more, rsrc4(rb04, kt + 3 < KT), rsrc4(rb14, kt + 3 < KT), sgpr(k_base + (kt + 3) * BK));  // weights of step kt + 3 -> stage 1
      }
    };
    [[maybe_unused]] auto k_loop = [&](auto full_c, int n_tt) {
      for (int kt = 0; kt < KT; kt += 2) {
        __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's part of the stage has landed
        __syncthreads();                      // everyone's part has; everyone is done reading the other stage
        if (kt + 1 < KT) issue_loads(1, kt + 1);
        compute(0, full_c, n_tt);
        if (kt + 1 < KT) {
          __builtin_amdgcn_s_waitcnt(0x0f70);
          __syncthreads();
          if (kt + 2 < KT) issue_loads(0, kt + 2);
          compute(1, full_c, n_tt);
        }
      }
    };
    // Three stages: steps kt and kt + 1 are on their way when step kt is waited for (a wave's loads return in
    // order: its loads of step kt have landed when at most those of step kt + 1 are outstanding); behind the barrier
    // everyone has read stage (kt + 2) % 3, which held step kt - 1, and step kt + 2 is requested into it.
    [[maybe_unused]] auto k_loop3 = [&](auto full_c, int n_tt) {
      constexpr int PER_STEP = A_SLABS + 4;  // global->LDS loads of a wave per K step
      auto step = [&](int kt, int stage, int stage_next2) {
        // wait and barrier as one assembly statement: __syncthreads() carries a fence that waits for every
        // outstanding global->LDS load, the ones of step kt + 1 included
        if (kt + 1 < KT) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(PER_STEP) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" : : : "memory");
        if (kt + 2 < KT) issue_loads(stage_next2, kt + 2);
        compute(stage, full_c, n_tt);
      };
      for (int kt = 0; kt < KT; kt += 3) {
        step(kt, 0, 2);
        if (kt + 1 < KT) step(kt + 1, 1, 0);
        if (kt + 2 < KT) step(kt + 2, 2, 1);
      }
    };
    const int my_rows = __builtin_amdgcn_readfirstlane(cur.rows_here) - wt * WAVE_TOK;  // rows of the tile in this wave's half
    if constexpr (RING3) {
      if (my_rows > 32 * (TT - 1)) k_loop3(std::true_type{}, TT);
      else k_loop3(std::false_type{}, my_rows <= 0 ? 0 : (my_rows + 31) / 32);
    } else if constexpr (FP8 && !LIGHT) {
      k_loop_fp8();
    } else {
      if (my_rows > 32 * (TT - 1)) k_loop(std::true_type{}, TT);
      else k_loop(std::false_type{}, my_rows <= 0 ? 0 : (my_rows + 31) / 32);
    }
    // Every wave is done reading both stages: stage 0 can take the next tile's first K step, stage 1 the
    // staged outputs of this one (it is not loaded into again before the barrier of that K step).
    __syncthreads();
    if (nxt.g >= 0) {
      set_src(nxt, gi_nxt);
      kt_real = nxt.nkt;
      issue_loads(0, 0);
      if constexpr (RING3) {
        if (nxt.nkt > 1) issue_loads(1, 1);
      }
    }
    epilogue(cur);
    cur = nxt;
  }
}

// ---- split K: adding the parts up ---------------------------------------------------------------------------
// out[r, n] = bf16( (sum over parts of partial[p][r][n]) * scale(r) ), parts in ascending order (deterministic);
// scale(r) = scale_input * scale_weight of the Linear of the group that owns row r (fp8), 1 for bf16 weights.
// end: gate and residual of a feed-forward branch in the same pass. Dense branch of 768 rows: this kernel 8.2 us and a gate and
// residual kernel of 4.8 behind it, 8.8 together.
struct SplitKReduceArgs {
  const float* partial;     // [nparts][rows_dyn + rows_static][n_out]
  long long part_stride;
  int nparts, nparts_static, n_out, rows_dyn, rows_static, n_dyn;  // parts of the dynamic rows, of the static rows
  int scaled;               // 1: scale_input * scale_weight (fp8), 2: scale_weight rounded to bf16 (one-byte weights, bf16 arithmetic)
  const int32_t* offsets;   // segment bounds of the dynamic rows, n_dyn + 1 entries
  const float* sw[MAX_GROUPS];   // scale_weight per group (fp8); the static group is entry n_dyn
  const float* sin[MAX_GROUPS];  // scale_input per group or NULL
  uint16_t* out_dyn;        // [rows_dyn, n_out] bf16
  uint16_t* out_static;     // [rows_static, n_out] bf16
  HdmoeGatedResidual end;   // of the static rows; gate NULL = none
};

// two packed bf16 values: bf16(bf16(gate * y) + residual)
__device__ __forceinline__ uint32_t gate_and_add(uint32_t g, uint32_t y, uint32_t r) {
#pragma clang fp contract(off)
  auto lo = [](uint32_t v) { return __uint_as_float(v << 16); };
  auto hi = [](uint32_t v) { return __uint_as_float(v & 0xffff0000u); };
  const uint32_t p = hdmoe_dev_pack_bf16(lo(g) * lo(y), hi(g) * hi(y));
  return hdmoe_dev_pack_bf16(lo(p) + lo(r), hi(p) + hi(r));
}

__global__ __launch_bounds__(256) void splitk_reduce_kernel(const SplitKReduceArgs a) {
  const int rows = a.rows_dyn + a.rows_static;
  const int per_row = a.n_out / 4;  // threads per row, 4 features each
  const long long total = (long long)rows * per_row;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (long long)gridDim.x * blockDim.x) {
    const int r = (int)(i / per_row), c = (int)(i % per_row) * 4;
    int g = a.n_dyn;  // the static group
    if (r < a.rows_dyn) {
      g = 0;
      while (g + 1 < a.n_dyn && r >= a.offsets[g + 1]) ++g;
    }
    float sc = 1.0f;
    if (a.scaled == 1) sc = (a.sin[g] ? *a.sin[g] : 1.0f) * *a.sw[g];
    if (a.scaled == 2 && a.sw[g] != nullptr) sc = hdmoe_dev_round_bf16(*a.sw[g]);
    const float* src = a.partial + (size_t)r * a.n_out + c;
    float4 s = *reinterpret_cast<const float4*>(src);
    const int np = r < a.rows_dyn ? a.nparts : a.nparts_static;
    for (int p = 1; p < np; ++p) {
      const float4 t = *reinterpret_cast<const float4*>(src + (size_t)p * (size_t)a.part_stride);
      s.x += t.x; s.y += t.y; s.z += t.z; s.w += t.w;
    }
    uint2 o;
    o.x = hdmoe_dev_pack_bf16(s.x * sc, s.y * sc);
    o.y = hdmoe_dev_pack_bf16(s.z * sc, s.w * sc);
    if (a.end.gate != nullptr && r >= a.rows_dyn) {
      const int rs = r - a.rows_dyn;
      const uint2 g = *reinterpret_cast<const uint2*>(a.end.gate + (size_t)(rs / a.end.rows_per_batch) * a.n_out + c);
      const uint2 x = *reinterpret_cast<const uint2*>(a.end.residual + (size_t)rs * a.n_out + c);
      o.x = gate_and_add(g.x, o.x, x.x);
      o.y = gate_and_add(g.y, o.y, x.y);
    }
    uint16_t* dst = r < a.rows_dyn ? a.out_dyn + (size_t)r * a.n_out + c : a.out_static + (size_t)(r - a.rows_dyn) * a.n_out + c;
    *reinterpret_cast<uint2*>(dst) = o;
  }
}

void fill_segments(GemmArgs& args) {
  for (int g = 0; g < args.G; ++g) args.seg[g] = {args.g[g].row_begin, args.g[g].row_end, args.g[g].n_out, args.g[g].kbytes};
}

template <int MODE, int TT = 4, bool LIGHT = false>
int launch_grouped(GemmArgs& args, int tile_bound, hipStream_t s, const char* what) {
  // The opt-in for more than 64 KiB of dynamic LDS is a per-device function attribute: remembered per device
  // and instantiation (a race between two threads sets it twice, which is harmless).
  constexpr int SMEM = TileCfg<TT>::SMEM + (MODE == FP8_SWIGLU && LIGHT ? (HDMOE_ROUTE_SLOTS + NTHREADS / 64 * HDMOE_MAX_EXPERTS) * 4 : 0);
  static_assert(SMEM <= 160 * 1024, "a CU's LDS");
  static bool attr_set[64] = {};
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64) device = -1;
  if (device < 0 || !attr_set[device]) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&grouped_gemm_kernel<MODE, TT, LIGHT>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, SMEM);
    if (e != hipSuccess) return hdmoe_fail(HDMOE_E_LAUNCH, "%s: hipFuncSetAttribute: %s", what, hipGetErrorString(e));
    if (device >= 0) attr_set[device] = true;
  }
  if (tile_bound <= 0) return HDMOE_OK;
  fill_segments(args);
  // persistent blocks: one per CU (128 KiB of LDS allow no second one), a multiple of the XCD count
  int grid = (tile_bound + HDMOE_NUM_XCD - 1) / HDMOE_NUM_XCD * HDMOE_NUM_XCD;
  if (grid > HDMOE_NUM_CU) grid = HDMOE_NUM_CU;
  hipLaunchKernelGGL((grouped_gemm_kernel<MODE, TT, LIGHT>), dim3(grid), dim3(NTHREADS), SMEM, s, args);
  return hdmoe_check_launch(what);
}

#include "gemm4w.h"
#include "swiglu4w.h"
#include "swiglu224.h"

// Bytes that the parts of tail tiles take in a launch, 0: none is cut. n_dyn groups with rows_mean rows each when the routing is
// even (their real sizes are known on the device only), and rows_static of one more; kb: K in bytes of 16-bit activations. Whether
// tiles may get cut: by the plan of an even routing, and of one whose experts are two standard deviations (counts are about
// binomial) below or above it. Without dynamic groups the three are the same and the plan is known here.
size_t g4_tail_room(int n_dyn, int rows_mean, int n_out_dyn, int kb_dyn, int rows_static, int n_out_static, int kb_static,
                    int feat, bool w8) {
  if (n_dyn > 0 && rows_static > 0 && kb_dyn != kb_static) return 0;   // tiles of two lengths: one cut does not even them out
  const int kb = n_dyn > 0 ? kb_dyn : kb_static, min_pairs = w8 ? 3 : 2;
  if (kb % (2 * BK) != 0 || kb / (2 * BK) < min_pairs) return 0;
  size_t most = 0;
  for (int k = n_dyn > 0 ? -1 : 1; k <= 1; ++k) {
    long tiles = 0, padding = 0;
    auto add = [&](int groups, int rows, int n_out) {
      const long mt = (rows + G4_BM - 1) / G4_BM, nt = (long)groups * (n_out / feat);
      tiles += mt * nt;
      padding += (mt * G4_BM - rows) * nt;
    };
    if (n_dyn > 0) add(n_dyn, max(0, rows_mean + k * (int)(2 * sqrt((double)rows_mean))), n_out_dyn);
    if (rows_static > 0) add(1, rows_static, n_out_static);
    if (tiles <= 0 || tiles > 24 * HDMOE_NUM_CU) continue;             // one round of more than 24 is not worth a launch
    const G4Tail t = g4_plan_tail((int)tiles, HDMOE_NUM_CU, kb / (2 * BK), min_pairs, (int)padding);
    if (t.parts > 1) most = n_dyn > 0 ? G4_TAIL_BYTES : (size_t)t.parts * t.tiles * G4_BM * 256 * 4;
  }
  return most;
}

// Whether tiles of two lengths are dealt out by g4_two_lengths: up to seven quarters of a round of the long ones (measured there).
bool g4_two_pays(const GemmArgs& args, int rows_mean) {
  long longs = 0;
  for (int g = 0; g < args.G; ++g) {
    const GemmGroup& gg = args.g[g];
    if ((gg.row_begin < 0) == (args.spread > 0)) longs += (long)((gg.row_begin < 0 ? rows_mean : gg.row_end - gg.row_begin) + G4_BM - 1) / G4_BM * (gg.n_out / BN);
  }
  return 4 * longs <= 7 * HDMOE_NUM_CU;
}

template <G4Type TY, int EPI>
int launch_gemm4w(GemmArgs& args, int rows_mean, hipStream_t s, const char* what) {
  constexpr int FEAT = EPI == G4_SWIGLU ? 128 : 256;
  static bool attr_set[64] = {};
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64) device = -1;
  if (device < 0 || !attr_set[device]) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm4w_kernel<TY, EPI>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, G4_SMEM);
    if (e != hipSuccess) return hdmoe_fail(HDMOE_E_LAUNCH, "%s: hipFuncSetAttribute: %s", what, hipGetErrorString(e));
    if (device >= 0) attr_set[device] = true;
  }
  fill_segments(args);
  if (EPI == G4_PARTIAL || TY == G4_F8) args.tail = nullptr;
  if (args.tail != nullptr) {
    const GemmGroup& first = args.g[0];
    const GemmGroup& last = args.g[args.G - 1];
    const bool has_static = last.row_begin >= 0;   // at most one static group, the last
    if (g4_tail_room(has_static ? args.G - 1 : args.G, rows_mean, first.n_out, first.kbytes,
                     has_static ? last.row_end - last.row_begin : 0, last.n_out, last.kbytes, FEAT, TY == G4_W8) == 0)
      args.tail = nullptr;
  }
  args.cap = args.spread != 0 ? (g4_two_pays(args, rows_mean) ? -1 : 0) : g4_host_cap(args, FEAT, TY == G4_W8 ? 3 : 2, HDMOE_NUM_CU);
  // one block per CU whatever the number of tiles: a block without any ends at once
  hipLaunchKernelGGL((gemm4w_kernel<TY, EPI>), dim3(HDMOE_NUM_CU), dim3(G4_THREADS), G4_SMEM, s, args);
  if constexpr (EPI != G4_PARTIAL && TY != G4_F8) {
    if (args.tail != nullptr)
      hipLaunchKernelGGL((gemm4w_tail_kernel<TY, EPI>), dim3(4 * HDMOE_NUM_CU), dim3(256), 0, s, args, HDMOE_NUM_CU);
  }
  return hdmoe_check_launch(what);
}

int launch_swiglu4w(GemmArgs& args, int tile_bound, hipStream_t s, const char* what) {
  static bool attr_set[64] = {};
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64) device = -1;
  if (device < 0 || !attr_set[device]) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&swiglu4w_kernel),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, W4_SMEM);
    if (e != hipSuccess) return hdmoe_fail(HDMOE_E_LAUNCH, "%s: hipFuncSetAttribute: %s", what, hipGetErrorString(e));
    if (device >= 0) attr_set[device] = true;
  }
  if (tile_bound <= 0) return HDMOE_OK;
  fill_segments(args);
  int grid = (tile_bound + HDMOE_NUM_XCD - 1) / HDMOE_NUM_XCD * HDMOE_NUM_XCD;
  if (grid > HDMOE_NUM_CU) grid = HDMOE_NUM_CU;
  hipLaunchKernelGGL(swiglu4w_kernel, dim3(grid), dim3(W4_THREADS), W4_SMEM, s, args);
  return hdmoe_check_launch(what);
}

template <bool CLAMP>
int launch_swiglu224(GemmArgs& args, hipStream_t s, const char* what) {
  static bool attr_set[64] = {};
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64) device = -1;
  if (device < 0 || !attr_set[device]) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&swiglu224_kernel<CLAMP>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, S224_SMEM);
    if (e != hipSuccess) return hdmoe_fail(HDMOE_E_LAUNCH, "%s: hipFuncSetAttribute: %s", what, hipGetErrorString(e));
    if (device >= 0) attr_set[device] = true;
  }
  fill_segments(args);
  // one block per CU whatever the number of tiles: a block without any ends at once
  hipLaunchKernelGGL(swiglu224_kernel<CLAMP>, dim3(HDMOE_NUM_CU), dim3(G4_THREADS), S224_SMEM, s, args);
  return hdmoe_check_launch(what);
}

// bytes of an activation
inline int elem_bytes(int weight_dtype) { return weight_dtype == HDMOE_W_E4M3FN ? 1 : 2; }

int check_dtype(int weight_dtype, const char* what, bool upcast_ok = false) {
  if (upcast_ok && weight_dtype == HDMOE_W_E4M3FN_UPCAST) return HDMOE_OK;
  if (weight_dtype != HDMOE_W_BF16 && weight_dtype != HDMOE_W_E4M3FN)
    return hdmoe_fail(HDMOE_E_SHAPE, "%s: weight_dtype=%d is neither HDMOE_W_BF16 nor HDMOE_W_E4M3FN", what, weight_dtype);
  return HDMOE_OK;
}

}  // namespace

// ---- which kernel runs a feed-forward contraction ---------------------------------------------------------------
// Two process-wide switches choose between kernels with the same results bit for bit (hdmoe_set_kernel_form). Their
// initial values come from the environment variables HDMOE_SWIGLU4W / HDMOE_LIGHT, read once ("0" = never, anything
// else = always, unset = the launcher's own rule).
namespace {
std::atomic<int> g_form[HDMOE_NUM_FORMS] = {{HDMOE_FORM_AUTO}, {HDMOE_FORM_AUTO}};
std::once_flag g_form_once;
void form_init() {
  static const char* const names[HDMOE_NUM_FORMS] = {"HDMOE_SWIGLU4W", "HDMOE_LIGHT"};
  for (int i = 0; i < HDMOE_NUM_FORMS; ++i) {
    const char* v = getenv(names[i]);
    if (v != nullptr) g_form[i].store(v[0] == '0' ? HDMOE_FORM_NEVER : HDMOE_FORM_ALWAYS, std::memory_order_relaxed);
  }
}
int form_of(int which) {
  std::call_once(g_form_once, form_init);
  return g_form[which].load(std::memory_order_relaxed);
}

// The kernels a contraction of the feed-forward can run on.
enum GemmForm {
  FORM_SPLIT_K,    // plain modes cut along K (few tiles); its own choice of tile inside
  FORM_RING3,      // 128-token tiles, three LDS stages, token blocks without rows skipped
  FORM_LIGHT4,     // 256-token tiles, token blocks without rows skipped
  FORM_W4,         // fp8 gate/up: the 4-wave kernel (256-token tiles)
  FORM_TALL5,      // 320-token tiles
  FORM_SHORT3,     // 192-token tiles (fp8 gate/up)
  FORM_S224,       // fp8 gate/up: the 4-wave kernel on 224-token tiles (swiglu224.h)
  FORM_BASE4       // 256-token tiles
};

struct GemmShape {
  bool swiglu, fp8, split, w8;
  int rows_dyn, n_dyn, rows_static;  // rows_static = 0: no static group
  int N_dyn, N_static;
  int kbytes;                        // K of a gate/up contraction in bytes
  bool w4_fits;                      // the 4-wave kernel takes these operands (swiglu4w_fits)
  bool s224_fits;                    // the one on 224-token tiles does (swiglu224_fits)
  bool g4_takes;                     // K is of the kind that gemm4w_kernel takes
};

// Expected tiles with evenly loaded experts, static round-robin over the CUs, and a fixed cost per tile of about one
// 32-token block: rounds x (TT + 1). The taller tile wins when it does not add a round.
long expected_tiles_of(const GemmShape& sh, int bm) {
  const int fpt = sh.swiglu ? BN / 2 : BN;
  long tiles = 0;
  if (sh.n_dyn > 0) tiles += (long)sh.n_dyn * ((sh.rows_dyn / sh.n_dyn + bm - 1) / bm) * (sh.N_dyn / fpt);
  if (sh.rows_static > 0) tiles += (long)((sh.rows_static + bm - 1) / bm) * (sh.N_static / fpt);
  return tiles;
}
long expected_tiles(const GemmShape& sh, int tt) { return expected_tiles_of(sh, 64 * tt); }
long expected_tile_cost(const GemmShape& sh, int tt) {
  return ((expected_tiles(sh, tt) + HDMOE_NUM_CU - 1) / HDMOE_NUM_CU) * (tt + 1);
}

// The 192-token tile for fp8 gate/up: only without routed groups (a dense feed-forward). Where it saves a round's height there:
// 768 tokens by 6912 features, whole branch 86.1 -> 77.4 us, 300 tokens 78.1 -> 69.0, 1500 tokens 132.2 -> 127.6. With experts of
// uneven size the model says the same and is wrong (layer of 768 tokens 183.8 -> 189.8 us, 384 tokens 140.1 -> 141.5). It has to
// pay by 15 %: the 4-wave kernel hides part of its epilogue, which the model does not know.
bool short_tile_pays(const GemmShape& sh) {
  if (!sh.fp8 || !sh.swiglu || sh.split || sh.n_dyn > 0) return false;
  const long c4 = expected_tile_cost(sh, 4), c5 = expected_tile_cost(sh, 5);
  return 20 * expected_tile_cost(sh, 3) <= 17 * (c4 < c5 ? c4 : c5);
}

// Whether fp8 gate/up runs on 224-token tiles (tt: height of the other kernel's tiles in blocks of 64). Both sides are rounds of tiles, in
// hundredths of a round of high 224-token tiles (s224_price, with the kernel's choice of styles) and in units of expected_tile_cost; a round here
// takes 70 / 21 of them (8192 tokens: 28.8 us, the 320-token tile of 6 units 45), and 15 / 21 go for the last tile's activation, which nothing
// hides. Segments are taken even, and a standard deviation apart (tokens that go to 2 of n experts), half the price each: 512 tokens on 4 experts
// are not 4 tiles of 256. A tile of the other kernel that is not full costs up to a quarter less: zeros take little power, and the clock follows.
// Whole pass, us, the other kernel, this one (weights from memory): layers of 4 experts, 257 tokens 107 112 (left to the other up to 320), 350 129
// 111, 512 133 132, 700 165 143, 1024 188 177, 4096 493 452; 8 experts, 400 174 168, 500 179 190 (other), 1000 229 228, 1300 310 252; 6 experts,
// 700 170 178 (other), 950 245 203; 16 experts, 1950 387 398 (other), 2200 478 435; width 4096, 617 303 277; dense, 400 rows 50.7 49.5, 577 55.0
// 57.4 (other: 513 to 768), 950 73 74 (other: 897 to 1280), 1300 88 85, 2200 113 117 (other: 2049 to 2304), 3584 162 158, 4096 187 169; 32768
// features, 480 rows 136 145 (other). Where it errs: width 4096, 448 tokens 217 232; 4 experts without a shared one, 993 tokens 144 150.
// A dense feed-forward of up to 384 rows stays on 192-token tiles, where low tiles would be faster (Linears with and without scale_input, 257 rows
// 49.2 47.3, 300 50.2 47.9, 384 52.7 49.2): tests/test_gpu_fp8_dense_tiles.py has 300 rows of that width on them. And one or two groups are taken
// at s224_cost, without the price of weights read again (two experts of 16384 features, 452 tokens: 125.7 132.0): tests/test_gpu_swiglu224.py has
// such sizes on this kernel.
bool s224_pays(const GemmShape& sh, int tt) {
  double price = 0, other = 0;
  for (int spread = 0; spread < 2; ++spread) {
    struct { int rows, cols; } part[3];   // segments of one size: rows of each, tiles along the features of all of them
    int n = 0;
    if (sh.n_dyn > 0) {
      const int mean = (sh.rows_dyn + sh.n_dyn - 1) / sh.n_dyn, cols = sh.N_dyn / S224_FEAT;
      const int sd = spread == 0 || sh.n_dyn <= 2 ? 0 : (int)lround(sqrt((double)mean * (sh.n_dyn - 2) / sh.n_dyn));
      part[n++] = {mean + sd, (sh.n_dyn + 1) / 2 * cols};
      part[n++] = {mean > sd ? mean - sd : 0, sh.n_dyn / 2 * cols};
    }
    const int n_routed = n;
    if (sh.rows_static > 0) part[n++] = {sh.rows_static, sh.N_static / S224_FEAT};
    int cols = 0, shift = 4;
    for (int i = 0; i < n; ++i) cols += part[i].cols;
    int best = 0, whole = 0;   // the kernel's own choice of styles (tile_mix)
    for (int c = 0; c < S224_STYLES * S224_STYLES; ++c) {
      S224Tiles tiles = {0, 0, 0, 0};
      for (int i = 0; i < n; ++i) s224_add(tiles, s224_mix(part[i].rows, i < n_routed ? c / S224_STYLES : c % S224_STYLES), part[i].cols);
      if (c == 0) shift = s224_shift(cols, sh.kbytes, tiles.highs);
      const int p = sh.n_dyn == 1 || sh.n_dyn == 2 ? s224_cost(tiles.highs, tiles.lows) : s224_price(tiles, shift);
      if (c == 0) {
        whole = best = p;
        if (tiles.highs > S224_TILES || (sh.n_dyn <= 0 && sh.rows_static <= 2 * TileCfg<3>::BM)) break;
      } else if (s224_low_pays(p, whole) && p < best) {
        best = p;
      }
    }
    price += 0.5 * best;
    long tiles = 0;
    double rows = 0;
    for (int i = 0; i < n; ++i) {
      tiles += (long)((part[i].rows + 64 * tt - 1) / (64 * tt)) * part[i].cols;
      rows += (double)part[i].rows * part[i].cols;
    }
    if (tiles > 0) other += 0.5 * ((tiles + HDMOE_NUM_CU - 1) / HDMOE_NUM_CU) * (tt + 1) * (0.75 + 0.25 * rows / (64.0 * tt * tiles));
  }
  return 70 * price + 15 * S224_HIGH <= 21 * S224_HIGH * other;
}

// light: the token blocks of a tile that hold no rows are skipped (fp8: the compiler-scheduled K loop instead of the
// assembly loop, which multiplies padding like rows; 16-bit weights always skip them and take from this only the
// three-stage ring).
// fp8_g4: an fp8 contraction without activation runs on gemm4w_kernel (cut along K or not).
struct FormChoice { GemmForm form; bool light, ring16, tall, one_round5, short3, fp8_g4; };
FormChoice pick_form(const GemmShape& sh) {
  const int f_light = form_of(HDMOE_FORM_LIGHT), f_4w = form_of(HDMOE_FORM_SWIGLU4W);
  const bool few_rows = hdmoe_few_rows(sh.rows_dyn, sh.n_dyn, sh.rows_static);
  FormChoice c;
  // forcing the 4-wave kernel also keeps the light form's default off
  c.light = sh.fp8 && (f_light != HDMOE_FORM_AUTO ? f_light == HDMOE_FORM_ALWAYS
                                                   : few_rows && !(sh.swiglu && f_4w == HDMOE_FORM_ALWAYS));
  c.ring16 = !sh.fp8 && !sh.w8 && few_rows && f_light != HDMOE_FORM_NEVER;
  // (16-bit weights: where the taller tile fits one round of blocks and the 256-token tile needs a second, e.g. 257 to 320
  // tokens of a layer with a shared expert: 93 against 96 us in the gate/up contraction)
  c.one_round5 = !sh.fp8 && !sh.w8 && sh.swiglu && expected_tiles(sh, 5) <= HDMOE_NUM_CU && expected_tiles(sh, 4) > HDMOE_NUM_CU;
  // (16-bit weights: the gate/up contraction that stays with the 8-wave kernel, 2560 rows of 4 experts by 6912 features, K = 2624: 178
  // against 198 us; the down projection measured slower on the taller tile)
  c.tall = (sh.fp8 || (sh.swiglu && !sh.g4_takes)) && !sh.split && !c.light && expected_tile_cost(sh, 5) < expected_tile_cost(sh, 4);
  // fp8 down projection on the 4-wave kernel. Whole layer, 8- against 4-wave, us: cut along K 260 tokens 110, 103; 600 177, 169; 1024 226, 207; 1536
  // 254, 240; 2000 304, 284; whole tiles 4000 537, 503; 5000 649, 624 (the 8-wave kernel's 320-token tiles would take 0.8 of the rounds of whole
  // 256-token ones); 8000 969, 917. With 0.6 of their rounds too, now that tiles are as high as their rows need and of two lengths: 2100 tokens 279, 252;
  // 2300 299, 279; 2560 346, 303, skewed 352, 306; dense branch of 6700 rows 300.1, 301.7, 8000 346.9, 344.3. Not with a forced form: the parts of a cut
  // projection end elsewhere here (on pairs of K steps); uncut the bytes are the same.
  c.fp8_g4 = sh.fp8 && !sh.swiglu && sh.g4_takes && !c.light && f_light == HDMOE_FORM_AUTO && f_4w == HDMOE_FORM_AUTO;
  if (c.fp8_g4) c.tall = false;
  c.short3 = !c.light && f_4w != HDMOE_FORM_ALWAYS && short_tile_pays(sh);
  if (f_light == HDMOE_FORM_AUTO && f_4w == HDMOE_FORM_AUTO && !c.light &&
      sh.fp8 && sh.swiglu && sh.s224_fits && s224_pays(sh, c.short3 ? 3 : c.tall ? 5 : 4)) {
    c.tall = c.short3 = false;
    c.form = FORM_S224;
    return c;
  }
  if (c.short3) { c.tall = false; c.form = FORM_SHORT3; return c; }
  if (sh.split) { c.form = FORM_SPLIT_K; return c; }
  // Light form, gate/up: with every segment inside one 128-token tile (up to 128 tokens in a top-2 layer of 4 experts)
  // the three-stage ring of the down projection pays here too (whole layer 78 -> 73 us at 16 tokens, 80 -> 75 at 128;
  // at 256 tokens the shared expert's second m-tile costs more than the ring gains: 93 -> 105 us).
  if ((c.light || c.ring16) && sh.swiglu && sh.rows_static <= TileCfg<2>::BM &&
      (sh.n_dyn <= 0 || sh.rows_dyn <= TileCfg<2>::BM / 2 * sh.n_dyn)) {
    c.form = FORM_RING3;
    return c;
  }
  if (c.light) { c.form = FORM_LIGHT4; return c; }
  // The 4-wave form of the gate/up kernel on 256-token tiles (swiglu4w.h) takes the launch where neither the 224-token nor the
  // 320-token tile does (2-3 % faster there than the 8-wave kernel: part of its epilogue hides in the K loop).
  const bool want4w = f_4w != HDMOE_FORM_AUTO ? f_4w == HDMOE_FORM_ALWAYS : !c.tall;
  if (sh.fp8 && sh.swiglu && want4w && sh.w4_fits) { c.form = FORM_W4; return c; }
  c.form = c.tall ? FORM_TALL5 : FORM_BASE4;
  return c;
}

// The form of a gate/up contraction that does its own dispatch: a light one by the sizes alone.
FormChoice routing_form(const GemmShape& sh) {
  FormChoice c = {};
  c.light = true;
  c.form = sh.rows_static <= TileCfg<2>::BM && sh.rows_dyn <= TileCfg<2>::BM / 2 * sh.n_dyn ? FORM_RING3 : FORM_LIGHT4;
  return c;
}

// Whether gate/up on 16-bit activations runs on the 4-wave kernel: what fits it, but for the three-stage ring (every segment inside a 128-token
// tile) and the case one_round5 (hdmoe_launch_ffn_gemm). Of the ring's sizes a dense feed-forward goes to the 4-wave kernel where that cuts its
// tiles along K (has_room: the working memory holds the parts), so that more of the CUs fetch weights. Whole branch in bf16, us, ring -> cut: 2560 x
// 6912 (54 tiles in 4 parts), 1 row 59.3 -> 47.9, 64 67.0 -> 54.1, 128 79.4 -> 61.4; 2560 x 1024, 64 38.7 -> 32.8; 4096 x 11008 (2 parts) 96.0 -> 89.4; 5120 x
// 13824 (2 parts) 134.4 -> 116.6. Not cut, ring and 4-wave kernel: 2560 x 6912 without the room, 64 rows 66.9 72.9; 512 x 6912 28.3 30.8; 2560 x 16384,
// 64 rows 91.2 96.2; 2560 x 32768 138.7 141.8. (512 x 256, which are two tiles, 18.3 20.8: under a tile for each XCD it is the launch that counts, and
// tests/test_gpu_dense_few_rows.py has these on the 4-wave kernel.)
bool swiglu_on_g4(const GemmShape& sh, bool has_room) {
  if (sh.fp8 || !sh.g4_takes) return false;
  if (sh.w8) return true;
  if (hdmoe_few_rows(sh.rows_dyn, sh.n_dyn, sh.rows_static) && sh.rows_static <= TileCfg<2>::BM &&
      (sh.n_dyn <= 0 || sh.rows_dyn <= TileCfg<2>::BM / 2 * sh.n_dyn)) {
    if (sh.n_dyn > 0) return false;
    return sh.N_static / (BN / 2) < HDMOE_NUM_XCD ||
           (has_room && g4_tail_room(0, 0, 0, 0, sh.rows_static, sh.N_static, sh.kbytes, BN / 2, false) > 0);
  }
  return !pick_form(sh).one_round5;
}

// Whether the 4-wave kernel takes contractions of these lengths (rows = 0: no such group)
bool g4_takes_k(int rows_dyn, int kb_dyn, int rows_static, int kb_static) {
  auto ok = [](int rows, int kb) { return rows <= 0 || (kb % (2 * BK) == 0 && kb >= 4 * BK); };
  return ok(rows_dyn, kb_dyn) && ok(rows_static, kb_static);
}
}  // namespace

// Whether the gate/up contraction of a layer can do its own dispatch (HdmoeRoute): what runs on the light form, a slot per thread.
bool hdmoe_gate_up_routes(int weight_dtype, int rows_dyn, int n_dyn, int rows_static, int N_dyn, int N_static) {
  if (weight_dtype != HDMOE_W_E4M3FN || n_dyn <= 0 || rows_dyn > HDMOE_ROUTE_SLOTS) return false;
  GemmShape sh = {};
  sh.swiglu = sh.fp8 = true;
  sh.rows_dyn = rows_dyn; sh.n_dyn = n_dyn; sh.rows_static = rows_static;
  sh.N_dyn = N_dyn; sh.N_static = N_static;
  return pick_form(sh).light;
}

extern "C" int hdmoe_set_kernel_form(int which, int value) {
  if (which < 0 || which >= HDMOE_NUM_FORMS || value < HDMOE_FORM_AUTO || value > HDMOE_FORM_ALWAYS)
    return hdmoe_fail(HDMOE_E_SHAPE, "hdmoe_set_kernel_form: which=%d value=%d", which, value);
  std::call_once(g_form_once, form_init);
  g_form[which].store(value, std::memory_order_relaxed);
  return HDMOE_OK;
}

extern "C" int hdmoe_get_kernel_form(int which) {
  if (which < 0 || which >= HDMOE_NUM_FORMS) return hdmoe_fail(HDMOE_E_SHAPE, "hdmoe_get_kernel_form: which=%d", which);
  return form_of(which);
}

// Shared by hdmoe_grouped_swiglu / hdmoe_grouped_down / hdmoe_linear / hdmoe_moe_ffn.
// groups: n_dyn experts with device-side segments, optionally one static group (the shared expert).
// end (optional): gate and residual behind a down projection that is cut along K and added up here (partial, reduce).
// gather_dyn (optional): the routed rows are not materialised in segment order; row r of the segments is row
// gather_dyn[r] of a_dyn, which holds gather_rows rows.
int hdmoe_launch_ffn_gemm(bool swiglu, int weight_dtype, const uint8_t* a_dyn, const int32_t* offsets, int rows_dyn,
                          int n_dyn, const hdmoe_ffn_weights* experts, uint8_t* out_dyn, const uint8_t* a_static,
                          int rows_static, const hdmoe_ffn_weights* shared, uint8_t* out_static, int K_dyn, int N_dyn,
                          int K_static, int N_static, hipStream_t s, const char* what,
                          const int32_t* gather_dyn = nullptr, int gather_rows = 0, float* partial = nullptr,
                          int nparts = 1, int gather_shift = 0, bool reduce = true,
                          const HdmoeSplitPlan* plan = nullptr, const HdmoeAltOperand* alt = nullptr,
                          float* tail = nullptr, const HdmoeGatedResidual* end = nullptr, const HdmoeRoute* route = nullptr) {
  const bool w8 = weight_dtype == HDMOE_W_E4M3FN_UPCAST;  // one-byte weights, 16-bit arithmetic
  const int eb = elem_bytes(weight_dtype);
  const bool fp8 = weight_dtype == HDMOE_W_E4M3FN;
  const int feat_per_tile = swiglu ? BN / 2 : BN;
  // Split K (on the 128-token tile of the light form; fp8 on the 4-wave kernel: tiles of plan->bm tokens, 128 to 256; else the
  // 256-token tile): nparts = the most parts any entry of the plan cuts a tile into (the partial-sum buffer holds that many); no plan =
  // every tile in nparts parts
  const bool split = !swiglu && partial != nullptr && nparts > 1;
  GemmShape shape;
  shape.swiglu = swiglu; shape.fp8 = fp8; shape.split = split; shape.w8 = w8;
  shape.rows_dyn = rows_dyn; shape.n_dyn = n_dyn; shape.rows_static = shared != nullptr ? rows_static : 0;
  shape.N_dyn = N_dyn; shape.N_static = N_static;
  shape.w4_fits = true;  // settled below, once the groups are filled in
  const int K_any = n_dyn > 0 ? K_dyn : K_static;
  shape.kbytes = K_any * eb;
  shape.s224_fits = fp8 && swiglu && K_any % (2 * BK) == 0 && K_any >= 16 * BK && (shape.rows_static == 0 || K_static == K_any);
  const bool has_next = n_dyn > 0 ? experts[0].scale_in2 != nullptr : shared != nullptr && shared->scale_in2 != nullptr;
  for (int e = 0; e < n_dyn; ++e) shape.s224_fits = shape.s224_fits && (experts[e].scale_in2 != nullptr) == has_next;
  if (shape.rows_static > 0) shape.s224_fits = shape.s224_fits && (shared->scale_in2 != nullptr) == has_next;
  shape.g4_takes = g4_takes_k(n_dyn > 0 ? rows_dyn : 0, K_dyn * eb, shape.rows_static, K_static * eb);
  FormChoice choice = pick_form(shape);
  if (route != nullptr) choice = routing_form(shape);
  const bool light = choice.light, ring16 = choice.ring16, tall = choice.tall;
  const int BM = tall || choice.one_round5 ? TileCfg<5>::BM : choice.short3 ? TileCfg<3>::BM : TileCfg<4>::BM;  // tokens per block tile of the kernel that will run
  const int gather_rows_max = (alt != nullptr && alt->rows > gather_rows) ? alt->rows : gather_rows;
  if (gather_dyn != nullptr && (unsigned long long)gather_rows_max * K_dyn * eb >= (1ull << 31))
    return hdmoe_fail(HDMOE_E_SHAPE, "%s: %d gathered rows of %d bytes exceed the 2 GiB offset range", what,
                      gather_rows_max, K_dyn * eb);
  // few rows and 16-bit weights: the 8-wave kernels, whose forms (ring or not) give the same bytes
  const bool few_rows = !w8 && hdmoe_few_rows(shape.rows_dyn, shape.n_dyn, shape.rows_static);
  GemmArgs args;
  memset(&args, 0, sizeof(args));
  if (alt != nullptr && gather_dyn != nullptr) args.alt = *alt;
  args.nparts = 1;
  args.tail = tail;
  args.offsets = route != nullptr ? nullptr : offsets;
  args.n_offsets = n_dyn;
  if (route != nullptr) args.route = *route;
  int G = 0, tile_bound = 0;
  const int rows_mean = n_dyn > 0 ? rows_dyn / n_dyn : 0;
  for (int e = 0; e < n_dyn; ++e, ++G) {
    GemmGroup& gg = args.g[G];
    const hdmoe_ffn_weights& w = experts[e];
    gg.a = a_dyn;
    gg.gather = gather_dyn;
    gg.gather_shift = gather_shift;
    gg.a_rows = gather_rows;
    gg.out = out_dyn;
    gg.row_begin = -1;
    gg.dyn = e;
    gg.n_out = N_dyn;
    gg.kbytes = K_dyn * eb;
    if (swiglu) {
      gg.b0 = static_cast<const uint8_t*>(w.w1); gg.b1 = static_cast<const uint8_t*>(w.w3);
      gg.sb0 = w.scale_w1; gg.sb1 = w.scale_w3; gg.s_in = w.scale_in1; gg.s_in_b = w.scale_in3; gg.s_next = w.scale_in2;
    } else {
      gg.b0 = static_cast<const uint8_t*>(w.w2); gg.sb0 = w.scale_w2; gg.s_in = w.scale_in2;
    }
    if (!gg.b0 || (swiglu && !gg.b1)) return hdmoe_fail(HDMOE_E_NULL, "%s: expert %d has a NULL weight", what, e);
    if (fp8 && (!gg.sb0 || (swiglu && !gg.sb1)))
      return hdmoe_fail(HDMOE_E_NULL, "%s: expert %d has a NULL scale_weight", what, e);
  }
  int tb_dyn = 0, tb_static = 0;  // the two summands of tile_bound
  if (n_dyn > 0) tb_dyn = (rows_dyn / BM + n_dyn) * (N_dyn / feat_per_tile);
  tile_bound += tb_dyn;
  if (shared != nullptr && rows_static > 0) {
    GemmGroup& gg = args.g[G];
    const hdmoe_ffn_weights& w = *shared;
    gg.a = a_static;
    gg.out = out_static;
    gg.row_begin = 0;
    gg.row_end = rows_static;
    gg.n_out = N_static;
    gg.kbytes = K_static * eb;
    if (swiglu) {
      gg.b0 = static_cast<const uint8_t*>(w.w1); gg.b1 = static_cast<const uint8_t*>(w.w3);
      gg.sb0 = w.scale_w1; gg.sb1 = w.scale_w3; gg.s_in = w.scale_in1; gg.s_in_b = w.scale_in3; gg.s_next = w.scale_in2;
    } else {
      gg.b0 = static_cast<const uint8_t*>(w.w2); gg.sb0 = w.scale_w2; gg.s_in = w.scale_in2;
    }
    if (!gg.b0 || (swiglu && !gg.b1)) return hdmoe_fail(HDMOE_E_NULL, "%s: static group has a NULL weight", what);
    if (fp8 && (!gg.sb0 || (swiglu && !gg.sb1)))
      return hdmoe_fail(HDMOE_E_NULL, "%s: static group has a NULL scale_weight", what);
    tb_static = ((rows_static + BM - 1) / BM) * (N_static / feat_per_tile);
    tile_bound += tb_static;
    ++G;
  }
  args.G = G;
  // tiles of the static group are shorter or longer than the experts' when the two K differ (down projection)
  if (n_dyn > 0 && shared != nullptr && rows_static > 0 && K_static != K_dyn) args.spread = K_static < K_dyn ? 1 : -1;
  if (split) {
    // fp32 partial sums [nparts][rows_dyn + rows_static][N] (N_dyn == N_static is required), then the kernel that
    // adds them up, applies the scales and rounds to bf16
    if (n_dyn > 0 && shared != nullptr && rows_static > 0 && N_dyn != N_static)
      return hdmoe_fail(HDMOE_E_SHAPE, "%s: split K needs one output width, got %d and %d", what, N_dyn, N_static);
    const int N = n_dyn > 0 ? N_dyn : N_static;
    const int rows_all = (n_dyn > 0 ? rows_dyn : 0) + ((shared != nullptr && rows_static > 0) ? rows_static : 0);
    args.nparts = nparts;  // > 1: every group leaves fp32 sums
    args.part_stride = (long long)rows_all * N;
    for (int g = 0; g < G; ++g)
      args.g[g].pout = partial + (args.g[g].row_begin < 0 ? 0 : (size_t)(n_dyn > 0 ? rows_dyn : 0) * N);
    constexpr int BM2 = TileCfg<2>::BM;
    if (plan != nullptr && plan->n >= 1 && plan->n <= HDMOE_PLAN_MAX && plan->bm > 0) {
      args.plan = *plan;  // as the caller's other kernel sees it, tile height and limit included
    } else {
      args.plan.n = 1;
      args.plan.pd[0] = args.plan.ps[0] = nparts;
      args.plan.bm = (light || ring16) ? BM2 : BM;
      args.plan.max_tiles = HDMOE_NUM_CU;
    }
    if (reduce && args.plan.n > 1) {  // splitk_reduce_kernel takes a fixed cut: the plan's last entry
      args.plan.pd[0] = args.plan.pd[args.plan.n - 1];
      args.plan.ps[0] = args.plan.ps[args.plan.n - 1];
      args.plan.n = 1;
    }
    for (int i = 0; i < args.plan.n; ++i)
      if (args.plan.pd[i] < 1 || args.plan.pd[i] > nparts || args.plan.ps[i] < 1 || args.plan.ps[i] > nparts)
        return hdmoe_fail(HDMOE_E_SHAPE, "%s: split plan entry %d cuts in %d / %d parts, buffer holds %d", what, i,
                          args.plan.pd[i], args.plan.ps[i], nparts);
    // grid: enough blocks for the entry with the most tiles
    int tb_light = 0;  // the light form cut along K runs on 128-token tiles with a three-stage ring
    tile_bound = 0;
    for (int i = 0; i < args.plan.n; ++i) {
      const int tb = tb_dyn * args.plan.pd[i] + tb_static * args.plan.ps[i];
      if (tb > tile_bound) tile_bound = tb;
      if (light || ring16) {
        int tl = 0;
        if (n_dyn > 0) tl += (rows_dyn / BM2 + n_dyn) * (N_dyn / feat_per_tile) * args.plan.pd[i];
        if (shared != nullptr && rows_static > 0)
          tl += ((rows_static + BM2 - 1) / BM2) * (N_static / feat_per_tile) * args.plan.ps[i];
        if (tl > tb_light) tb_light = tl;
      }
    }
    const bool g4 = !fp8 && !few_rows && gemm4w_fits(args, w8);
    if (w8 && !g4) return hdmoe_fail(HDMOE_E_SHAPE, "%s: K=%d / %d in %d parts does not fit the kernel for one-byte weights", what, K_dyn, K_static, nparts);
    const int rc = light ? launch_grouped<FP8_PLAIN, 2, true>(args, tb_light, s, what)
                   : w8 ? launch_gemm4w<G4_W8, G4_PARTIAL>(args, rows_mean, s, what)
                   : ring16 ? launch_grouped<BF16_PLAIN, 2, true>(args, tb_light, s, what)
                   : fp8 && choice.fp8_g4 && gemm4w_fits(args, false) ? launch_gemm4w<G4_F8, G4_PARTIAL>(args, rows_mean, s, what)
                   : fp8 ? launch_grouped<FP8_PLAIN>(args, tile_bound, s, what)
                   : g4 ? launch_gemm4w<G4_BF16, G4_PARTIAL>(args, rows_mean, s, what)
                        : launch_grouped<BF16_PLAIN>(args, tile_bound, s, what);
    if (rc != HDMOE_OK) return rc;
    if (!reduce) return HDMOE_OK;  // the caller's next kernel adds the parts up (hdmoe_launch_combine_partials)
    SplitKReduceArgs ra;
    memset(&ra, 0, sizeof(ra));
    ra.partial = partial;
    ra.part_stride = args.part_stride;
    ra.nparts = args.plan.pd[0];
    ra.nparts_static = args.plan.ps[0];
    ra.n_out = N;
    ra.rows_dyn = n_dyn > 0 ? rows_dyn : 0;
    ra.rows_static = (shared != nullptr && rows_static > 0) ? rows_static : 0;
    ra.n_dyn = n_dyn;
    ra.scaled = fp8 ? 1 : w8 ? 2 : 0;
    ra.offsets = offsets;
    for (int g = 0; g < G; ++g) {
      const int slot = args.g[g].row_begin < 0 ? args.g[g].dyn : n_dyn;
      ra.sw[slot] = args.g[g].sb0;
      ra.sin[slot] = args.g[g].s_in;
    }
    ra.out_dyn = reinterpret_cast<uint16_t*>(out_dyn);
    ra.out_static = reinterpret_cast<uint16_t*>(out_static);
    if (end != nullptr) ra.end = *end;
    const long long work = (long long)rows_all * (N / 4);
    int blocks = (int)((work + 255) / 256);
    if (blocks > HDMOE_NUM_CU * 8) blocks = HDMOE_NUM_CU * 8;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(splitk_reduce_kernel, dim3(blocks), dim3(256), 0, s, ra);
    return hdmoe_check_launch(what);
  }
  if (!fp8) {
    // The 4-wave kernel (gemm4w.h) takes whatever fits it: a K step of a 256 x 256 tile takes 1.36 to 1.45 us there and
    // 1.7 to 1.8 us in the 8-wave kernel (16384 x 13824 x 2560: 0.81 against 0.96 ms). Left to the 8-wave kernels: the
    // three-stage ring for gate/up with every segment inside a 128-token tile (16-bit weights, unless cut: swiglu_on_g4), the case one_round5, K that is
    // not a multiple of 128, and, where tiles cannot be cut (no room for the parts), one Linear on up to 128 rows (2560 x 2560: 37
    // against 43 us: the 8-wave kernel leaves out the token blocks without rows).
    const bool g4 = gemm4w_fits(args, w8);
    if (w8) {
      if (!g4) return hdmoe_fail(HDMOE_E_SHAPE, "%s: K=%d / %d does not fit the kernel for one-byte weights", what, K_dyn, K_static);
      return swiglu ? launch_gemm4w<G4_W8, G4_SWIGLU>(args, rows_mean, s, what)
                    : launch_gemm4w<G4_W8, G4_PLAIN>(args, rows_mean, s, what);
    }
    if (choice.one_round5) return launch_grouped<BF16_SWIGLU, 5>(args, tile_bound, s, what);
    if (swiglu && g4 && swiglu_on_g4(shape, tail != nullptr)) return launch_gemm4w<G4_BF16, G4_SWIGLU>(args, rows_mean, s, what);
    if (!swiglu && g4 && (tail != nullptr || rows_mean > 128 || rows_static > 128))
      return launch_gemm4w<G4_BF16, G4_PLAIN>(args, rows_mean, s, what);
  }
  if (choice.fp8_g4 && gemm4w_fits(args, false)) return launch_gemm4w<G4_F8, G4_PLAIN>(args, rows_mean, s, what);
  if (fp8 && swiglu && route == nullptr) {
    long long op_bytes = (long long)(gather_dyn != nullptr ? gather_rows_max : rows_dyn) * K_dyn;
    if ((long long)rows_static * K_static > op_bytes) op_bytes = (long long)rows_static * K_static;
    shape.w4_fits = swiglu4w_fits(args, op_bytes);
    shape.s224_fits = shape.s224_fits && swiglu224_fits(args);
    choice = pick_form(shape);
    if (choice.form == FORM_S224) return args.g[0].s_next == nullptr ? launch_swiglu224<true>(args, s, what) : launch_swiglu224<false>(args, s, what);
  }
  switch (choice.form) {
    case FORM_RING3: {
      constexpr int BM2 = TileCfg<2>::BM;
      int tb = 0;
      if (n_dyn > 0) tb += (rows_dyn / BM2 + n_dyn) * (N_dyn / feat_per_tile);
      if (shared != nullptr && rows_static > 0) tb += ((rows_static + BM2 - 1) / BM2) * (N_static / feat_per_tile);
      return fp8 ? launch_grouped<FP8_SWIGLU, 2, true>(args, tb, s, what)
                 : launch_grouped<BF16_SWIGLU, 2, true>(args, tb, s, what);
    }
    case FORM_LIGHT4:
      return swiglu ? launch_grouped<FP8_SWIGLU, 4, true>(args, tile_bound, s, what)
                    : launch_grouped<FP8_PLAIN, 4, true>(args, tile_bound, s, what);
    case FORM_W4: {
      int tb = 0;
      if (n_dyn > 0) tb += (rows_dyn / W4_BM + n_dyn) * (N_dyn / W4_FEAT);
      if (shared != nullptr && rows_static > 0) tb += ((rows_static + W4_BM - 1) / W4_BM) * (N_static / W4_FEAT);
      return launch_swiglu4w(args, tb, s, what);
    }
    case FORM_SHORT3:
      return launch_grouped<FP8_SWIGLU, 3>(args, tile_bound, s, what);
    case FORM_TALL5:
      if (fp8) return swiglu ? launch_grouped<FP8_SWIGLU, 5>(args, tile_bound, s, what)
                             : launch_grouped<FP8_PLAIN, 5>(args, tile_bound, s, what);
      return launch_grouped<BF16_SWIGLU, 5>(args, tile_bound, s, what);
    default:
      break;
  }
  if (fp8) return swiglu ? launch_grouped<FP8_SWIGLU>(args, tile_bound, s, what)
                         : launch_grouped<FP8_PLAIN>(args, tile_bound, s, what);
  return swiglu ? launch_grouped<BF16_SWIGLU>(args, tile_bound, s, what)
                : launch_grouped<BF16_PLAIN>(args, tile_bound, s, what);
}

// An fp8 Linear with a bias that the 4-wave kernel does not take (K no multiple of 256): the 192-token tile of the 8-wave kernel, where its
// rounds of tiles cost a tenth less than those of 256 tokens (as expected_tile_cost counts them: rounds x (TT + 1)).
static bool fp8_linear_192(int rows, int N) {
  auto cost = [&](int tt) { return (long)(((rows + 64 * tt - 1) / (64 * tt) * (N / BN) + HDMOE_NUM_CU - 1) / HDMOE_NUM_CU) * (tt + 1); };
  return 10 * cost(3) <= 9 * cost(4);
}

// Name of the kernel the gate/up contraction of a layer runs on (T tokens, E routed experts top-2 plus a shared expert
// if Hs > 0), by the launcher's own rule and the current form switches: for reports that name the dominant kernel.
extern "C" const char* hdmoe_gate_up_kernel_name(int weight_dtype, int T, int E, int D, int H, int Hs,
                                                 int has_scale_in2) {
  if (check_dtype(weight_dtype, "hdmoe_gate_up_kernel_name", true) != HDMOE_OK || T <= 0 || E < 0 || D <= 0 || H <= 0)
    return "";
  GemmShape sh;
  sh.swiglu = true; sh.fp8 = weight_dtype == HDMOE_W_E4M3FN; sh.split = false; sh.w8 = weight_dtype == HDMOE_W_E4M3FN_UPCAST;
  sh.rows_dyn = E > 0 ? T * HDMOE_TOPK : 0; sh.n_dyn = E; sh.rows_static = Hs > 0 ? T : 0;
  sh.N_dyn = H; sh.N_static = Hs;
  const int kb = D * elem_bytes(weight_dtype);
  sh.kbytes = kb;
  sh.g4_takes = kb % (2 * BK) == 0 && kb >= 4 * BK;
  sh.s224_fits = sh.fp8 && kb % (2 * BK) == 0 && kb >= 16 * BK && H % S224_FEAT == 0 && (Hs <= 0 || Hs % S224_FEAT == 0);
  sh.w4_fits = sh.fp8 && has_scale_in2 != 0 && kb % (2 * BK) == 0 && kb >= 16 * BK && H % W4_FEAT == 0 &&
               (Hs <= 0 || Hs % W4_FEAT == 0) && (long long)T * kb < (1ll << 31);
  switch (pick_form(sh).form) {
    case FORM_RING3:
      if (swiglu_on_g4(sh, true)) return "gemm4w_kernel<SWIGLU>";
      return sh.fp8 ? "grouped_gemm_kernel<FP8_SWIGLU, 2, LIGHT>" : "grouped_gemm_kernel<BF16_SWIGLU, 2, LIGHT>";
    case FORM_LIGHT4: return "grouped_gemm_kernel<FP8_SWIGLU, 4, LIGHT>";
    case FORM_W4: return "swiglu4w_kernel";
    case FORM_S224: return "swiglu224_kernel";
    case FORM_SHORT3: return "grouped_gemm_kernel<FP8_SWIGLU, 3>";
    case FORM_TALL5: return sh.fp8 ? "grouped_gemm_kernel<FP8_SWIGLU, 5>" : "grouped_gemm_kernel<BF16_SWIGLU, 5>";
    default:
      if (pick_form(sh).one_round5) return "grouped_gemm_kernel<BF16_SWIGLU, 5>";
      if (swiglu_on_g4(sh, true)) return "gemm4w_kernel<SWIGLU>";
      return sh.fp8 ? "grouped_gemm_kernel<FP8_SWIGLU, 4>" : "grouped_gemm_kernel<BF16_SWIGLU, 4>";
  }
}

// The same for an fp8 contraction without activation: a down projection (E experts' segments of rows_dyn rows together, rows_static
// of one more) in `parts` parts along K, or a Linear (E = 0) with a bias.
extern "C" const char* hdmoe_plain_kernel_name(int rows_dyn, int E, int K_dyn, int rows_static, int K_static, int N, int parts,
                                               int has_bias) {
  if (rows_dyn < 0 || E < 0 || E > HDMOE_MAX_EXPERTS || rows_static < 0 || N <= 0 || N % BN != 0 || parts < 1) return "";
  const int n_dyn = rows_dyn > 0 ? E : 0;
  auto bad = [](int rows, int K) { return rows > 0 && (K <= 0 || K % BK != 0); };
  if (bad(n_dyn, K_dyn) || bad(rows_static, K_static) || (n_dyn == 0 && rows_static == 0)) return "";
  const bool takes = g4_takes_k(n_dyn > 0 ? rows_dyn : 0, K_dyn, rows_static, K_static);
  if (has_bias != 0) {
    if (takes) return "gemm4w_kernel<F8, BIAS>";
    return fp8_linear_192(rows_static, N) ? "grouped_gemm_kernel<FP8_PLAIN_BIAS, 3>" : "grouped_gemm_kernel<FP8_PLAIN_BIAS, 4>";
  }
  GemmShape sh;
  sh.swiglu = false; sh.fp8 = true; sh.split = parts > 1; sh.w8 = false; sh.w4_fits = sh.s224_fits = false; sh.kbytes = 0;
  sh.rows_dyn = n_dyn > 0 ? rows_dyn : 0; sh.n_dyn = n_dyn; sh.rows_static = rows_static;
  sh.N_dyn = sh.N_static = N;
  sh.g4_takes = takes;
  const FormChoice c = pick_form(sh);
  const int shortest = n_dyn > 0 && (rows_static == 0 || K_dyn < K_static) ? K_dyn : K_static;
  if (c.fp8_g4 && shortest / (2 * BK) / parts >= 2) return parts > 1 ? "gemm4w_kernel<F8, PARTIAL>" : "gemm4w_kernel<F8, PLAIN>";
  if (c.light) return parts > 1 ? "grouped_gemm_kernel<FP8_PLAIN, 2, LIGHT>" : "grouped_gemm_kernel<FP8_PLAIN, 4, LIGHT>";
  return parts == 1 && c.tall ? "grouped_gemm_kernel<FP8_PLAIN, 5>" : "grouped_gemm_kernel<FP8_PLAIN, 4>";
}

// How the down projection of a layer is cut along K: a pure function of the sizes, so that the workspace layout and
// the launch agree. With few tiles (small token counts) most CUs would idle through a long K loop. Returns the most
// parts any entry of the plan cuts a tile into (the partial-sum buffer is sized for it; 1 = no cut) and fills *plan.
//
// Cost model in units of one K step of one tile: a tile costs its steps + 3 (prologue and epilogue); one round of
// blocks lasts as long as its longest tile; more tiles than CUs last about the total divided by the CUs plus half a
// tile of slack; a cut adds the fp32 partial sums written and read again (8 bytes per output and part; they stay in
// the memory-side cache at these sizes, about 10 TB/s; one step is about 1.4 us).
// less_room: the cut of few rows that takes less room, for a workspace that holds no more (hdmoe_moe_ffn).
int hdmoe_down_parts(int rows_dyn, int n_dyn, int rows_static, int N, int K_dyn, int K_static, int weight_dtype,
                     HdmoeSplitPlan* plan, bool less_room) {
  HdmoeSplitPlan local;
  HdmoeSplitPlan& pl = plan != nullptr ? *plan : local;
  memset(&pl, 0, sizeof(pl));
  pl.bm = TileCfg<4>::BM;
  pl.max_tiles = HDMOE_NUM_CU;
  auto fixed = [&](int parts) {
    pl.n = 1;
    pl.pd[0] = pl.ps[0] = pl.fixed_pd = pl.fixed_ps = parts;
    return parts;
  };
  const int eb = elem_bytes(weight_dtype);
  const int nt = N / BN;
  const bool dyn = n_dyn > 0 && rows_dyn > 0;
  const int ktd = dyn ? K_dyn * eb / BK : 0, kts = rows_static > 0 ? K_static * eb / BK : 0;
  if ((!dyn && rows_static <= 0) || nt <= 0 || (ktd <= 0 && kts <= 0)) return fixed(1);

  // Few rows per segment (the rule of the light form in hdmoe_launch_ffn_gemm): the launch runs on 128-token
  // tiles with K steps requested two ahead, and is bound by how fast the weights arrive, not by its K loops. (e4m3fn weights in bf16 run on 256-row
  // tiles, of which the rows can make fewer: for them the count below is the most, and from 129 tokens on five and three parts would fit.) A layer: the most parts whose
  // tiles fit one round of blocks however the rows fall to the experts (the sizes alone say, so that a row's sums do not depend on the
  // others' routing), the shared expert's tiles in as many as make them about as long, rounded up first. Three parts of every tile up to 128
  // tokens, two up to 256 -> this (weights from memory, two inputs each; rounded down only where the experts' tiles gain a part by it: 8
  // experts, 256 tokens in fp8 (2, 2) parts 166.9, (2, 1) 170.2), us: fp8, 16 tokens 69.0 64.2 -> 66.7 61.3, 64 73.0 70.8 -> 70.2 67.1, 128
  // 77.8 77.3 -> 75.0 74.4, 256 99.2 95.7 -> 94.0 91.4; bf16, 64 115.9 110.1 -> 110.3 102.4, 256 157.1 148.3 -> 146.2 139.9; e4m3fn weights in bf16,
  // 64 109.4 108.6 -> 100.0 98.7, 256 134.6 135.3 -> 121.3 120.4. (Five parts of every tile, the shared expert's too: 64 tokens in fp8 72.3; the
  // most parts that fit the real segments, picked on the device: 256 tokens 95.1, 200 89.0 where this has 90.8.)
  // A dense feed-forward, what fits no round, and less_room: about 150 blocks keep enough loads in flight; segments counted 1.5 times the mean.
  if (hdmoe_few_rows(rows_dyn, n_dyn, rows_static)) {
    const int bm2 = TileCfg<2>::BM;
    pl.bm = bm2;
    long t2 = 0;
    if (dyn) {
      const long seg = ((long)rows_dyn * 3 / 2 + n_dyn - 1) / n_dyn;
      t2 += (long)n_dyn * ((seg + bm2 - 1) / bm2) * nt;
    }
    if (rows_static > 0) t2 += (long)((rows_static + bm2 - 1) / bm2) * nt;
    int kt2 = ktd > kts ? ktd : kts;
    if (weight_dtype == HDMOE_W_E4M3FN_UPCAST && ktd > 0 && kts > 0) kt2 = ktd < kts ? ktd : kts;  // no part under three pairs of steps
    long parts = (150 + t2 - 1) / t2;
    if (parts > HDMOE_NUM_CU / t2) parts = HDMOE_NUM_CU / t2;
    if (parts > 6) parts = 6;
    while (parts > 1 && kt2 / parts < 6) --parts;
    if (ktd > 0 && kts > 0 && !less_room) {   // (a width under one K step: no cut, and the call is refused)
      const long mt_s = (rows_static + bm2 - 1) / bm2;
      long mt_d = rows_dyn > n_dyn ? (rows_dyn - n_dyn) / bm2 + n_dyn : rows_dyn;   // the most that the rows make
      if (mt_d > n_dyn * mt_s) mt_d = n_dyn * mt_s;                                 // (no expert has a token twice)
      for (int pd = 6; pd > 1; --pd)
        for (int ps = (int)fmin((pd * kts + ktd - 1) / ktd, pd); ps >= 1 && 2 * pd * kts <= (2 * ps + 1) * ktd; --ps) {
          if (pd <= parts && ps * ktd < pd * kts) continue;
          if (ktd / pd < 6 || kts / ps < 6 || (mt_d * pd + mt_s * ps) * nt > HDMOE_NUM_CU) continue;
          pl.n = 1;
          pl.pd[0] = pl.fixed_pd = pd;
          pl.ps[0] = pl.fixed_ps = ps;
          return pd;
        }
    }
    return fixed(parts < 1 ? 1 : (int)parts);
  }

  // A dense feed-forward in fp8 on the 4-wave kernel, whose tiles can be lower (gemm4w.h): parts on the lowest tiles that fill a round of CUs.
  // In hundredths of a pair of K steps (24.6 ns) as in g4_cap_cost; a part's sums written and read again at about 5 TB/s, 100 for the kernel that
  // adds them up. Whole tiles have 18 more per pair: each of their steps waits for the memory that cold weights come from (0.6 us a pair, nothing
  // where the caches have them; parts share that wait). Whole branch, D = 2560, H = 6912, us, on 256-token tiles (6 to 3 parts) -> this, weights in the
  // caches: 300 rows 61.0 -> 53.7 (6 parts), 512 63.4 -> 56.7 (4), 768 67.9 -> 61.2 (3), 1024 85.9 -> 79.5 (3), 1536 104.2 -> 97.1 (2). Beyond, cold and in
  // the caches, on 256-token tiles, whole on lower ones, this: 1600 113.8 108.2, 120.2 103.5, 113.5 102.2; 1800 117.9 113.6, 121.1 106.2, 114.6 108.6;
  // 2048 134.8 130.0, 138.7 120.7, 131.3 125.1 (192-token tiles); whole from 2168 rows on: 2300 142.4 135.3, 142.3 126.5.
  // Width 4096, 1700 rows: 207 202, 222 194, 207 202 (two parts on 224-token tiles); 1000 rows 147 141 on 256-token tiles in four parts, 153 137 here (two of 128).
  if (weight_dtype == HDMOE_W_E4M3FN && !dyn && kts % 2 == 0 && kts >= 4) {
    constexpr int PAIR[5] = {58, 70, 80, 90, 100}, COLD = 18;
    const int pairs = kts / 2;
    auto rounds = [&](int bm, int parts) { return ((long)(rows_static + bm - 1) / bm * nt * parts + HDMOE_NUM_CU - 1) / HDMOE_NUM_CU; };
    double best_cost = 1e30;
    int best = 1, height = 8;
    for (int h = 4; h <= 8; ++h) best_cost = fmin(best_cost, (double)rounds(32 * h, 1) * (pairs * PAIR[h - 4] + G4_TILE_COST) + COLD * pairs);
    best_cost *= 0.95;   // a cut has to pay
    for (int parts = 2; parts <= 6 && pairs / parts >= 3; ++parts)
      for (int h = 4; h <= 8; ++h) {
        const double cost = (double)rounds(32 * h, parts) * ((pairs + parts - 1) / parts * PAIR[h - 4] + G4_TILE_COST) + (double)parts * rows_static * N * 8.0 / 123e3 + 100.0;
        if (cost < best_cost) { best = parts; height = h; best_cost = cost; }
      }
    pl.bm = 32 * height;
    return fixed(best);
  }
  // A layer in fp8 on that kernel: the most parts whose tiles fit one round of blocks, on 128-token tiles with even segments (the device takes
  // higher ones where its segments do not fit, g4_cut_height), else on 256-token tiles with segments a standard deviation above the mean
  // (g4_likely_tiles; width 4096, 500 tokens: (2, 1) parts 271 us, whole tiles 290); beyond that none (g4_two_lengths deals the tiles out).
  // The shared expert's tiles in as many parts as make them about as long. Whole layer, us, candidates on 256-token tiles of which the device
  // took the first that fitted (one at most sizes, seven around 500 tokens) -> this (three inputs each): 350 tokens 118 -> 113 ((2, 1) parts of
  // 128), 400 123 -> 118, 450 150 -> 143, 500 147 -> 144, 640 145 -> 141 ((2, 1) of 256; of 128 in two rounds 164, whole tiles 157), 768 158 ->
  // 156, 900 202 -> 199, 1024 209 -> 204 (whole), 1600 the same, 2000 266 -> 248. Not under 150 rows an expert: 300 tokens 106, 106, 260 103, 105.
  if (weight_dtype == HDMOE_W_E4M3FN && dyn && rows_static > 0 && rows_dyn >= 150 * n_dyn && ktd % 2 == 0 && kts % 2 == 0 && ktd >= 4 && kts >= 4) {
    for (int bm : {128, 256}) {
      const int mt_d = bm == 128 ? n_dyn * (((rows_dyn + n_dyn - 1) / n_dyn + bm - 1) / bm) : g4_likely_tiles(rows_dyn, n_dyn, bm);
      const int mt_s = (rows_static + bm - 1) / bm;
      for (int pd = 6; pd >= 2; --pd) {
        const int ps = (int)fmin(fmax((double)pd * kts / ktd + 0.5, 1.0), (double)pd);
        if (ktd / 2 / pd < 3 || kts / 2 / ps < 3 || (mt_d * pd + mt_s * ps) * nt > HDMOE_NUM_CU) continue;
        pl.n = 1;
        pl.pd[0] = pl.fixed_pd = pd;
        pl.ps[0] = pl.fixed_ps = ps;
        pl.bm = bm;
        const int high = g4_cut_height(bm, rows_dyn, n_dyn, rows_static, pd, ps, nt);
        pl.bm_else = high > bm ? high : 0;
        return pd;
      }
    }
    return fixed(1);
  }
  const int bm = TileCfg<4>::BM;
  const double red_unit = (double)N * 8.0 / 10e12 / 1.4e-6;  // K steps per row and part of partial sums
  if (!dyn || rows_static <= 0) {
    // one kind of group: every tile in the same number of parts, whole rounds of tiles
    double tiles = 0;
    if (dyn) tiles += 1.12 * n_dyn * ((rows_dyn / n_dyn + bm - 1) / bm) * nt;
    if (rows_static > 0) tiles += (double)((rows_static + bm - 1) / bm) * nt;
    const int kt = ktd > kts ? ktd : kts;
    const double rows_all = (double)(dyn ? rows_dyn : 0) + (rows_static > 0 ? rows_static : 0);
    int best = 1;
    double best_cost = 0;
    for (int parts = 1; parts <= 6 && kt / parts >= 6; ++parts) {
      const double rounds = (double)(long)((tiles * parts + HDMOE_NUM_CU - 1) / HDMOE_NUM_CU);
      const double cost = rounds * ((double)kt / parts + 3.0) + (parts > 1 ? parts * rows_all * red_unit : 0.0);
      if (parts == 1 || cost < best_cost * 0.95) {  // a cut has to pay
        best = parts;
        best_cost = cost;
      }
    }
    return fixed(best);
  }

  // Experts and a static group (the layer). Their tiles have different K (HiDream: 6912 and 3584), and cutting the
  // static group's tiles in ps = pd * kts / ktd parts makes all tiles about equally long.
  // Candidates, most parts first, every tile alike before the equalising cut: the cuts whose tiles fit one round of
  // blocks with every expert at the mean segment size. The device takes the first that really fits (measured on 4
  // experts + shared expert, fp8 and bf16: 320-384 tokens (4,4) or (4,2), 512 tokens (3,3) or (3,2), 640-896 tokens
  // (2,2) or (2,1), 1024 tokens (2,1), each 2-10 % ahead of any cut that needs a second round).
  const int mt_d_mean = n_dyn * ((rows_dyn / n_dyn + bm - 1) / bm), mt_s = (rows_static + bm - 1) / bm;
  pl.n = 0;
  auto candidate = [&](int pd, int ps) {
    if (pl.n >= HDMOE_PLAN_MAX - 1 || (mt_d_mean * pd + mt_s * ps) * nt > HDMOE_NUM_CU) return;
    for (int i = 0; i < pl.n; ++i)
      if (pl.pd[i] == pd && pl.ps[i] == ps) return;
    pl.pd[pl.n] = pd;
    pl.ps[pl.n] = ps;
    ++pl.n;
  };
  for (int pd = 6; pd >= 2; --pd) {
    if (ktd / pd < 6) continue;
    int ps = (int)((double)pd * kts / ktd + 0.5);
    if (ps < 1) ps = 1;
    if (ps > pd) ps = pd;
    while (ps > 1 && kts / ps < 6) --ps;
    if (kts / pd >= 6) candidate(pd, pd);
    candidate(pd, ps);
  }
  // A first candidate that still fits with every expert one standard deviation above the mean segment (the counts
  // are about binomial) is taken as it is: the kernels then have nothing to decide (the decision costs them about a
  // microsecond each).
  const double mu = (double)rows_dyn / n_dyn;
  if (pl.n > 0) {
    const int mt_d_hi = n_dyn * (int)(((long)(mu + sqrt(mu)) + bm - 1) / bm);
    if ((mt_d_hi * pl.pd[0] + mt_s * pl.ps[0]) * nt <= HDMOE_NUM_CU) {
      pl.n = 1;
      pl.fixed_pd = pl.pd[0];
      pl.fixed_ps = pl.ps[0];
      return pl.pd[0];
    }
  }
  // 16-bit activations on the 4-wave kernel: where no candidate fits, whole tiles, dealt out by g4_two_lengths if that is so for even segments.
  // The cost model's cut in more than a round -> this, layers, us: bf16, 1024 tokens with an expert above 512 rows 339 -> 306, 1800 469 -> 434, 2040 489 ->
  // 459; e4m3fn weights, 1024 318 -> 265, 1800 441 -> 415, 2040 456 -> 433.
  const bool whole16 = weight_dtype != HDMOE_W_E4M3FN && ktd % 2 == 0 && kts % 2 == 0 && ktd >= 6 && kts >= 6;
  if (whole16 && pl.n == 0) return fixed(1);
  // Last entry, for when no candidate fits: the cheapest cut by the cost model. With candidates listed, their not
  // fitting means ragged segments, and the experts' m-tiles are counted one standard deviation above the mean
  // segment (counts are about binomial); with none, 12 % above the mean.
  const double seg = pl.n > 0 ? mu + sqrt(mu) : mu;
  const double td = (pl.n > 0 ? 1.0 : 1.12) * n_dyn * (double)(((long)seg + bm - 1) / bm) * nt, ts = (double)mt_s * nt;
  int best_d = 1, best_s = 1;
  double best_cost = 0;
  for (int pd = 1; pd <= 6 && (pd == 1 || ktd / pd >= 6); ++pd)
    for (int ps = 1; ps <= pd && (ps == 1 || kts / ps >= 6); ++ps) {
      const double ld = (double)ktd / pd + 3.0, ls = (double)kts / ps + 3.0;
      const double tiles = td * pd + ts * ps, longest = ld > ls ? ld : ls;
      double cost = tiles <= HDMOE_NUM_CU ? longest : (td * pd * ld + ts * ps * ls) / HDMOE_NUM_CU + 0.5 * longest;
      if (pd > 1) cost += ((double)rows_dyn * pd + (double)rows_static * ps) * red_unit;
      if ((pd == 1 && ps == 1) || cost < best_cost * 0.95) {
        best_d = pd;
        best_s = pd > 1 ? ps : 1;
        best_cost = cost;
      }
    }
  pl.fixed_pd = best_d;
  pl.fixed_ps = best_s;
  pl.pd[pl.n] = whole16 ? 1 : best_d;
  pl.ps[pl.n] = whole16 ? 1 : best_s;
  ++pl.n;
  int most = best_d;
  for (int i = 0; i < pl.n; ++i) most = pl.pd[i] > most ? pl.pd[i] : most;
  if (most == 1) return fixed(1);  // nothing is cut
  return most;
}

// Linear with bias and optional GELU over expert row segments plus an optional static group:
// the two stages of a GELU feed-forward (/root/reference/comfy/ldm/hunyuan3dv2_1/hunyuandit.py:28-50, 114-188).
// tail, scratch: room of gemm4w_kernel (G4_TAIL_BYTES; G4_SCRATCH per block, GELU only) or NULL.
template <typename W>
int hdmoe_launch_linear_groups(const uint8_t* a_dyn, const int32_t* offsets, int rows_dyn, int n_dyn, const W* experts,
                               uint8_t* out_dyn, const uint8_t* a_static, int rows_static, const W* shared,
                               uint8_t* out_static, int K, int N, int act, hipStream_t s, const char* what, bool f16,
                               const int32_t* gather, int gather_rows, int gather_shift, bool w8 = false,
                               float* tail = nullptr, uint8_t* scratch = nullptr) {
  if (gather != nullptr && (unsigned long long)gather_rows * K * 2 >= (1ull << 31))
    return hdmoe_fail(HDMOE_E_SHAPE, "%s: %d gathered rows of %d bytes exceed the 2 GiB offset range", what, gather_rows,
                      K * 2);
  GemmArgs args;
  memset(&args, 0, sizeof(args));
  args.nparts = 1;
  args.tail = tail;
  args.scratch = scratch;
  args.offsets = offsets;
  args.n_offsets = n_dyn;
  int G = 0;
  auto fill = [&](GemmGroup& gg, const W& w) {
    gg.b0 = static_cast<const uint8_t*>(w.weight);
    gg.bias = static_cast<const uint16_t*>(w.bias);
    if constexpr (std::is_same_v<W, hdmoe_linear_group>) gg.sb0 = w.scale;
    gg.act = act;
    gg.n_out = N;
    gg.kbytes = K * 2;
  };
  for (int e = 0; e < n_dyn; ++e, ++G) {
    GemmGroup& gg = args.g[G];
    fill(gg, experts[e]);
    gg.a = a_dyn;
    gg.gather = gather;
    gg.gather_shift = gather_shift;
    gg.a_rows = gather_rows;
    gg.out = out_dyn;
    gg.row_begin = -1;
    gg.dyn = e;
    if (!gg.b0) return hdmoe_fail(HDMOE_E_NULL, "%s: expert %d has a NULL weight", what, e);
  }
  if (shared != nullptr && rows_static > 0) {
    GemmGroup& gg = args.g[G];
    fill(gg, *shared);
    gg.a = a_static;
    gg.out = out_static;
    gg.row_begin = 0;
    gg.row_end = rows_static;
    if (!gg.b0) return hdmoe_fail(HDMOE_E_NULL, "%s: static group has a NULL weight", what);
    ++G;
  }
  args.G = G;
  // The 4-wave kernel wherever it fits; it needs room of its own for the activation, and room for the parts of tiles where
  // a few tiles have to be cut. Without that room and with up to 128 rows a group the 8-wave kernel is the faster one (see
  // hdmoe_launch_ffn_gemm; 8 experts on 600 rows and one more on 300, 2048 x 8192: 104 against 108 us).
  const int rows_mean = n_dyn > 0 ? rows_dyn / n_dyn : 0;
  const bool g4 = gemm4w_fits(args, w8);
  if (w8) {
    if (!g4 || f16 || act == HDMOE_ACT_GELU)
      return hdmoe_fail(HDMOE_E_SHAPE, "%s: K=%d act=%d does not fit the kernel for one-byte weights", what, K, act);
    return launch_gemm4w<G4_W8, G4_BIAS>(args, rows_mean, s, what);
  }
  if (g4 && act == HDMOE_ACT_GELU && scratch != nullptr)
    return f16 ? launch_gemm4w<G4_F16, G4_GELU>(args, rows_mean, s, what)
               : launch_gemm4w<G4_BF16, G4_GELU>(args, rows_mean, s, what);
  const int rows_all = (n_dyn > 0 ? rows_dyn : 0) + (shared != nullptr ? rows_static : 0);
  const bool room = tail != nullptr && g4_tail_room(n_dyn, rows_mean, N, K * 2, shared != nullptr ? rows_static : 0, N, K * 2, BN, false) > 0;
  if (g4 && act == HDMOE_ACT_NONE && (room || rows_all > 128 * G))
    return f16 ? launch_gemm4w<G4_F16, G4_BIAS>(args, rows_mean, s, what)
               : launch_gemm4w<G4_BF16, G4_BIAS>(args, rows_mean, s, what);
  // The 8-wave kernel, by the rule of the feed-forward contractions: the 320-token tile when it saves a round of tiles. A
  // segment is taken one standard deviation of an even routing above the mean (at a mean that is a multiple of the tile height half the
  // segments need one tile more). GELU, 8 experts on 5000 rows and one more on 2500, 2048 x 8192: 330 us on 256-token tiles, 272 on 320.
  auto tiles = [&](int tt) {
    const int bm = 64 * tt, seg = rows_mean + (int)sqrtf((float)rows_mean);
    long n = 0;
    if (n_dyn > 0) n += (long)n_dyn * ((seg + bm - 1) / bm) * (N / BN);
    if (shared != nullptr && rows_static > 0) n += (long)((rows_static + bm - 1) / bm) * (N / BN);
    return n;
  };
  auto cost = [&](int tt) { return (tiles(tt) + HDMOE_NUM_CU - 1) / HDMOE_NUM_CU * (tt + 1); };
  const bool tall = cost(5) < cost(4);
  const int BM = tall ? TileCfg<5>::BM : TileCfg<4>::BM;
  int tile_bound = 0;
  if (n_dyn > 0) tile_bound += (rows_dyn / BM + n_dyn) * (N / BN);
  if (shared != nullptr && rows_static > 0) tile_bound += ((rows_static + BM - 1) / BM) * (N / BN);
  if (tall) return f16 ? launch_grouped<F16_PLAIN_BIAS, 5>(args, tile_bound, s, what)
                       : launch_grouped<BF16_PLAIN_BIAS, 5>(args, tile_bound, s, what);
  return f16 ? launch_grouped<F16_PLAIN_BIAS>(args, tile_bound, s, what)
             : launch_grouped<BF16_PLAIN_BIAS>(args, tile_bound, s, what);
}

// One Linear with an optional bias over all rows of `a` (either weight type): a single static group.
int hdmoe_launch_linear_bias(int weight_dtype, const uint8_t* a, int rows, int K, int N, const uint8_t* w,
                             const float* scale_w, const float* scale_in, const uint16_t* bias, uint8_t* out,
                             hipStream_t s, const char* what) {
  const bool fp8 = weight_dtype == HDMOE_W_E4M3FN;
  if (!fp8) {
    const hdmoe_linear_weights lw = {w, bias};
    return hdmoe_launch_linear_groups(static_cast<const uint8_t*>(nullptr), nullptr, 0, 0, static_cast<const hdmoe_linear_weights*>(nullptr),
                                      nullptr, a, rows, &lw, out, K, N, HDMOE_ACT_NONE, s, what, weight_dtype == HDMOE_W_F16,
                                      nullptr, 0, 0);
  }
  GemmArgs args;
  memset(&args, 0, sizeof(args));
  args.nparts = 1;
  GemmGroup& gg = args.g[0];
  gg.a = a;
  gg.out = out;
  gg.row_begin = 0;
  gg.row_end = rows;
  gg.n_out = N;
  gg.kbytes = K * elem_bytes(weight_dtype);
  gg.b0 = w;
  gg.sb0 = scale_w;
  gg.s_in = scale_in;
  gg.bias = bias;
  gg.act = HDMOE_ACT_NONE;
  args.G = 1;
  auto tiles = [&](int tt) { return (rows + 64 * tt - 1) / (64 * tt) * (N / BN); };
  if (gemm4w_fits(args, false)) return launch_gemm4w<G4_F8, G4_BIAS>(args, rows, s, what);
  if (fp8_linear_192(rows, N)) return launch_grouped<FP8_PLAIN_BIAS, 3>(args, tiles(3), s, what);
  return launch_grouped<FP8_PLAIN_BIAS>(args, tiles(4), s, what);
}

// Size rules shared by the entry points: K bytes per row must be a multiple of the
// 128-byte K step; total bytes of each operand must fit the 32-bit buffer range.
int hdmoe_check_gemm_shape(const char* what, int weight_dtype, long rows, int K, int N, int feat_per_tile) {
  if (int rc = check_dtype(weight_dtype, what, true)) return rc;
  const int eb = elem_bytes(weight_dtype);
  if (rows < 0 || K <= 0 || N <= 0 || (K * eb) % BK != 0 || N % feat_per_tile != 0)
    return hdmoe_fail(HDMOE_E_SHAPE, "%s: rows=%ld K=%d N=%d (K*%d must be a multiple of %d, N of %d)", what, rows, K,
                      N, eb, BK, feat_per_tile);
  if ((unsigned long long)rows * K * eb >= (1ull << 32) || (unsigned long long)rows * N * 2 >= (1ull << 40))
    return hdmoe_fail(HDMOE_E_SHAPE, "%s: rows=%ld K=%d exceeds the 4 GiB buffer range", what, rows, K);
  return HDMOE_OK;
}

extern "C" int hdmoe_grouped_swiglu(int weight_dtype, const void* a, const int32_t* offsets, int rows_total, int E,
                                    int D, int H, const hdmoe_ffn_weights* experts, void* h, hdmoe_stream_t stream) {
  HDMOE_REQUIRE_PTR(a);
  HDMOE_REQUIRE_PTR(offsets);
  HDMOE_REQUIRE_PTR(experts);
  HDMOE_REQUIRE_PTR(h);
  if (E < 1 || E > HDMOE_MAX_EXPERTS) return hdmoe_fail(HDMOE_E_SHAPE, "hdmoe_grouped_swiglu: E=%d", E);
  if (int rc = check_dtype(weight_dtype, "hdmoe_grouped_swiglu")) return rc;
  if (int rc = hdmoe_check_gemm_shape("hdmoe_grouped_swiglu", weight_dtype, rows_total, D, H, BN / 2)) return rc;
  if (weight_dtype == HDMOE_W_E4M3FN)
    for (int e = 0; e < E; ++e)
      if (int rc = hdmoe_check_scale_in13("hdmoe_grouped_swiglu", experts[e], e)) return rc;
  if (rows_total == 0) return HDMOE_OK;
  return hdmoe_launch_ffn_gemm(true, weight_dtype, static_cast<const uint8_t*>(a), offsets, rows_total, E, experts,
                               static_cast<uint8_t*>(h), nullptr, 0, nullptr, nullptr, D, H, 0, 0,
                               static_cast<hipStream_t>(stream), "hdmoe_grouped_swiglu");
}

extern "C" int hdmoe_grouped_down(int weight_dtype, const void* h, const int32_t* offsets, int rows_total, int E, int H,
                                  int D, const hdmoe_ffn_weights* experts, void* y_bf16, hdmoe_stream_t stream) {
  HDMOE_REQUIRE_PTR(h);
  HDMOE_REQUIRE_PTR(offsets);
  HDMOE_REQUIRE_PTR(experts);
  HDMOE_REQUIRE_PTR(y_bf16);
  if (E < 1 || E > HDMOE_MAX_EXPERTS) return hdmoe_fail(HDMOE_E_SHAPE, "hdmoe_grouped_down: E=%d", E);
  if (int rc = check_dtype(weight_dtype, "hdmoe_grouped_down")) return rc;
  if (int rc = hdmoe_check_gemm_shape("hdmoe_grouped_down", weight_dtype, rows_total, H, D, BN)) return rc;
  if (rows_total == 0) return HDMOE_OK;
  return hdmoe_launch_ffn_gemm(false, weight_dtype, static_cast<const uint8_t*>(h), offsets, rows_total, E, experts,
                               static_cast<uint8_t*>(y_bf16), nullptr, 0, nullptr, nullptr, H, D, 0, 0,
                               static_cast<hipStream_t>(stream), "hdmoe_grouped_down");
}

extern "C" int hdmoe_linear(int weight_dtype, const void* a, int rows, int K, int N, const void* w,
                            const float* scale_w_dev, const float* scale_in_dev, void* out_bf16,
                            hdmoe_stream_t stream) {
  HDMOE_REQUIRE_PTR(a);
  HDMOE_REQUIRE_PTR(w);
  HDMOE_REQUIRE_PTR(out_bf16);
  if (int rc = check_dtype(weight_dtype, "hdmoe_linear")) return rc;
  if (int rc = hdmoe_check_gemm_shape("hdmoe_linear", weight_dtype, rows, K, N, BN)) return rc;
  if (weight_dtype == HDMOE_W_E4M3FN) HDMOE_REQUIRE_PTR(scale_w_dev);
  if (rows == 0) return HDMOE_OK;
  hdmoe_ffn_weights fw;
  memset(&fw, 0, sizeof(fw));
  fw.w2 = w;
  fw.scale_w2 = scale_w_dev;
  fw.scale_in2 = scale_in_dev;
  return hdmoe_launch_ffn_gemm(false, weight_dtype, nullptr, nullptr, 0, 0, nullptr, nullptr,
                               static_cast<const uint8_t*>(a), rows, &fw, static_cast<uint8_t*>(out_bf16), 0, 0, K, N,
                               static_cast<hipStream_t>(stream), "hdmoe_linear");
}

extern "C" int hdmoe_linear_bias(int weight_dtype, const void* a, int rows, int K, int N, const void* w,
                                 const float* scale_w_dev, const float* scale_in_dev, const void* bias_bf16,
                                 void* out_bf16, hdmoe_stream_t stream) {
  if (bias_bf16 == nullptr && weight_dtype != HDMOE_W_F16)
    return hdmoe_linear(weight_dtype, a, rows, K, N, w, scale_w_dev, scale_in_dev, out_bf16, stream);
  HDMOE_REQUIRE_PTR(a);
  HDMOE_REQUIRE_PTR(w);
  HDMOE_REQUIRE_PTR(out_bf16);
  if (weight_dtype != HDMOE_W_F16)
    if (int rc = check_dtype(weight_dtype, "hdmoe_linear_bias")) return rc;
  if (int rc = hdmoe_check_gemm_shape("hdmoe_linear_bias", weight_dtype == HDMOE_W_F16 ? HDMOE_W_BF16 : weight_dtype,
                                      rows, K, N, BN))
    return rc;
  if (weight_dtype == HDMOE_W_E4M3FN) HDMOE_REQUIRE_PTR(scale_w_dev);
  if (rows == 0) return HDMOE_OK;
  return hdmoe_launch_linear_bias(weight_dtype, static_cast<const uint8_t*>(a), rows, K, N,
                                  static_cast<const uint8_t*>(w), scale_w_dev, scale_in_dev,
                                  static_cast<const uint16_t*>(bias_bf16), static_cast<uint8_t*>(out_bf16),
                                  static_cast<hipStream_t>(stream), "hdmoe_linear_bias");
}

namespace {
int grouped_linear_entry(const char* what, bool f16, const void* a_bf16, const int32_t* offsets, int rows_total, int E,
                         const hdmoe_linear_weights* experts, void* out_bf16, const void* a_static_bf16,
                         int rows_static, const hdmoe_linear_weights* shared, void* out_static_bf16, int K, int N, int act,
                         hdmoe_stream_t stream, const int32_t* perm = nullptr, int T = 0) {
  if (perm != nullptr && (T <= 0 || rows_total != T * HDMOE_TOPK))
    return hdmoe_fail(HDMOE_E_SHAPE, "%s: rows_total=%d is not %d slots of T=%d tokens", what, rows_total, HDMOE_TOPK, T);
  if (E < 0 || E > HDMOE_MAX_EXPERTS) return hdmoe_fail(HDMOE_E_SHAPE, "%s: E=%d", what, E);
  if (act != HDMOE_ACT_NONE && act != HDMOE_ACT_GELU) return hdmoe_fail(HDMOE_E_SHAPE, "%s: act=%d", what, act);
  if (E > 0) {
    HDMOE_REQUIRE_PTR(a_bf16);
    HDMOE_REQUIRE_PTR(offsets);
    HDMOE_REQUIRE_PTR(experts);
    HDMOE_REQUIRE_PTR(out_bf16);
  }
  if (rows_static > 0) {
    HDMOE_REQUIRE_PTR(a_static_bf16);
    HDMOE_REQUIRE_PTR(shared);
    HDMOE_REQUIRE_PTR(out_static_bf16);
  }
  if (rows_static < 0) return hdmoe_fail(HDMOE_E_SHAPE, "%s: rows_static=%d", what, rows_static);
  const long rows_max = rows_total > rows_static ? rows_total : rows_static;
  if (int rc = hdmoe_check_gemm_shape(what, HDMOE_W_BF16, rows_max, K, N, BN)) return rc;  // same sizes for fp16
  if ((E == 0 || rows_total == 0) && rows_static == 0) return HDMOE_OK;
  return hdmoe_launch_linear_groups(static_cast<const uint8_t*>(a_bf16), offsets, rows_total, rows_total > 0 ? E : 0,
                                    experts, static_cast<uint8_t*>(out_bf16), static_cast<const uint8_t*>(a_static_bf16),
                                    rows_static, shared, static_cast<uint8_t*>(out_static_bf16), K, N, act,
                                    static_cast<hipStream_t>(stream), what, f16, perm, T, perm != nullptr ? 1 : 0);
}
}  // namespace

extern "C" int hdmoe_grouped_linear(const void* a_bf16, const int32_t* offsets, int rows_total, int E,
                                    const hdmoe_linear_weights* experts, void* out_bf16, const void* a_static_bf16,
                                    int rows_static, const hdmoe_linear_weights* shared, void* out_static_bf16, int K,
                                    int N, int act, hdmoe_stream_t stream) {
  return grouped_linear_entry("hdmoe_grouped_linear", false, a_bf16, offsets, rows_total, E, experts, out_bf16,
                              a_static_bf16, rows_static, shared, out_static_bf16, K, N, act, stream);
}

extern "C" int hdmoe_grouped_linear_f16(const void* a_f16, const int32_t* offsets, int rows_total, int E,
                                        const hdmoe_linear_weights* experts, void* out_f16, const void* a_static_f16,
                                        int rows_static, const hdmoe_linear_weights* shared, void* out_static_f16,
                                        int K, int N, int act, hdmoe_stream_t stream) {
  return grouped_linear_entry("hdmoe_grouped_linear_f16", true, a_f16, offsets, rows_total, E, experts, out_f16,
                              a_static_f16, rows_static, shared, out_static_f16, K, N, act, stream);
}

// The first Linear of the experts on the tokens themselves: sorted row r is token perm[r] / 2 (the rows the boolean
// masks of the reference select, read through the dispatch permutation instead of from a copy in expert order).
extern "C" int hdmoe_grouped_linear_tokens(int act_dtype, const void* x, int T, const int32_t* perm,
                                           const int32_t* offsets, int E, const hdmoe_linear_weights* experts, void* out,
                                           const hdmoe_linear_weights* shared, void* out_shared, int K, int N, int act,
                                           hdmoe_stream_t stream) {
  HDMOE_REQUIRE_PTR(perm);
  if (act_dtype != HDMOE_W_BF16 && act_dtype != HDMOE_W_F16)
    return hdmoe_fail(HDMOE_E_SHAPE, "hdmoe_grouped_linear_tokens: act_dtype=%d is neither HDMOE_W_BF16 nor HDMOE_W_F16",
                      act_dtype);
  if (T < 0 || E < 1) return hdmoe_fail(HDMOE_E_SHAPE, "hdmoe_grouped_linear_tokens: T=%d E=%d", T, E);
  if (T == 0) return HDMOE_OK;
  return grouped_linear_entry("hdmoe_grouped_linear_tokens", act_dtype == HDMOE_W_F16, x, offsets, T * HDMOE_TOPK, E,
                              experts, out, x, shared != nullptr ? T : 0, shared, out_shared, K, N, act, stream, perm, T);
}

// The same Linear for callers that bring working memory (hdmoe_linear_args in hdmoe.h): tiles that would leave most of the
// chip idle are cut along K, and the GELU hides behind the next tile.
namespace {
int linear_groups_check(const hdmoe_linear_args* p) {
  const char* what = "hdmoe_linear_groups";
  const bool w8 = p->weight_dtype == HDMOE_W_E4M3FN_UPCAST;
  if ((p->act_dtype != HDMOE_W_BF16 && p->act_dtype != HDMOE_W_F16) || (w8 ? p->act_dtype != HDMOE_W_BF16 : p->weight_dtype != p->act_dtype))
    return hdmoe_fail(HDMOE_E_SHAPE, "%s: act_dtype=%d weight_dtype=%d", what, p->act_dtype, p->weight_dtype);
  if (p->E < 0 || p->E > HDMOE_MAX_EXPERTS || p->rows < 0 || p->rows_static < 0 || p->T < 0)
    return hdmoe_fail(HDMOE_E_SHAPE, "%s: E=%d rows=%d rows_static=%d T=%d", what, p->E, p->rows, p->rows_static, p->T);
  if (p->act != HDMOE_ACT_NONE && p->act != HDMOE_ACT_GELU) return hdmoe_fail(HDMOE_E_SHAPE, "%s: act=%d", what, p->act);
  if (p->perm != nullptr && p->rows != p->T * HDMOE_TOPK)
    return hdmoe_fail(HDMOE_E_SHAPE, "%s: rows=%d is not %d slots of T=%d tokens", what, p->rows, HDMOE_TOPK, p->T);
  const long rows_max = p->rows > p->rows_static ? p->rows : p->rows_static;
  return hdmoe_check_gemm_shape(what, HDMOE_W_BF16, rows_max, p->K, p->N, BN);
}
// what the kernels that run can use: room for the activation, and for the parts of tail tiles
size_t linear_groups_scratch(const hdmoe_linear_args* p) {
  if (p->act != HDMOE_ACT_GELU || !g4_takes_k(1, p->K * 2, 0, 0)) return 0;
  return hdmoe_align_up((size_t)HDMOE_NUM_CU * G4_SCRATCH, 256);
}
size_t linear_groups_tail(const hdmoe_linear_args* p) {
  if (p->fixed_k_cut != 0) return 0;
  const int n_dyn = p->rows > 0 ? p->E : 0;
  return g4_tail_room(n_dyn, n_dyn > 0 ? p->rows / n_dyn : 0, p->N, p->K * 2, p->rows_static, p->N, p->K * 2, BN,
                      p->weight_dtype == HDMOE_W_E4M3FN_UPCAST);
}
}  // namespace

extern "C" size_t hdmoe_linear_groups_workspace_bytes(const hdmoe_linear_args* p) {
  if (p == nullptr || linear_groups_check(p) != HDMOE_OK) return 0;
  return linear_groups_scratch(p) + linear_groups_tail(p);
}

extern "C" int hdmoe_linear_groups(const hdmoe_linear_args* p, hdmoe_stream_t stream) {
  HDMOE_REQUIRE_PTR(p);
  if (int rc = linear_groups_check(p)) return rc;
  if (p->E > 0 && p->rows > 0) {
    HDMOE_REQUIRE_PTR(p->a);
    HDMOE_REQUIRE_PTR(p->offsets);
    HDMOE_REQUIRE_PTR(p->experts);
    HDMOE_REQUIRE_PTR(p->out);
  }
  if (p->rows_static > 0) {
    HDMOE_REQUIRE_PTR(p->a_static);
    HDMOE_REQUIRE_PTR(p->shared);
    HDMOE_REQUIRE_PTR(p->out_static);
  }
  uint8_t* ws = static_cast<uint8_t*>(p->workspace);
  if (ws != nullptr && (p->workspace_bytes < hdmoe_linear_groups_workspace_bytes(p) || (reinterpret_cast<uintptr_t>(ws) & 255)))
    return hdmoe_fail(HDMOE_E_WORKSPACE, "hdmoe_linear_groups: workspace %zu bytes, need %zu (256-byte aligned)",
                      p->workspace_bytes, hdmoe_linear_groups_workspace_bytes(p));
  if ((p->E == 0 || p->rows == 0) && p->rows_static == 0) return HDMOE_OK;
  const size_t sb = linear_groups_scratch(p);
  return hdmoe_launch_linear_groups(static_cast<const uint8_t*>(p->a), p->offsets, p->rows, p->rows > 0 ? p->E : 0, p->experts,
                                    static_cast<uint8_t*>(p->out), static_cast<const uint8_t*>(p->a_static), p->rows_static,
                                    p->shared, static_cast<uint8_t*>(p->out_static), p->K, p->N, p->act,
                                    static_cast<hipStream_t>(stream), "hdmoe_linear_groups", p->act_dtype == HDMOE_W_F16,
                                    p->perm, p->T, p->perm != nullptr ? 1 : 0, p->weight_dtype == HDMOE_W_E4M3FN_UPCAST,
                                    ws != nullptr && linear_groups_tail(p) > 0 ? reinterpret_cast<float*>(ws + sb) : nullptr,
                                    ws != nullptr && sb > 0 ? ws : nullptr);
}

// The plan of gemm4w_kernel's tail tiles for `tiles` tiles of K elements with `padding` rows without a row of a segment between
// them (0 to 255 per tile): whole rounds, tiles left over, and the parts that each of those is cut into. For tests and reports.
extern "C" int hdmoe_tail_plan(int weight_dtype, int tiles, int K, int padding, int* rounds, int* left) {
  if (tiles <= 0 || K <= 0 || K > 0x7fff * BK / 2 || padding < 0 || padding / tiles >= G4_BM) return 0;
  const G4Tail t = g4_plan_tail(tiles, HDMOE_NUM_CU, K / BK, weight_dtype == HDMOE_W_E4M3FN_UPCAST ? 3 : 2, padding);
  if (rounds != nullptr) *rounds = t.rounds;
  if (left != nullptr) *left = t.tiles;
  return t.parts;
}

// Height of the tiles of a Linear on 16-bit activations that is given the working memory it asks for: 256, or fewer rows where no
// tile is cut and lower ones fill the rounds better (g4_best_cap). For tests and reports.
extern "C" int hdmoe_linear_tile_rows(int weight_dtype, int rows, int K, int N) {
  const bool w8 = weight_dtype == HDMOE_W_E4M3FN_UPCAST;
  if ((!w8 && weight_dtype != HDMOE_W_BF16 && weight_dtype != HDMOE_W_F16) || rows <= 0 || K <= 0 || N <= 0 || N % BN != 0 ||
      K > 0x7fff * BK / 2 || K % BK != 0 || K / BK < (w8 ? 3 : 2))
    return 0;
  GemmArgs args;
  memset(&args, 0, sizeof(args));
  args.G = 1;
  args.g[0].row_end = rows;
  args.g[0].n_out = N;
  args.g[0].kbytes = K * 2;
  float room = 0.0f;
  if (g4_tail_room(0, 0, 0, 0, rows, N, K * 2, BN, w8) > 0) args.tail = &room;
  else if (rows <= 128 && !w8) return 0;   // the 8-wave kernel's
  const int cap = g4_host_cap(args, BN, w8 ? 3 : 2, HDMOE_NUM_CU);
  return 32 * (cap > 0 ? g4_heights(rows, cap).height : G4_BM / 32);
}

// The same for a Linear on e4m3fn activations that the 4-wave kernel takes.
extern "C" int hdmoe_fp8_linear_tile_rows(int rows, int K, int N) {
  if (rows <= 0 || K <= 0 || N <= 0 || N % BN != 0 || K > 0x7fff * BK || K % BK != 0 || !g4_takes_k(0, 0, rows, K)) return 0;
  GemmArgs args;
  memset(&args, 0, sizeof(args));
  args.G = 1;
  args.g[0].row_end = rows;
  args.g[0].n_out = N;
  args.g[0].kbytes = K;
  const int cap = g4_host_cap(args, BN, 2, HDMOE_NUM_CU);
  return 32 * g4_heights(cap > 0 || rows < G4_BM ? rows : G4_BM, cap > 0 ? cap : G4_BM / 32).height;
}

// What g4_two_lengths makes of a layer's down projection (E segments of `rows` rows each and K elements of e4m3fn, one more of rows_static and
// K_static): the longest block in hundredths of a pair of K steps, 0 for sizes it does not take. For tests and reports.
extern "C" int hdmoe_two_lengths(int E, const int* rows, int K, int rows_static, int K_static, int N, int cap_long, int cap_short, int* light_rounds) {
  auto cap_ok = [](int cap) { return cap >= G4_MIN_BLOCKS && cap <= G4_BM / 32; };
  if (E <= 0 || E > HDMOE_MAX_EXPERTS || rows == nullptr || rows_static <= 0 || K <= 0 || K_static <= 0 || K % (2 * BK) != 0 || K_static % (2 * BK) != 0 ||
      N <= 0 || N % BN != 0 || !cap_ok(cap_long) || !cap_ok(cap_short))
    return 0;
  struct Sizes {
    int E, K, K_static, N, rows_static;
    const int* of;
    bool dynamic(int g) const { return g < E; }
    int rows(int g) const { return g < E ? of[g] : rows_static; }
    int bytes(int g) const { return g < E ? K : K_static; }
    int ntiles(int, int feat) const { return N / feat; }
  };
  const G4Two t = g4_two_lengths(Sizes{E, K, K_static, N, rows_static, rows}, E + 1, K >= K_static ? 1 : -1, BN, cap_long, cap_short);
  if (light_rounds != nullptr) *light_rounds = t.light_rounds;
  return t.cost;
}

// Bytes a feed-forward's contractions on 16-bit activations can use for the parts of tail tiles: E experts of hidden width H on
// rows_dyn rows together, one more of width Hs on rows_static. down_uncut: its down projection is not cut along K by itself.
size_t hdmoe_tail_bytes(int weight_dtype, int rows_dyn, int E, int rows_static, int D, int H, int Hs, bool down_uncut) {
  if (weight_dtype == HDMOE_W_E4M3FN) return 0;
  const bool w8 = weight_dtype == HDMOE_W_E4M3FN_UPCAST;
  const int n_dyn = rows_dyn > 0 ? E : 0, mean = n_dyn > 0 ? rows_dyn / n_dyn : 0;
  GemmShape sh;
  sh.swiglu = true; sh.fp8 = false; sh.split = false; sh.w8 = w8; sh.w4_fits = sh.s224_fits = false; sh.kbytes = D * 2;
  sh.rows_dyn = rows_dyn; sh.n_dyn = n_dyn; sh.rows_static = rows_static;
  sh.N_dyn = H; sh.N_static = Hs;
  sh.g4_takes = g4_takes_k(rows_dyn, D * 2, rows_static, D * 2);
  const size_t up = swiglu_on_g4(sh, true) ? g4_tail_room(n_dyn, mean, H, D * 2, rows_static, Hs, D * 2, BN / 2, w8) : 0;
  const size_t down = down_uncut ? g4_tail_room(n_dyn, mean, D, H * 2, rows_static, D, Hs * 2, BN, w8) : 0;
  return up > down ? up : down;
}
