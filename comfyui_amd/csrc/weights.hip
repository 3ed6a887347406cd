// Weight-side maintenance for scaled-fp8 Linears: stochastic rounding of a patched weight back to
// float8_e4m3fn, fused with the division by scale_weight
// (/root/reference/comfy/ops.py:419-426 set_weight -> /root/reference/comfy/float.py:14-67).
//
// As in the reference the value is first rounded to float16; it then lands on one of its two e4m3fn neighbours,
// the upper one with probability equal to its fractional position between them (position + u floored, u uniform
// in [0,1)), magnitudes of 448 and more saturate to +-448, zero stays zero. The uniform numbers are not torch's:
// element i takes word (i & 3) of Philox4x32-10(counter = i >> 2, key = seed), 24 bits of it, so the result depends
// only on (value, seed, i).
#include <hip/hip_fp16.h>

#include "common.h"
#include "numfmt.h"
#include "philox.h"

namespace {

constexpr int THREADS = 256;
constexpr int GROUPS = 4;                       // groups of 4 elements per thread, THREADS apart
constexpr long CHUNK = (long)THREADS * GROUPS;  // groups per block

// What bounds the kernel: vector instructions (18 32 x 32 -> 64 bit products and 50 other operations for the random words of 4
// elements, about 25 per element beside them): 24 us where the bytes take 14 us at 6.4 TB/s. Hence no branches per element, a division
// by the one divisor that multiplies by its reciprocal, and all loads of a thread (16 or 8 bytes each) in flight at once.
// 6912 x 2560 fp32 on MI355X, whole set_weight: 37.9 us with the general division, branches, element loads and a copy of the
// result into the weight; 24.4 us.

// |value| already rounded to float16 (as fp32), one 32-bit random word -> e4m3fn code without sign
__device__ __forceinline__ uint32_t sr_code(float a, uint32_t rnd) {
  const float u = (float)(rnd >> 8) * 0x1p-24f;
  const int e = max((int)(__float_as_uint(a) >> 23), 120);  // biased exponent; 120: everything below the smallest normal, 2^-6
  // normal binade 2^(e-127) * (1 + k/8): position in eighths, counted from the binade's start; below: steps of 2^-9
  const float scaled = a * __uint_as_float((uint32_t)(257 - max(e, 121)) << 23);
  const float pos = e > 120 ? scaled - 8.0f : scaled;                  // exact
  uint32_t code = ((uint32_t)(e - 120) << 3) + (uint32_t)(pos + u);     // 0..8, 8 carries into the next binade
  code = a < 448.0f ? code : 0x7eu;                                    // 448 and beyond (inf too) saturate
  return a != a ? 0x7fu : code;
}

// Division of many values by one divisor, with the bits of a correctly rounded division wherever the float16 or bf16 rounding
// that follows can tell (P. Markstein, IBM J. Res. Dev. 34 (1990): with y = RN(1/s) and a quotient q within one unit in the
// last place, RN(q + RN(x - q s) y) is RN(x / s); the first product may be off by more, so the step is taken twice).
// Needs the remainders exact: |s| in [2^-40, 2^40]; a quotient below 2^-50 may lose digits and is 0 in float16 either way;
// one of 2^20 or more is kept as the plain product (it saturates, and infinities and NaN pass unharmed).
template <bool ANY_DIVISOR>
struct Divider {
  float s, y;
  __device__ __forceinline__ explicit Divider(float d) : s(d), y(ANY_DIVISOR ? 0.0f : __fdiv_rn(1.0f, d)) {}
  __device__ __forceinline__ float operator()(float x) const {
    if (ANY_DIVISOR) return __fdiv_rn(x, s);
    const float p = x * y;
    float q = __builtin_fmaf(__builtin_fmaf(-p, s, x), y, p);
    q = __builtin_fmaf(__builtin_fmaf(-q, s, x), y, q);
    return __builtin_fabsf(p) < 0x1p20f ? q : p;
  }
};

// The raw 4 elements of a group; WIDE: the source is aligned to a group. Past the end: zeros.
template <typename SRC>
struct Raw4 { SRC v[4]; };

template <typename SRC, bool WIDE>
__device__ __forceinline__ Raw4<SRC> load_group(const SRC* src, long n, long g) {
  Raw4<SRC> r;
  if (WIDE && g * 4 + 3 < n) {
    if constexpr (sizeof(SRC) == 4) {
      const float4 v = *reinterpret_cast<const float4*>(src + g * 4);
      r.v[0] = v.x; r.v[1] = v.y; r.v[2] = v.z; r.v[3] = v.w;
    } else {
      const uint2 v = *reinterpret_cast<const uint2*>(src + g * 4);
      r.v[0] = (SRC)(v.x & 0xffffu); r.v[1] = (SRC)(v.x >> 16); r.v[2] = (SRC)(v.y & 0xffffu); r.v[3] = (SRC)(v.y >> 16);
    }
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) r.v[j] = g * 4 + j < n ? src[g * 4 + j] : SRC(0);
  }
  return r;
}

template <typename SRC, bool ANY_DIVISOR>
__device__ __forceinline__ void round_groups(const Raw4<SRC> (&raw)[GROUPS], long n, long g0, float scale, const uint32_t key[2],
                                             uint8_t* out) {
  // bf16 weights: the reference divides two bf16 tensors, so the scale and the quotient are rounded to bf16
  constexpr bool BF16 = sizeof(SRC) == 2;
  const Divider<ANY_DIVISOR> div(scale);
  const uint32_t ctr1 = (uint32_t)((uint64_t)blockIdx.x * CHUNK >> 32);   // a chunk does not cross 2^32
#pragma unroll
  for (int i = 0; i < GROUPS; ++i) {
    const long g = g0 + i * THREADS;
    if (g * 4 >= n) return;
    const uint32_t ctr[4] = {(uint32_t)g, ctr1, 0u, 0u};
    uint32_t r[4];
    hdmoe_philox4x32_10(ctr, key, r);
    uint32_t packed = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float q;
      if constexpr (BF16) q = hdmoe_round_bf16(div(hdmoe_bf16_to_f32(raw[i].v[j])));
      else q = div(raw[i].v[j]);
      const float x = __half2float(__float2half_rn(q));
      // an exact zero stays +0 (the reference multiplies by sign(0) = 0); a value rounded down to zero keeps its sign
      const uint32_t code = sr_code(__builtin_fabsf(x), r[j]);
      const uint32_t sign = x != 0.0f ? (__float_as_uint(x) >> 24) & 0x80u : 0u;
      packed |= (code | sign) << (8 * j);
    }
    if (g * 4 + 3 < n) {
      *reinterpret_cast<uint32_t*>(out + g * 4) = packed;
    } else {
      for (int j = 0; g * 4 + j < n; ++j) out[g * 4 + j] = (uint8_t)(packed >> (8 * j));
    }
  }
}

template <typename SRC, bool WIDE>
__global__ __launch_bounds__(THREADS) void stochastic_round_kernel(const SRC* __restrict__ src, long n,
                                                                   const float* __restrict__ scale, uint32_t seed_lo,
                                                                   uint32_t seed_hi, uint8_t* __restrict__ out) {
  const uint32_t key[2] = {seed_lo, seed_hi};
  const long g0 = (long)blockIdx.x * CHUNK + threadIdx.x;
  Raw4<SRC> raw[GROUPS];
#pragma unroll
  for (int i = 0; i < GROUPS; ++i) raw[i] = load_group<SRC, WIDE>(src, n, g0 + i * THREADS);
  float s = scale ? *scale : 1.0f;
  if (sizeof(SRC) == 2) s = hdmoe_round_bf16(s);
  const float m = __builtin_fabsf(s);
  if (m >= 0x1p-40f && m <= 0x1p40f) round_groups<SRC, false>(raw, n, g0, s, key, out);
  else round_groups<SRC, true>(raw, n, g0, s, key, out);
}

template <typename SRC>
void launch(const void* src, int64_t n, const float* scale, uint64_t seed, void* out, hipStream_t stream) {
  const long blocks = ((n + 3) / 4 + CHUNK - 1) / CHUNK;
  const bool wide = ((uintptr_t)src & (4 * sizeof(SRC) - 1)) == 0;   // a view may start anywhere
  hipLaunchKernelGGL((wide ? stochastic_round_kernel<SRC, true> : stochastic_round_kernel<SRC, false>), dim3((uint32_t)blocks),
                     dim3(THREADS), 0, stream, static_cast<const SRC*>(src), (long)n, scale, (uint32_t)seed,
                     (uint32_t)(seed >> 32), static_cast<uint8_t*>(out));
}

}  // namespace

extern "C" int hdmoe_stochastic_round_e4m3fn(int src_dtype, const void* src, int64_t n, const float* scale_dev,
                                             uint64_t seed, void* out_e4m3fn, hdmoe_stream_t stream) {
  HDMOE_REQUIRE_PTR(src);
  HDMOE_REQUIRE_PTR(out_e4m3fn);
  if (n < 0) return hdmoe_fail(HDMOE_E_SHAPE, "hdmoe_stochastic_round_e4m3fn: n=%lld", (long long)n);
  if (src_dtype != HDMOE_SRC_BF16 && src_dtype != HDMOE_SRC_F32)
    return hdmoe_fail(HDMOE_E_SHAPE, "hdmoe_stochastic_round_e4m3fn: src_dtype=%d is neither HDMOE_SRC_BF16 nor HDMOE_SRC_F32",
                      src_dtype);
  if (((uintptr_t)out_e4m3fn & 3u) != 0)
    return hdmoe_fail(HDMOE_E_SHAPE, "hdmoe_stochastic_round_e4m3fn: output must be 4-byte aligned");
  if (n == 0) return HDMOE_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (src_dtype == HDMOE_SRC_F32) launch<float>(src, n, scale_dev, seed, out_e4m3fn, s);
  else launch<uint16_t>(src, n, scale_dev, seed, out_e4m3fn, s);
  return hdmoe_check_launch("hdmoe_stochastic_round_e4m3fn");
}
