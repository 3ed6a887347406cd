// Weight-side maintenance for scaled-fp8 Linears: stochastic rounding of a patched weight back to
// float8_e4m3fn, fused with the division by scale_weight
// (/root/reference/comfy/ops.py:419-426 set_weight -> /root/reference/comfy/float.py:14-67).
//
// As in the reference the value is first rounded to float16; it then lands on one of its two e4m3fn neighbours,
// the upper one with probability equal to its fractional position between them (position + u floored, u uniform
// in [0,1)), magnitudes of 448 and more saturate to +-448, zero stays zero. The uniform numbers are not torch's:
// element i takes word (i & 3) of Philox4x32-10(counter = i >> 2, key = seed), 24 bits of it, so the result depends
// only on (value, seed, i).
#include "common.h"
#include "numfmt.h"
#include "philox.h"

namespace {

constexpr int THREADS = 256;
constexpr int GROUPS = 4;                       // groups of 4 elements per thread, THREADS apart
constexpr long CHUNK = (long)THREADS * GROUPS;  // groups per block

// What bounds the kernel: vector instructions (18 32 x 32 -> 64 bit products, which are the larger half of the time, and 18 other
// operations for the random words of 4 elements, about 22 per element beside them; the bytes take 14 us at 6.4 TB/s). Hence no branches per element, one product
// where the division's last bits cannot matter, the rounding on float16 bits, two values to a register where the instruction set
// has it, and all loads of a thread (16 or 8 bytes each) in flight at once. 6912 x 2560 fp32 on MI355X, whole set_weight: 24.4 us with a
// corrected division and fp32 arithmetic for every element, 19.8 us so; bf16 30.0 -> 21.7.

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// two values rounded to float16 (to nearest even)
__device__ __forceinline__ uint32_t half_pair(float a, float b) {
  const f32x2 v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2));
}
__device__ __forceinline__ u16x2 pk(uint32_t v) { return __builtin_bit_cast(u16x2, v); }

// Four values in float16 (packed pairs), four random words -> four e4m3fn bytes.
// Normal binades: a float16's exponent and mantissa are the code's with 7 more bits, so the sum of mantissa and u (in 128ths of a step)
// carries into the code by itself. Below 2^-6: steps of 2^-9 from zero. The sum is rounded to fp32 once.
__device__ __forceinline__ uint32_t sr_bytes(const uint32_t (&w)[2], const uint32_t (&rnd)[4]) {
  u16x2 code[2], odd = {0, 0};
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const uint32_t mag = w[p] & 0x7fff7fffu, mant = w[p] & 0x03ff03ffu;
    odd = __builtin_elementwise_max(odd, pk(mag) - pk(0x00010001u));      // zeros and NaN: 0x7c00 and above
    uint32_t sum[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const float a = (float)__builtin_bit_cast(f16x2, mag)[h];
      const float m = (float)(h ? mant >> 16 : mant & 0xffffu);
      const float t = a < 0x1p-6f ? a * 65536.0f : m;
      sum[h] = (uint32_t)__builtin_fmaf((float)(rnd[2 * p + h] >> 8), 0x1p-17f, t);   // up to 1152
    }
    const u16x2 expo = __builtin_elementwise_max(pk(w[p] & 0x7c007c00u), pk(0x20002000u)) - pk(0x20002000u);
    code[p] = __builtin_elementwise_min((expo + pk(sum[0] | sum[1] << 16)) >> 7, pk(0x007e007eu));   // 448 and beyond (inf too) saturate
  }
  uint32_t codes = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, code[1]), __builtin_bit_cast(uint32_t, code[0]), 0x06040200u);
  uint32_t signs = __builtin_amdgcn_perm(w[1], w[0], 0x07050301u) & 0x80808080u;
  if (__any(max(odd.x, odd.y) >= 0x7c00)) {   // somewhere in the wave
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t mag = (j & 1 ? w[j >> 1] >> 16 : w[j >> 1]) & 0x7fffu;
      if (mag > 0x7c00u) codes |= 0x7fu << (8 * j);
      // a zero becomes +0 (the reference multiplies by sign(0) = 0); a value rounded down to zero keeps its sign
      if (mag == 0) signs &= ~(0x80u << (8 * j));
    }
  }
  return codes | signs;
}

// Division of many values by one divisor, with the bits of a correctly rounded division wherever the float16 or bf16 rounding
// that follows can tell (P. Markstein, IBM J. Res. Dev. 34 (1990): with y = RN(1/s) and a quotient q within one unit in the
// last place, RN(q + RN(x - q s) y) is RN(x / s); the first product may be off by more, so the step is taken twice).
// Needs the remainders exact: |s| in [2^-40, 2^40]; a quotient below 2^-50 may lose digits and is 0 in float16 either way;
// one of 2^20 or more is kept as the plain product (it saturates, and infinities and NaN pass unharmed).
// The plain product and the correctly rounded quotient are both within 0.75 * 2^-22 of the product: where the ends of an interval of twice that
// round to the same number, so do they (rounding is monotonic). That settles all but one in 950 fp32 values (normally distributed, largest
// at 448; 3 m in 4096 for a mantissa m), and so three of four waves, which have 256 each, take no correction.
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
    float x[4];
    uint32_t w[2];
    bool settled = !ANY_DIVISOR;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (BF16) x[j] = hdmoe_bf16_to_f32(raw[i].v[j]);
      else x[j] = raw[i].v[j];
    }
    // two values in the format the quotient is rounded to first: bf16 for bf16 weights
    auto pair = [](float a, float b) { return BF16 ? hdmoe_dev_pack_bf16(a, b) : half_pair(a, b); };
    if constexpr (!ANY_DIVISOR) {
      constexpr float LOW = 1.0f - 0x1.8p-22f, HIGH = 1.0f + 0x1.8p-22f;
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const float a = x[2 * p] * div.y, b = x[2 * p + 1] * div.y;
        w[p] = pair(a * LOW, b * LOW);
        settled = settled && w[p] == pair(a * HIGH, b * HIGH);
      }
    }
    if (!__all(settled)) {
#pragma unroll
      for (int p = 0; p < 2; ++p) w[p] = pair(div(x[2 * p]), div(x[2 * p + 1]));
    }
    if constexpr (BF16) {
#pragma unroll
      for (int p = 0; p < 2; ++p) w[p] = half_pair(__uint_as_float(w[p] << 16), __uint_as_float(w[p] & 0xffff0000u));
    }
    const uint32_t packed = sr_bytes(w, r);
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
