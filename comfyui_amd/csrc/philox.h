// Philox4x32-10 counter-based generator (Salmon, Moraes, Dror, Shaw: "Parallel random numbers: as easy as
// 1, 2, 3", SC'11), written from the published round function. One call turns a 128-bit counter and a 64-bit
// key into four 32-bit words; there is no state, so element i of a tensor always draws the same numbers
// whatever the launch shape. Shared by the HIP kernels and the CPU checker.
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#define HDMOE_PHILOX_HD __host__ __device__ __forceinline__
#else
#define HDMOE_PHILOX_HD static inline
#endif

HDMOE_PHILOX_HD uint32_t hdmoe_xor3(uint32_t a, uint32_t b, uint32_t c) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);   // one instruction, which the compiler does not form by itself
#else
  return a ^ b ^ c;
#endif
}

HDMOE_PHILOX_HD void hdmoe_philox4x32_10(const uint32_t ctr[4], const uint32_t key[2], uint32_t out[4]) {
  uint32_t c0 = ctr[0], c1 = ctr[1], c2 = ctr[2], c3 = ctr[3];
  uint32_t k0 = key[0], k1 = key[1];
#if defined(__HIPCC__)
#pragma unroll   // products of a counter word that is zero or the same for the whole wave drop out
#endif
  for (int r = 0; r < 10; ++r) {
    const uint64_t p0 = (uint64_t)0xD2511F53u * c0;
    const uint64_t p1 = (uint64_t)0xCD9E8D57u * c2;
    const uint32_t n0 = hdmoe_xor3((uint32_t)(p1 >> 32), c1, k0);
    const uint32_t n1 = (uint32_t)p1;
    const uint32_t n2 = hdmoe_xor3((uint32_t)(p0 >> 32), c3, k1);
    const uint32_t n3 = (uint32_t)p0;
    c0 = n0; c1 = n1; c2 = n2; c3 = n3;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
  out[0] = c0; out[1] = c1; out[2] = c2; out[3] = c3;
}
