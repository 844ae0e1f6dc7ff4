// Key-similarity cap of a kv-block: the device code shared by the stand-alone kernel and the pooling pass that forms the cap beside
// the pooled rows.  A thread owns 8 consecutive tokens x 8 channels, D / 8 neighbouring lanes a token group.
#pragma once
#include "psa_common.h"

namespace psa_ksim_row {

// this thread's part of the 8 squared norms and of the dots (0,1) (2,3) (4,5) (6,7) | (0,3) (4,7) | (0,7) of its token group
__device__ __forceinline__ void pair_sums(const float (&f)[8][8], float (&v)[15]) {
#pragma unroll
  for (int i = 0; i < 15; ++i) v[i] = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] += f[i][e] * f[i][e];
    v[8] += f[0][e] * f[1][e];
    v[9] += f[2][e] * f[3][e];
    v[10] += f[4][e] * f[5][e];
    v[11] += f[6][e] * f[7][e];
    v[12] += f[0][e] * f[3][e];
    v[13] += f[4][e] * f[7][e];
    v[14] += f[0][e] * f[7][e];
  }
}
// ... summed over the lpr lanes of the group
__device__ __forceinline__ void group_sums(float (&v)[15], int lpr) {
  for (int o = lpr >> 1; o > 0; o >>= 1) {
#pragma unroll
    for (int i = 0; i < 15; ++i) v[i] += __shfl_xor(v[i], o, 64);
  }
}
// the group's cosines at distance 1, 3 and 7
__device__ __forceinline__ void group_cosines(const float (&v)[15], float& c2, float& c4, float& c8) {
  float n[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) n[i] = sqrtf(v[i] + 1e-12f);
  c2 = v[8] / (n[0] * n[1] + 1e-6f) + v[9] / (n[2] * n[3] + 1e-6f) + v[10] / (n[4] * n[5] + 1e-6f) + v[11] / (n[6] * n[7] + 1e-6f);
  c4 = v[12] / (n[0] * n[3] + 1e-6f) + v[13] / (n[4] * n[7] + 1e-6f);
  c8 = v[14] / (n[0] * n[7] + 1e-6f);
}
// a > b as IEEE 754 has it, false where either is no number, in every file that includes this: without NaN semantics (psa_estimate.hip)
// the compiler may turn the comparison round and call a NaN above everything.  The bits go through an empty assembly statement, or
// the test for a NaN would be dropped as one that never holds.
__device__ __forceinline__ bool above(float a, float b) {
  uint32_t x = __builtin_bit_cast(uint32_t, a), y = __builtin_bit_cast(uint32_t, b);
  asm("" : "+v"(x), "+v"(y));
  constexpr uint32_t INF = 0x7f800000u, ABS = 0x7fffffffu;
  return (x & ABS) <= INF && (y & ABS) <= INF && __builtin_bit_cast(float, x) > __builtin_bit_cast(float, y);
}
// cap of a block of bn tokens from the cosines of its bn / 8 groups: 1 where a mean cosine is no number (a key that is not finite, or whose
// squared norm is not)
__device__ __forceinline__ int block_cap(const float* c2, const float* c4, const float* c8, int bn, float t2, float t4, float t8) {
  const int ng = bn >> 3;
  float s2 = 0.f, s4 = 0.f, s8 = 0.f;
  for (int i = 0; i < ng; ++i) {
    s2 += c2[i];
    s4 += c4[i];
    s8 += c8[i];
  }
  s2 /= (float)(bn >> 1);
  s4 /= (float)(bn >> 2);
  s8 /= (float)(bn >> 3);
  int lv = 1;
  if (above(s2, t2)) lv = 2;
  if (above(s4, t4)) lv = 4;
  if (above(s8, t8)) lv = 8;
  return lv;
}

}  // namespace psa_ksim_row
