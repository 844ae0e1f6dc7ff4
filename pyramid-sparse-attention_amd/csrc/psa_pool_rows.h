// Pyramid pooling of K and V: the device code shared by the pooling kernel (psa_pool.hip) and the launches that pool beside other work.
#pragma once
#include "psa_common.h"
#include "psa_ksim_row.h"

struct PoolParams {
  const char* src[2];    // element pointers as bytes; strides below are in elements
  int64_t sb[2], sh[2], sl[2];
  char* dst[2];
  int H, L, D;
  int64_t npad;
  const int32_t* index;  // indexed form: source row of every position, else null
  char* ord[2];          // indexed form: the re-ordered rows [B, H, L, D] (strides ob / oh / ol)
  int64_t ob[2], oh[2], ol[2];
  int32_t* cap;          // with a similarity cap: [B, H, npad / bn]
  int bn;
  float t2, t4, t8;
};

// a 16-byte chunk of a row as floats, and back (rounded to the element type, nearest even)
struct PoolF32 {
  static constexpr int CH = 4, ES = 4;
  typedef float f32x4_t __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ void unpack(const u32x4& w, float* f) {
    const f32x4_t x = __builtin_bit_cast(f32x4_t, w);  // (the whole vector at once: a bit cast of one element of a vector is not addressable)
    f[0] = x.x; f[1] = x.y; f[2] = x.z; f[3] = x.w;
  }
  static __device__ __forceinline__ u32x4 pack(float* f) {  // (fp32: nothing to round)
    f32x4_t x;
    x.x = f[0]; x.y = f[1]; x.z = f[2]; x.w = f[3];
    return __builtin_bit_cast(u32x4, x);
  }
};
template <class ET>
struct Pool16 {
  static constexpr int CH = 8, ES = 2;
  static __device__ __forceinline__ void unpack(const u32x4& w, float* f) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f[2 * j] = ET::from_bits(w[j] & 0xffffu);
      f[2 * j + 1] = ET::from_bits(w[j] >> 16);
    }
  }
  static __device__ __forceinline__ u32x4 pack(float* f) {  // rounds f in place
    u32x4 r;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      r[j] = ET::pack2(f[2 * j], f[2 * j + 1]);
      f[2 * j] = ET::from_bits(r[j] & 0xffffu);
      f[2 * j + 1] = ET::from_bits(r[j] >> 16);
    }
    return r;
  }
};

// mean of two rows, rounded to the element type: returned both packed and as floats for the next level
template <class PT>
__device__ __forceinline__ u32x4 mean2(const float* a, const float* b, float* out) {
#pragma unroll
  for (int j = 0; j < PT::CH; ++j) out[j] = (a[j] + b[j]) * 0.5f;
  return PT::pack(out);
}

template <bool INDEXED, bool CAP, class PT>
__device__ __forceinline__ void pool_rows(const PoolParams& p, int bx, int bh, int which, int64_t BH) {
  constexpr int CH = PT::CH, ES = PT::ES;
  const int b = bh / p.H, h = bh % p.H;
  const int chunks = p.D / CH;
  const int64_t unit = (int64_t)bx * 256 + threadIdx.x;
  const int64_t g = unit / chunks;  // group of 8 tokens
  const int c = (int)(unit % chunks);
  const int64_t n8 = p.npad >> 3;
  const bool live = g < n8;  // (with a cap the workgroup meets at a barrier: idle threads, whole kv-blocks of them, stay)
  if (!CAP && !live) return;

  const char* src = p.src[which] + (b * p.sb[which] + h * p.sh[which] + c * CH) * ES;
  const int64_t sl = p.sl[which] * ES;
  float f[8][CH];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    int64_t row = g * 8 + i;
    const bool real = row < p.L && (!CAP || live);
    row = real ? row : (int64_t)(p.L - 1);
    const int64_t srow = INDEXED ? (int64_t)clamp_row(p.index[row], p.L) : row;
    u32x4 w = *(const u32x4*)(src + srow * sl);
    if (INDEXED && real)
      __builtin_nontemporal_store(w, (u32x4*)(p.ord[which] + (b * p.ob[which] + h * p.oh[which] + row * p.ol[which] + c * CH) * ES));
    PT::unpack(w, f[i]);
  }
  float l2[4][CH], l4[2][CH], l8[CH];
  u32x4 o2[4], o4[2], o8;
#pragma unroll
  for (int i = 0; i < 4; ++i) o2[i] = mean2<PT>(f[2 * i], f[2 * i + 1], l2[i]);
#pragma unroll
  for (int i = 0; i < 2; ++i) o4[i] = mean2<PT>(l2[2 * i], l2[2 * i + 1], l4[i]);
  o8 = mean2<PT>(l4[0], l4[1], l8);

  if (!CAP || live) {
    // pooled buffer: [level 2 | level 4 | level 8], each [B*H, npad/l, D] contiguous
    const int64_t D = (int64_t)p.D * ES;  // bytes per row
    char* d2 = p.dst[which];
    char* d4 = d2 + BH * (p.npad >> 1) * D;
    char* d8 = d4 + BH * (p.npad >> 2) * D;
    // streaming stores: the pooled rows are not read again by this kernel and would only push the inputs of the
    // next rows out of the caches (measured at the Wan2.1 shape: 70 -> 55 us)
#pragma unroll
    for (int i = 0; i < 4; ++i) __builtin_nontemporal_store(o2[i], (u32x4*)(d2 + ((int64_t)bh * (p.npad >> 1) + g * 4 + i) * D + c * 16));
#pragma unroll
    for (int i = 0; i < 2; ++i) __builtin_nontemporal_store(o4[i], (u32x4*)(d4 + ((int64_t)bh * (p.npad >> 2) + g * 2 + i) * D + c * 16));
    __builtin_nontemporal_store(o8, (u32x4*)(d8 + ((int64_t)bh * (p.npad >> 3) + g) * D + c * 16));
  }
  if constexpr (CAP) {
    if (which == 0) {  // uniform
      __shared__ float s_cos[3][32];
      float v[15];
      psa_ksim_row::pair_sums(f, v);
      psa_ksim_row::group_sums(v, chunks);
      const int gw = (int)threadIdx.x / chunks;  // token group inside the workgroup
      if (c == 0) psa_ksim_row::group_cosines(v, s_cos[0][gw], s_cos[1][gw], s_cos[2][gw]);
      __syncthreads();
      const int per = p.bn >> 3;  // token groups per kv-block
      if (live && c == 0 && gw % per == 0)
        p.cap[(int64_t)bh * (p.npad / p.bn) + g / per] = psa_ksim_row::block_cap(s_cos[0] + gw, s_cos[1] + gw, s_cos[2] + gw, p.bn, p.t2, p.t4, p.t8);
    }
  }
}

// Checks the arguments of a pooling pass and fills its parameters (psa_pool.hip).  cap, thresholds: null, or the similarity cap too.
int psa_pool_params(PoolParams& p, psa_tensor4 k, psa_tensor4 v, const int32_t* index, const psa_tensor4* k_ord, const psa_tensor4* v_ord,
                    void* k_pool, void* v_pool, int B, int Hkv, int L, int D, int block_n, int32_t* cap, const float* thresholds);
// The pooling kernel with the cap, bf16 rows, for parameters from there.
void psa_pool_launch_cap(const PoolParams& p, int nx, int heads, hipStream_t stream);
