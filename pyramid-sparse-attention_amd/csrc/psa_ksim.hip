// Key-similarity cap ("sim mask"): per kv-block, the mean cosine similarity of token pairs at
// distance 1, 3 and 7 inside aligned groups of 2, 4 and 8 tokens decides up to which level the
// block's keys may be pooled.
//
// HBM-bound: one pass over K.  A workgroup owns one kv-block; a thread owns 8 consecutive tokens x 8
// channels (16-byte loads, D/8 lanes per row), forms the partial dot products and squared norms of
// its channels, and the D/8 lanes of a token group reduce them with butterflies.
#include "psa_common.h"
#include "psa_ksim_row.h"

namespace {

struct KsimParams {
  const uint16_t* k;  // bf16 or fp16
  int64_t sb, sh, sl;
  int32_t* out;
  int H, L, D, bn, Nk;
  float t2, t4, t8;
};

template <class ET>
__global__ __launch_bounds__(256) void psa_ksim_kernel(KsimParams p) {
  __shared__ float s_part[3][16];
  const int lpr = p.D >> 3;
  const int J = blockIdx.x, bh = blockIdx.y, b = bh / p.H, h = bh % p.H;
  const int g = threadIdx.x / lpr, c = threadIdx.x % lpr;
  const uint16_t* src = p.k + b * p.sb + h * p.sh + c * 8;
  float f[8][8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    int64_t row = (int64_t)J * p.bn + g * 8 + i;
    row = row < p.L ? row : (int64_t)(p.L - 1);  // replicate padding
    const u32x4 w = *(const u32x4*)(src + row * p.sl);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f[i][2 * j] = ET::from_bits(w[j] & 0xffffu);
      f[i][2 * j + 1] = ET::from_bits(w[j] >> 16);
    }
  }
  float v[15];
  psa_ksim_row::pair_sums(f, v);
  psa_ksim_row::group_sums(v, lpr);
  if (c == 0) psa_ksim_row::group_cosines(v, s_part[0][g], s_part[1][g], s_part[2][g]);
  __syncthreads();
  if (threadIdx.x == 0) p.out[(int64_t)bh * p.Nk + J] = psa_ksim_row::block_cap(s_part[0], s_part[1], s_part[2], p.bn, p.t2, p.t4, p.t8);
}

}  // namespace

extern "C" int psa_ksim(psa_tensor4 k, int32_t* cap_out, int B, int H, int L, int D, int block_n, float thr2, float thr4,
                        float thr8, psa_stream_t stream) {
  PSA_REQUIRE(k.ptr && cap_out, PSA_ERR_ARG, "psa_ksim: null pointer");
  PSA_REQUIRE(B > 0 && H > 0 && L > 0, PSA_ERR_ARG, "psa_ksim: B, H, L must be positive");
  PSA_REQUIRE(D == 64 || D == 128, PSA_ERR_UNSUPPORTED, "psa_ksim: head dim %d not in {64, 128}", D);
  PSA_REQUIRE(block_n == 32 || block_n == 64 || block_n == 128, PSA_ERR_UNSUPPORTED, "psa_ksim: block_n=%d not in {32, 64, 128}", block_n);
  PSA_REQUIRE((int64_t)B * H <= 65535, PSA_ERR_UNSUPPORTED, "psa_ksim: B*H too large");
  PSA_REQUIRE(((uintptr_t)k.ptr % 16 == 0) && k.stride_b % 8 == 0 && k.stride_h % 8 == 0 && k.stride_l % 8 == 0, PSA_ERR_UNSUPPORTED,
              "psa_ksim: K must be 16-byte aligned with strides that are multiples of 8 elements");
  KsimParams p;
  p.k = (const uint16_t*)k.ptr; p.sb = k.stride_b; p.sh = k.stride_h; p.sl = k.stride_l;
  p.out = cap_out; p.H = H; p.L = L; p.D = D; p.bn = block_n; p.Nk = (L + block_n - 1) / block_n;
  p.t2 = thr2; p.t4 = thr4; p.t8 = thr8;
  const bool known = psa_dispatch16(k.dtype, [&](auto et) {
    hipLaunchKernelGGL(psa_ksim_kernel<decltype(et)>, dim3((unsigned)p.Nk, (unsigned)(B * H)), dim3((unsigned)((block_n / 8) * (D / 8))), 0,
                       (hipStream_t)stream, p);
  });
  PSA_REQUIRE(known, PSA_ERR_UNSUPPORTED, "psa_ksim: bf16 or fp16 keys only");
  return psa_check_launch("psa_ksim");
}
