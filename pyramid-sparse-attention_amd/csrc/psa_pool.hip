// Pyramid pooling of K and V: one pass over the inputs writes the 2x, 4x and 8x mean-pooled levels.
//
// HBM-bound.  Every thread owns 8 consecutive tokens x 16 bytes of channels (one 16-byte load per token: 8 channels
// of bf16 / fp16, 4 of fp32), so a group of neighbouring lanes reads whole rows; the three levels are reduced in
// registers and each level is rounded to the tensors' element type before it feeds the next (the reference
// materialises every level in that type).
// Rows past L replicate row L-1 (replicate padding to a multiple of block_n).
//
// Indexed form (token re-ordering fused into the pass): position i of the sequence that is pooled is source row
// index[i]; the re-ordered rows themselves are written out as well (the level-1 keys / values of the attention
// kernel), so no separate gather pass over K and V is needed.
//
// With a similarity cap (layers in one call) the workgroups of K form the cap of their kv-blocks from the rows that they hold
// anyway: the pass over K of psa_ksim.hip and its launch go (12 heads x 32760 tokens with re-ordering 112 + 21 -> 123 us, 4 heads x 32768
// without 22 + 10 -> 23).
#include "psa_pool_rows.h"

template <bool INDEXED, bool CAP, class PT>
__global__ __launch_bounds__(256) void psa_pool_kernel(PoolParams p) {
  pool_rows<INDEXED, CAP, PT>(p, (int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z, (int64_t)gridDim.y);
}

int psa_pool_params(PoolParams& p, psa_tensor4 k, psa_tensor4 v, const int32_t* index, const psa_tensor4* k_ord, const psa_tensor4* v_ord,
                    void* k_pool, void* v_pool, int B, int Hkv, int L, int D, int block_n, int32_t* cap, const float* thresholds) {
  PSA_REQUIRE(k.ptr && v.ptr && k_pool && v_pool, PSA_ERR_ARG, "psa_pool_kv: null pointer");
  PSA_REQUIRE(B > 0 && Hkv > 0 && L > 0, PSA_ERR_ARG, "psa_pool_kv: B, Hkv, L must be positive");
  PSA_REQUIRE(D > 0 && D % 8 == 0 && D <= 256, PSA_ERR_UNSUPPORTED, "psa_pool_kv: D=%d must be a multiple of 8, <= 256", D);
  PSA_REQUIRE(block_n >= 8 && block_n % 8 == 0, PSA_ERR_UNSUPPORTED, "psa_pool_kv: block_n=%d must be a multiple of 8", block_n);
  PSA_REQUIRE((int64_t)B * Hkv <= 65535, PSA_ERR_UNSUPPORTED, "psa_pool_kv: B*Hkv too large");
  PSA_REQUIRE(k.stride_l % 8 == 0 && v.stride_l % 8 == 0 && k.stride_h % 8 == 0 && v.stride_h % 8 == 0 &&
                  k.stride_b % 8 == 0 && v.stride_b % 8 == 0 && ((uintptr_t)k.ptr % 16 == 0) && ((uintptr_t)v.ptr % 16 == 0),
              PSA_ERR_UNSUPPORTED, "psa_pool_kv: inputs must be 16-byte aligned with strides that are multiples of 8");
  PSA_REQUIRE(k.dtype == v.dtype && (k.dtype == PSA_DTYPE_BF16 || k.dtype == PSA_DTYPE_F16 || k.dtype == PSA_DTYPE_F32), PSA_ERR_ARG,
              "psa_pool_kv: K and V must share one element type (bf16, fp16 or fp32)");
  p.src[0] = (const char*)k.ptr;
  p.src[1] = (const char*)v.ptr;
  p.sb[0] = k.stride_b; p.sh[0] = k.stride_h; p.sl[0] = k.stride_l;
  p.sb[1] = v.stride_b; p.sh[1] = v.stride_h; p.sl[1] = v.stride_l;
  p.dst[0] = (char*)k_pool;
  p.dst[1] = (char*)v_pool;
  p.H = Hkv; p.L = L; p.D = D;
  p.npad = (int64_t)((L + block_n - 1) / block_n) * block_n;
  p.index = index;
  p.ord[0] = p.ord[1] = nullptr;
  p.ob[0] = p.ob[1] = p.oh[0] = p.oh[1] = p.ol[0] = p.ol[1] = 0;
  if (index != nullptr) {
    const psa_tensor4* o[2] = {k_ord, v_ord};
    for (int t = 0; t < 2; ++t) {
      PSA_REQUIRE(o[t] && o[t]->ptr && ((uintptr_t)o[t]->ptr % 16 == 0) && o[t]->stride_l % 8 == 0 && o[t]->stride_h % 8 == 0 &&
                      o[t]->stride_b % 8 == 0,
                  PSA_ERR_ARG, "psa_pool_kv_indexed: the re-ordered outputs must be 16-byte aligned with strides that are multiples of 8");
      PSA_REQUIRE(o[t]->dtype == k.dtype, PSA_ERR_ARG, "psa_pool_kv_indexed: the re-ordered outputs must have the inputs' element type");
      p.ord[t] = (char*)o[t]->ptr;
      p.ob[t] = o[t]->stride_b; p.oh[t] = o[t]->stride_h; p.ol[t] = o[t]->stride_l;
    }
  }
  p.cap = cap;
  p.bn = block_n;
  p.t2 = p.t4 = p.t8 = 0.f;
  if (cap != nullptr) {
    // (a kv-block's threads, D / 8 * block_n / 8 of them, divide a workgroup)
    PSA_REQUIRE((D == 64 || D == 128) && (block_n == 32 || block_n == 64 || block_n == 128), PSA_ERR_UNSUPPORTED,
                "psa_ksim: D=%d, block_n=%d", D, block_n);
    PSA_REQUIRE(k.dtype != PSA_DTYPE_F32, PSA_ERR_UNSUPPORTED, "psa_ksim: bf16 or fp16 keys only");
    p.t2 = thresholds[0]; p.t4 = thresholds[1]; p.t8 = thresholds[2];
  }
  return PSA_OK;
}

static int pool_run(psa_tensor4 k, psa_tensor4 v, const int32_t* index, const psa_tensor4* k_ord, const psa_tensor4* v_ord,
                    void* k_pool, void* v_pool, int B, int Hkv, int L, int D, int block_n, psa_stream_t stream, int32_t* cap = nullptr,
                    const float* thresholds = nullptr) {
  PoolParams p;
  const int rc = psa_pool_params(p, k, v, index, k_ord, v_ord, k_pool, v_pool, B, Hkv, L, D, block_n, cap, thresholds);
  if (rc != PSA_OK) return rc;
  auto launch = [&](auto pt) {
    using PT = decltype(pt);
    const int64_t units = (p.npad / 8) * (D / PT::CH);
    dim3 grid((unsigned)((units + 255) / 256), (unsigned)(B * Hkv), 2);
    auto kernel = index != nullptr ? psa_pool_kernel<true, false, PT> : psa_pool_kernel<false, false, PT>;
    if constexpr (PT::ES == 2) {
      if (cap != nullptr) kernel = index != nullptr ? psa_pool_kernel<true, true, PT> : psa_pool_kernel<false, true, PT>;
    }
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, (hipStream_t)stream, p);
  };
  if (k.dtype == PSA_DTYPE_F32) launch(PoolF32{});
  else if (k.dtype == PSA_DTYPE_F16) launch(Pool16<EtF16>{});
  else launch(Pool16<EtBf16>{});
  return psa_check_launch("psa_pool_kv");
}

void psa_pool_launch_cap(const PoolParams& p, int nx, int heads, hipStream_t stream) {
  hipLaunchKernelGGL((psa_pool_kernel<false, true, Pool16<EtBf16>>), dim3((unsigned)nx, (unsigned)heads, 2), dim3(256), 0, stream, p);
}

// psa_pool_kv[_indexed] and, of the rows in the order in which they are pooled, psa_ksim (thresholds t2, t4, t8), in one pass
int psa_pool_kv_cap(psa_tensor4 k, psa_tensor4 v, const int32_t* index, const psa_tensor4* k_ord, const psa_tensor4* v_ord, void* k_pool,
                    void* v_pool, int32_t* cap, const float* thresholds, int B, int Hkv, int L, int D, int block_n, psa_stream_t stream) {
  PSA_REQUIRE(cap != nullptr && thresholds != nullptr, PSA_ERR_ARG, "psa_pool_kv_cap: null pointer");
  return pool_run(k, v, index, k_ord, v_ord, k_pool, v_pool, B, Hkv, L, D, block_n, stream, cap, thresholds);
}

extern "C" int psa_pool_kv(psa_tensor4 k, psa_tensor4 v, void* k_pool, void* v_pool, int B, int Hkv, int L, int D,
                           int block_n, psa_stream_t stream) {
  return pool_run(k, v, nullptr, nullptr, nullptr, k_pool, v_pool, B, Hkv, L, D, block_n, stream);
}

extern "C" int psa_pool_kv_indexed(psa_tensor4 k, psa_tensor4 v, const int32_t* index, psa_tensor4 k_ord, psa_tensor4 v_ord,
                                   void* k_pool, void* v_pool, int B, int Hkv, int L, int D, int block_n, psa_stream_t stream) {
  PSA_REQUIRE(index != nullptr, PSA_ERR_ARG, "psa_pool_kv_indexed: null index");
  return pool_run(k, v, index, &k_ord, &v_ord, k_pool, v_pool, B, Hkv, L, D, block_n, stream);
}
