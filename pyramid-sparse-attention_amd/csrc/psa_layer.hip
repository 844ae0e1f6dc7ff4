// The sparse layers as one library call each: every buffer carved from one workspace, every launch on one stream.  Host code
// only; the launches are those of the separate entry points, so the results are the same bits.  What it saves is the host's
// work per launch (argument conversion, allocations, stream and device look-ups of five to nine calls), which bounds small
// layers: 8 heads of 1000 tokens 82 -> 40 us, 2 fp32 heads of 4096 tokens 82 -> 57 us.
#include "psa_common.h"

// psa_level_map.hip
int psa_map_min_cap_heads(void* map, int map_elem_bytes, const int32_t* cap, int B, int Hq, int Hkv, int Mq, int Nk, psa_stream_t stream);

namespace {

// Consecutive parts of a workspace, 256-byte aligned.  What the estimate needs (gigabytes for long sequences of short blocks) is
// dead once the map exists: the parts of the stages behind it start where the estimate's do (reuse), in stream order.
struct Parts {
  int64_t at = 0, top = 0;
  int64_t take(int64_t bytes) {
    const int64_t off = at;
    at = (at + bytes + 255) & ~(int64_t)255;
    top = at > top ? at : top;
    return off;
  }
  void reuse(int64_t from) { at = from; }
};

// pools, walk (or row order) and attention of either layer
struct AttnParts {
  int64_t kp, vp, walk, order;
  bool has_walk;
};
void pool_parts(Parts& w, int elem, int B, int Hkv, int L, int D, int block_n, AttnParts& a) {
  const int64_t pool = psa_pool_elems(B, Hkv, L, D, block_n) * elem;
  a.kp = w.take(pool);
  a.vp = w.take(pool);
}
void walk_parts(Parts& w, int elem, int B, int Hq, int Hkv, int L, int D, int block_m, int block_n, int walk, AttnParts& a) {
  const int64_t walk_bytes = walk && elem == 2 ? psa_walk_bytes(B, Hq, Hkv, L, D, block_m, block_n) : 0;
  a.has_walk = walk_bytes > 0;
  a.walk = a.has_walk ? w.take(walk_bytes) : -1;
  a.order = a.has_walk ? -1 : w.take(psa_fwd_workspace_bytes(B, Hq, L, block_m));
}
int attn_run(const AttnParts& a, char* ws, psa_tensor4 q, const int32_t* index, psa_tensor4 k, psa_tensor4 v, const void* map, psa_tensor4 out,
             int B, int Hq, int Hkv, int L, int D, int block_m, int block_n, float sm_scale, int causal, psa_stream_t stream) {
  if (a.has_walk) {
    const int rc = psa_build_walk(map, 1, ws + a.walk, B, Hq, Hkv, L, D, block_m, block_n, causal, stream);
    if (rc != PSA_OK) return rc;
    return psa_fwd_walk(q, index, k, v, ws + a.kp, ws + a.vp, map, 1, ws + a.walk, out, nullptr, B, Hq, Hkv, L, D, block_m, block_n, sm_scale,
                        causal, stream);
  }
  if (index != nullptr)
    return psa_fwd_indexed(q, index, k, v, ws + a.kp, ws + a.vp, map, 1, out, nullptr, B, Hq, Hkv, L, D, block_m, block_n, sm_scale, causal,
                           ws + a.order, stream);
  return psa_fwd(q, k, v, ws + a.kp, ws + a.vp, map, 1, out, nullptr, B, Hq, Hkv, L, D, block_m, block_n, sm_scale, causal, ws + a.order, stream);
}

struct LayerParts {
  int64_t est, scores, k_ord, v_ord, bytes;
  AttnParts attn;
};
bool layer_parts(int elem, int B, int Hq, int Hkv, int L, int D, int block_m, int block_n, int indexed, int walk, LayerParts& p) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || L <= 0 || D <= 0 || block_m < 4 || block_n < 4 || (elem != 2 && elem != 4)) return false;
  const int64_t Mq = (L + block_m - 1) / block_m, Nk = (L + block_n - 1) / block_n;
  Parts w;
  const int64_t rows = indexed ? (int64_t)B * Hkv * L * D * elem : 0;
  p.k_ord = w.take(rows);
  p.v_ord = w.take(rows);
  if (indexed) pool_parts(w, elem, B, Hkv, L, D, block_n, p.attn);  // (filled with the ordered rows, before the estimate)
  const int64_t from = w.at;
  p.est = w.take(psa_estimate_workspace_bytes(B, Hq, L, L, block_m, block_n, block_m / 4, block_n / 4));
  p.scores = Nk > 4096 ? w.take((int64_t)B * Hq * Mq * Nk * 4) : -1;  // (maps too wide for the fused kernel's LDS)
  w.reuse(from);
  if (!indexed) pool_parts(w, elem, B, Hkv, L, D, block_n, p.attn);
  walk_parts(w, elem, B, Hq, Hkv, L, D, block_m, block_n, walk, p.attn);
  p.bytes = w.top;
  return true;
}

struct CausalParts {
  int64_t est, scores, map, cap, bytes;
  AttnParts attn;
};
bool causal_parts(int B, int Hq, int Hkv, int L, int D, int block, int stride, int chunk, CausalParts& p) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || L <= 0 || D <= 0 || block <= 0 || stride <= 0 || chunk <= 0) return false;
  const int64_t S = (L + block - 1) / block;
  Parts w;
  p.map = w.take((int64_t)B * Hq * S * S);
  p.cap = w.take((int64_t)B * Hkv * S * 4);
  const int64_t from = w.at;
  p.est = w.take(psa_estimate_xattn_workspace_bytes(B, Hq, L, L, block, stride, chunk));
  p.scores = w.take((int64_t)B * Hq * S * S * 4);
  w.reuse(from);
  pool_parts(w, 2, B, Hkv, L, D, block, p.attn);
  walk_parts(w, 2, B, Hq, Hkv, L, D, block, block, 1, p.attn);
  p.bytes = w.top;
  return true;
}

}  // namespace

extern "C" int64_t psa_layer_workspace_bytes(int elem_bytes, int B, int Hq, int Hkv, int L, int D, int block_m, int block_n, int indexed, int walk) {
  LayerParts p;
  return layer_parts(elem_bytes, B, Hq, Hkv, L, D, block_m, block_n, indexed, walk, p) ? p.bytes : 0;
}

extern "C" int psa_layer_fwd(psa_tensor4 q, psa_tensor4 k, psa_tensor4 v, const int32_t* token_index, const int32_t* off_q,
                             const int32_t* off_k, const float* sim_thresholds, int32_t* cap_out, void* workspace, void* map_out,
                             psa_tensor4 out, int B, int Hq, int Hkv, int L, int D, int block_m, int block_n, float sm_scale, int mode,
                             int n_items, const int32_t* item_level, const double* item_hi, int align_div, int text_blocks,
                             double min_full_attn_ratio, int walk, psa_stream_t stream) {
  PSA_REQUIRE(workspace != nullptr && map_out != nullptr, PSA_ERR_ARG, "psa_layer_fwd: null pointer");
  PSA_REQUIRE((uintptr_t)workspace % 256 == 0, PSA_ERR_ARG, "psa_layer_fwd: workspace must be 256-byte aligned");
  PSA_REQUIRE(sim_thresholds == nullptr || (cap_out != nullptr && Hq == Hkv), PSA_ERR_ARG, "psa_layer_fwd: the cap needs its buffer and as many kv heads as heads");
  LayerParts p;
  PSA_REQUIRE(layer_parts(q.dtype == PSA_DTYPE_F32 ? 4 : 2, B, Hq, Hkv, L, D, block_m, block_n, token_index != nullptr, walk, p), PSA_ERR_ARG,
              "psa_layer_fwd: bad shape");
  char* ws = (char*)workspace;
  const int Mq = (L + block_m - 1) / block_m, Nk = (L + block_n - 1) / block_n;
  int rc;
  if (token_index != nullptr) {
    psa_tensor4 ko = k, vo = v;
    ko.ptr = ws + p.k_ord;
    vo.ptr = ws + p.v_ord;
    ko.stride_l = vo.stride_l = D;
    ko.stride_h = vo.stride_h = (int64_t)L * D;
    ko.stride_b = vo.stride_b = (int64_t)Hkv * L * D;
    rc = psa_pool_kv_indexed(k, v, token_index, ko, vo, ws + p.attn.kp, ws + p.attn.vp, B, Hkv, L, D, block_n, stream);
    if (rc != PSA_OK) return rc;
    k = ko;
    v = vo;
  }
  if (sim_thresholds != nullptr) {
    rc = psa_ksim(k, cap_out, B, Hkv, L, D, block_n, sim_thresholds[0], sim_thresholds[1], sim_thresholds[2], stream);
    if (rc != PSA_OK) return rc;
  }
  float* scores = p.scores >= 0 ? (float*)(ws + p.scores) : nullptr;
  if (token_index != nullptr)
    rc = psa_estimate_sampled_map_indexed(q, token_index, k, off_q, off_k, scores, ws + p.est, B, Hq, Hkv, L, L, D, block_m, block_n, block_m / 4,
                                          block_n / 4, sm_scale, Mq, Nk, map_out, 1, mode, n_items, item_level, item_hi, align_div,
                                          text_blocks, min_full_attn_ratio, stream);
  else
    rc = psa_estimate_sampled_map(q, k, off_q, off_k, scores, ws + p.est, B, Hq, Hkv, L, L, D, block_m, block_n, block_m / 4, block_n / 4,
                                  sm_scale, Mq, Nk, map_out, 1, mode, n_items, item_level, item_hi, align_div, text_blocks,
                                  min_full_attn_ratio, stream);
  if (rc != PSA_OK) return rc;
  if (sim_thresholds != nullptr) {
    rc = psa_map_min_cap(map_out, 1, cap_out, (int64_t)B * Hq, Mq, Nk, stream);
    if (rc != PSA_OK) return rc;
  }
  if (token_index == nullptr) {
    rc = psa_pool_kv(k, v, ws + p.attn.kp, ws + p.attn.vp, B, Hkv, L, D, block_n, stream);
    if (rc != PSA_OK) return rc;
  }
  return attn_run(p.attn, ws, q, token_index, k, v, map_out, out, B, Hq, Hkv, L, D, block_m, block_n, sm_scale, 0, stream);
}

extern "C" int64_t psa_causal_layer_workspace_bytes(int B, int Hq, int Hkv, int L, int D, int block, int stride, int chunk) {
  CausalParts p;
  return causal_parts(B, Hq, Hkv, L, D, block, stride, chunk, p) ? p.bytes : 0;
}

extern "C" int psa_causal_layer_fwd(psa_tensor4 q, psa_tensor4 k, psa_tensor4 v, const float* sim_thresholds, void* workspace, psa_tensor4 out,
                                    int B, int Hq, int Hkv, int L, int D, int block, int stride, int chunk, float sm_scale, int mode,
                                    int n_items, const int32_t* item_level, const double* item_lo, const double* item_hi,
                                    int special_blocks, int causal, psa_stream_t stream) {
  PSA_REQUIRE(workspace != nullptr && sim_thresholds != nullptr, PSA_ERR_ARG, "psa_causal_layer_fwd: null pointer");
  PSA_REQUIRE((uintptr_t)workspace % 256 == 0, PSA_ERR_ARG, "psa_causal_layer_fwd: workspace must be 256-byte aligned");
  CausalParts p;
  PSA_REQUIRE(causal_parts(B, Hq, Hkv, L, D, block, stride, chunk, p), PSA_ERR_ARG, "psa_causal_layer_fwd: bad shape");
  char* ws = (char*)workspace;
  const int S = (L + block - 1) / block;
  int32_t* cap = (int32_t*)(ws + p.cap);
  int rc = psa_estimate_xattn(q, k, (float*)(ws + p.scores), ws + p.est, B, Hq, Hkv, L, L, D, block, stride, chunk, causal, stream);
  if (rc != PSA_OK) return rc;
  rc = psa_level_map_qwen((const float*)(ws + p.scores), ws + p.map, 1, (int64_t)B * Hq, S, mode, n_items, item_level, item_lo, item_hi,
                          special_blocks, causal, stream);
  if (rc != PSA_OK) return rc;
  rc = psa_ksim(k, cap, B, Hkv, L, D, block, sim_thresholds[0], sim_thresholds[1], sim_thresholds[2], stream);
  if (rc != PSA_OK) return rc;
  rc = psa_map_min_cap_heads(ws + p.map, 1, cap, B, Hq, Hkv, S, S, stream);
  if (rc != PSA_OK) return rc;
  rc = psa_pool_kv(k, v, ws + p.attn.kp, ws + p.attn.vp, B, Hkv, L, D, block, stream);
  if (rc != PSA_OK) return rc;
  return attn_run(p.attn, ws, q, nullptr, k, v, ws + p.map, out, B, Hq, Hkv, L, D, block, block, sm_scale, causal, stream);
}
