// The sparse layers as one library call each: every buffer carved from one workspace, every launch on one stream.  Host code
// only; the launches are those of the separate entry points, so the results are the same bits.  What it saves is the host's
// work per launch (argument conversion, allocations, stream and device look-ups of five to nine calls), which bounds small
// layers: 8 heads of 1000 tokens 82 -> 40 us, 2 fp32 heads of 4096 tokens 82 -> 57 us.
#include "psa_common.h"
#include "psa_pool_rows.h"
#include "psa_schedule.h"

// psa_level_map.hip
int psa_map_min_cap_heads(void* map, int map_elem_bytes, const int32_t* cap, int B, int Hq, int Hkv, int Mq, int Nk, psa_stream_t stream);
// psa_pool.hip
int psa_pool_kv_cap(psa_tensor4 k, psa_tensor4 v, const int32_t* index, const psa_tensor4* k_ord, const psa_tensor4* v_ord, void* k_pool,
                    void* v_pool, int32_t* cap, const float* thresholds, int B, int Hkv, int L, int D, int block_n, psa_stream_t stream);
// psa_estimate.hip, psa_xattn.hip
int psa_estimate_layer_map(psa_tensor4 q, psa_tensor4 k, const int32_t* off_q, const int32_t* off_k, const int32_t* q_index, float* scores,
                           void* workspace, int B, int Hq, int Hkv, int L, int D, int block_m, int block_n, float sm_scale, void* map_out, int mode,
                           int n_items, const int32_t* item_level, const double* item_hi, int align_div, int text_blocks,
                           double min_full_attn_ratio, const int32_t* cap, void* walk, bool* ended, const PoolParams* pool, psa_stream_t stream);
int psa_xattn_layer_map(psa_tensor4 q, psa_tensor4 k, psa_tensor4 v, void* workspace, void* k_pool, void* v_pool, int32_t* cap,
                        const float* thresholds, void* map, void* walk, int B, int Hq, int Hkv, int L, int D,
                        int block, int stride, int chunk, int mode, int n_items, const int32_t* item_level, const double* item_lo,
                        const double* item_hi, int special_blocks, int causal, psa_stream_t stream);

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
int attn_run(const AttnParts& a, char* ws, const void* kp, const void* vp, psa_tensor4 q, const int32_t* index, psa_tensor4 k, psa_tensor4 v, const void* map, psa_tensor4 out,
             int B, int Hq, int Hkv, int L, int D, int block_m, int block_n, float sm_scale, int causal, psa_stream_t stream) {
  if (a.has_walk) {
    const int rc = psa_build_walk(map, 1, ws + a.walk, B, Hq, Hkv, L, D, block_m, block_n, causal, stream);
    if (rc != PSA_OK) return rc;
    return psa_fwd_walk(q, index, k, v, kp, vp, map, 1, ws + a.walk, out, nullptr, B, Hq, Hkv, L, D, block_m, block_n, sm_scale,
                        causal, stream);
  }
  if (index != nullptr)
    return psa_fwd_indexed(q, index, k, v, kp, vp, map, 1, out, nullptr, B, Hq, Hkv, L, D, block_m, block_n, sm_scale, causal,
                           ws + a.order, stream);
  return psa_fwd(q, k, v, kp, vp, map, 1, out, nullptr, B, Hq, Hkv, L, D, block_m, block_n, sm_scale, causal, ws + a.order, stream);
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

namespace {
// What a layer may have beside its workspace, whose parts overlap in time: buffers that are filled while the estimate's scratch is
// still in use.  They let the level map's kernel write the tile records and the pooling pass form the similarity cap.  Pools that no
// cap is formed beside (capped == 0; token re-ordering, whose pools come first anyway) stay in the workspace: a layer of 12 heads x 32760 tokens
// takes 24 MiB here instead of 192.
struct LayerExtra {
  int64_t kp, vp, walk, bytes;
};
LayerExtra layer_extra(int elem, int B, int Hq, int Hkv, int L, int D, int block_m, int block_n, int indexed, int walk, bool capped) {
  LayerExtra e = {-1, -1, -1, 0};
  Parts w;
  const int64_t walk_bytes = walk && elem == 2 ? psa_walk_bytes(B, Hq, Hkv, L, D, block_m, block_n) : 0;
  if (walk_bytes > 0) e.walk = w.take(walk_bytes);
  if (capped && !indexed) {
    const int64_t pool = psa_pool_elems(B, Hkv, L, D, block_n) * elem;
    e.kp = w.take(pool);
    e.vp = w.take(pool);
  }
  e.bytes = w.top;
  return e;
}

// Layers whose pooling pass runs in the launch of the estimate's contraction (psa_estimate.hip) instead of one of its own: up to 32 MiB of K
// and V, 24 in fp32.  Such a launch is short, and its start and end are what it costs (a pass, us, before and after):
//   bf16  8 heads x 1000 x 64   41.0  38.4     24 x 5000 x 64   74.7  69.5     12 x 5400 x 128  95.8  90.5     8 x 8192 x 128  121.6 120.7
//   fp32  2 x 4096 x 64         56.5  52.7     4 x 6000 x 64   157.2 152.8     8 x 6000 x 64   223.8 217.1     8 x 8000 x 64   284.8 290.2
// Larger ones of 16 bits have the pass on a stream of its own.
bool pools_beside(int elem, int B, int Hkv, int L, int D) {
  return (int64_t)B * Hkv * L * D * elem * 2 <= (int64_t)(elem == 4 ? 24 : 32) << 20;
}
// The output as the estimate's scratch, which ends before the output is written: large enough, aligned, without gaps, and apart from the
// rows that are still to be read.  (In the workspace the scratch lies where the pools go.)
bool overlaps(const psa_tensor4& out, int64_t out_bytes, const psa_tensor4& t, int elem, int B, int H, int L, int D) {
  if (t.stride_b < 0 || t.stride_h < 0 || t.stride_l < 0) return true;
  const int64_t bytes = ((B - 1) * t.stride_b + (H - 1) * t.stride_h + (L - 1) * t.stride_l + D) * elem;
  const uintptr_t o = (uintptr_t)out.ptr, a = (uintptr_t)t.ptr;
  return o < a + (uintptr_t)bytes && a < o + (uintptr_t)out_bytes;
}
bool output_takes_scratch(const psa_tensor4& out, const psa_tensor4& q, const psa_tensor4& k, const psa_tensor4& v, int64_t scratch, int elem, int B,
                          int Hq, int Hkv, int L, int D) {
  const int64_t bytes = (int64_t)B * Hq * L * D * elem;
  const bool dense = (L == 1 || out.stride_l == D) && (Hq == 1 || out.stride_h == (int64_t)L * D) && (B == 1 || out.stride_b == (int64_t)Hq * L * D);
  return out.ptr != nullptr && (uintptr_t)out.ptr % 256 == 0 && dense && scratch <= bytes && !overlaps(out, bytes, q, elem, B, Hq, L, D) &&
         !overlaps(out, bytes, k, elem, B, Hkv, L, D) && !overlaps(out, bytes, v, elem, B, Hkv, L, D);
}
}  // namespace

extern "C" int64_t psa_layer_extra_bytes(int elem_bytes, int B, int Hq, int Hkv, int L, int D, int block_m, int block_n, int indexed, int walk) {
  LayerParts p;
  if (!layer_parts(elem_bytes, B, Hq, Hkv, L, D, block_m, block_n, indexed, walk, p)) return 0;
  return layer_extra(elem_bytes, B, Hq, Hkv, L, D, block_m, block_n, indexed, walk, true).bytes;
}

extern "C" int psa_layer_fwd(psa_tensor4 q, psa_tensor4 k, psa_tensor4 v, const int32_t* token_index, const int32_t* off_q,
                             const int32_t* off_k, const float* sim_thresholds, int32_t* cap_out, void* workspace, void* map_out,
                             psa_tensor4 out, int B, int Hq, int Hkv, int L, int D, int block_m, int block_n, float sm_scale, int mode,
                             int n_items, const int32_t* item_level, const double* item_hi, int align_div, int text_blocks,
                             double min_full_attn_ratio, int walk, psa_stream_t stream) {
  return psa_layer_fwd_extra(q, k, v, token_index, off_q, off_k, sim_thresholds, cap_out, workspace, nullptr, map_out, out, B, Hq, Hkv, L, D,
                             block_m, block_n, sm_scale, mode, n_items, item_level, item_hi, align_div, text_blocks, min_full_attn_ratio, walk,
                             stream);
}

extern "C" int psa_layer_fwd_extra(psa_tensor4 q, psa_tensor4 k, psa_tensor4 v, const int32_t* token_index, const int32_t* off_q,
                                   const int32_t* off_k, const float* sim_thresholds, int32_t* cap_out, void* workspace, void* extra,
                                   void* map_out, psa_tensor4 out, int B, int Hq, int Hkv, int L, int D, int block_m, int block_n,
                                   float sm_scale, int mode, int n_items, const int32_t* item_level, const double* item_hi, int align_div,
                                   int text_blocks, double min_full_attn_ratio, int walk, psa_stream_t stream) {
  PSA_REQUIRE(workspace != nullptr && map_out != nullptr, PSA_ERR_ARG, "psa_layer_fwd: null pointer");
  PSA_REQUIRE((uintptr_t)workspace % 256 == 0 && (uintptr_t)extra % 256 == 0, PSA_ERR_ARG, "psa_layer_fwd: workspace must be 256-byte aligned");
  PSA_REQUIRE(sim_thresholds == nullptr || (cap_out != nullptr && Hq == Hkv), PSA_ERR_ARG, "psa_layer_fwd: the cap needs its buffer and as many kv heads as heads");
  const int elem = q.dtype == PSA_DTYPE_F32 ? 4 : 2;
  LayerParts p;
  PSA_REQUIRE(layer_parts(elem, B, Hq, Hkv, L, D, block_m, block_n, token_index != nullptr, walk, p), PSA_ERR_ARG, "psa_layer_fwd: bad shape");
  LayerExtra e = {-1, -1, -1, 0};
  if (extra != nullptr) e = layer_extra(elem, B, Hq, Hkv, L, D, block_m, block_n, token_index != nullptr, walk, sim_thresholds != nullptr);
  char *ws = (char*)workspace, *ex = (char*)extra;
  char* kp = e.kp >= 0 ? ex + e.kp : ws + p.attn.kp;
  char* vp = e.vp >= 0 ? ex + e.vp : ws + p.attn.vp;
  void* const listed = e.walk >= 0 ? ex + e.walk : nullptr;  // the walk, where the map's kernel writes its records
  const int Mq = (L + block_m - 1) / block_m, Nk = (L + block_n - 1) / block_n;
  bool pooled = false, capped = false, beside = false;
  PoolParams pool;
  char* est_at = ws + p.est;  // the estimate's scratch
  int rc;
  if (token_index != nullptr) {
    psa_tensor4 ko = k, vo = v;
    ko.ptr = ws + p.k_ord;
    vo.ptr = ws + p.v_ord;
    ko.stride_l = vo.stride_l = D;
    ko.stride_h = vo.stride_h = (int64_t)L * D;
    ko.stride_b = vo.stride_b = (int64_t)Hkv * L * D;
    capped = pooled = true;
    if (sim_thresholds != nullptr)
      rc = psa_pool_kv_cap(k, v, token_index, &ko, &vo, kp, vp, cap_out, sim_thresholds, B, Hkv, L, D, block_n, stream);
    else
      rc = psa_pool_kv_indexed(k, v, token_index, ko, vo, kp, vp, B, Hkv, L, D, block_n, stream);
    if (rc != PSA_OK) return rc;
    k = ko;
    v = vo;
  } else if (sim_thresholds != nullptr && extra != nullptr) {
    beside = pools_beside(elem, B, Hkv, L, D);
    rc = beside ? psa_pool_params(pool, k, v, nullptr, nullptr, nullptr, kp, vp, B, Hkv, L, D, block_n, cap_out, sim_thresholds)
                : psa_pool_kv_cap(k, v, nullptr, nullptr, nullptr, kp, vp, cap_out, sim_thresholds, B, Hkv, L, D, block_n, stream);
    if (rc != PSA_OK) return rc;
    capped = pooled = true;
  } else if (p.scores < 0 && pools_beside(elem, B, Hkv, L, D)) {
    const int64_t scratch = psa_estimate_workspace_bytes(B, Hq, L, L, block_m, block_n, block_m / 4, block_n / 4);
    if (output_takes_scratch(out, q, k, v, scratch, elem, B, Hq, Hkv, L, D)) {
      rc = psa_pool_params(pool, k, v, nullptr, nullptr, nullptr, kp, vp, B, Hkv, L, D, block_n, nullptr, nullptr);
      if (rc != PSA_OK) return rc;
      est_at = (char*)out.ptr;
      pooled = beside = true;
    }
  }
  if (sim_thresholds != nullptr && !capped) {
    rc = psa_ksim(k, cap_out, B, Hkv, L, D, block_n, sim_thresholds[0], sim_thresholds[1], sim_thresholds[2], stream);
    if (rc != PSA_OK) return rc;
  }
  bool ended = false;
  rc = psa_estimate_layer_map(q, k, off_q, off_k, token_index, p.scores >= 0 ? (float*)(ws + p.scores) : nullptr, est_at, B, Hq, Hkv, L, D, block_m,
                              block_n, sm_scale, map_out, mode, n_items, item_level, item_hi, align_div, text_blocks, min_full_attn_ratio,
                              sim_thresholds != nullptr ? cap_out : nullptr, listed, &ended, beside ? &pool : nullptr, stream);
  if (rc != PSA_OK) return rc;
  if (sim_thresholds != nullptr && !ended) {
    rc = psa_map_min_cap(map_out, 1, cap_out, (int64_t)B * Hq, Mq, Nk, stream);
    if (rc != PSA_OK) return rc;
  }
  if (!pooled) {
    rc = psa_pool_kv(k, v, kp, vp, B, Hkv, L, D, block_n, stream);
    if (rc != PSA_OK) return rc;
  }
  if (ended && listed != nullptr) {
    psa_sched::Geometry g;
    PSA_REQUIRE(psa_schedule_geometry(B, Hq, Hkv, L, D, block_m, block_n, g), PSA_ERR_UNSUPPORTED, "psa_build_schedule: shape out of range");
    rc = psa_walk_order(listed, g, stream);
    if (rc != PSA_OK) return rc;
    return psa_fwd_walk(q, token_index, k, v, kp, vp, map_out, 1, listed, out, nullptr, B, Hq, Hkv, L, D, block_m, block_n, sm_scale, 0, stream);
  }
  return attn_run(p.attn, ws, kp, vp, q, token_index, k, v, map_out, out, B, Hq, Hkv, L, D, block_m, block_n, sm_scale, 0, stream);
}

extern "C" int psa_estimate_walk(psa_tensor4 q, psa_tensor4 k, const int32_t* off_q, const int32_t* off_k, const int32_t* token_index,
                                 const int32_t* cap, float* scores, void* workspace, void* map_out, void* walk, int B, int Hq, int Hkv, int L, int D,
                                 int block_m, int block_n, float sm_scale, int mode, int n_items, const int32_t* item_level,
                                 const double* item_hi, int align_div, int text_blocks, double min_full_attn_ratio, psa_stream_t stream) {
  psa_sched::Geometry g;
  PSA_REQUIRE(walk != nullptr && (uintptr_t)walk % 16 == 0, PSA_ERR_ARG, "psa_estimate_walk: walk must be 16-byte aligned");
  PSA_REQUIRE(psa_schedule_geometry(B, Hq, Hkv, L, D, block_m, block_n, g), PSA_ERR_UNSUPPORTED, "psa_estimate_walk: shape out of range");
  bool ended = false;
  int rc = psa_estimate_layer_map(q, k, off_q, off_k, token_index, scores, workspace, B, Hq, Hkv, L, D, block_m, block_n, sm_scale, map_out, mode,
                                  n_items, item_level, item_hi, align_div, text_blocks, min_full_attn_ratio, cap, walk, &ended, nullptr, stream);
  if (rc != PSA_OK) return rc;
  if (ended) return psa_walk_order(walk, g, stream);
  if (cap != nullptr) {
    rc = psa_map_min_cap(map_out, 1, cap, (int64_t)B * Hq, g.Mq, g.Nk, stream);
    if (rc != PSA_OK) return rc;
  }
  return psa_build_walk(map_out, 1, walk, B, Hq, Hkv, L, D, block_m, block_n, 0, stream);
}

extern "C" int64_t psa_causal_layer_workspace_bytes(int B, int Hq, int Hkv, int L, int D, int block, int stride, int chunk) {
  CausalParts p;
  return causal_parts(B, Hq, Hkv, L, D, block, stride, chunk, p) ? p.bytes : 0;
}

namespace {
struct CausalExtra {
  int64_t kp, vp, walk, bytes;
};
CausalExtra causal_extra(int B, int Hq, int Hkv, int L, int D, int block) {
  CausalExtra e;
  Parts w;
  const int64_t pool = psa_pool_elems(B, Hkv, L, D, block) * 2;
  e.kp = w.take(pool);
  e.vp = w.take(pool);
  const int64_t walk = psa_walk_bytes(B, Hq, Hkv, L, D, block, block);
  e.walk = walk > 0 ? w.take(walk) : -1;
  e.bytes = w.top;
  return e;
}
}  // namespace

extern "C" int64_t psa_causal_layer_extra_bytes(int B, int Hq, int Hkv, int L, int D, int block, int stride, int chunk) {
  CausalParts p;
  return causal_parts(B, Hq, Hkv, L, D, block, stride, chunk, p) ? causal_extra(B, Hq, Hkv, L, D, block).bytes : 0;
}

extern "C" int psa_causal_layer_fwd(psa_tensor4 q, psa_tensor4 k, psa_tensor4 v, const float* sim_thresholds, void* workspace, psa_tensor4 out,
                                    int B, int Hq, int Hkv, int L, int D, int block, int stride, int chunk, float sm_scale, int mode,
                                    int n_items, const int32_t* item_level, const double* item_lo, const double* item_hi,
                                    int special_blocks, int causal, psa_stream_t stream) {
  return psa_causal_layer_fwd_extra(q, k, v, sim_thresholds, workspace, nullptr, out, B, Hq, Hkv, L, D, block, stride, chunk, sm_scale, mode, n_items,
                                    item_level, item_lo, item_hi, special_blocks, causal, stream);
}

extern "C" int psa_causal_layer_fwd_extra(psa_tensor4 q, psa_tensor4 k, psa_tensor4 v, const float* sim_thresholds, void* workspace, void* extra,
                                          psa_tensor4 out, int B, int Hq, int Hkv, int L, int D, int block, int stride, int chunk,
                                          float sm_scale, int mode, int n_items, const int32_t* item_level, const double* item_lo,
                                          const double* item_hi, int special_blocks, int causal, psa_stream_t stream) {
  PSA_REQUIRE(workspace != nullptr && sim_thresholds != nullptr, PSA_ERR_ARG, "psa_causal_layer_fwd: null pointer");
  PSA_REQUIRE((uintptr_t)workspace % 256 == 0 && (uintptr_t)extra % 256 == 0, PSA_ERR_ARG, "psa_causal_layer_fwd: workspace must be 256-byte aligned");
  CausalParts p;
  PSA_REQUIRE(causal_parts(B, Hq, Hkv, L, D, block, stride, chunk, p), PSA_ERR_ARG, "psa_causal_layer_fwd: bad shape");
  char* ws = (char*)workspace;
  const int S = (L + block - 1) / block;
  int32_t* cap = (int32_t*)(ws + p.cap);
  void* const map = ws + p.map;
  int rc;
  // (a row's scores, levels and sorting scratch take 25 to 33 bytes of LDS per column: 100 KiB at 4096 columns, 132 just above, and from 5800 on
  // they do not fit together)
  if (extra != nullptr && S <= 4096) {
    const CausalExtra e = causal_extra(B, Hq, Hkv, L, D, block);
    char* ex = (char*)extra;
    void *kp = ex + e.kp, *vp = ex + e.vp, *walk = e.walk >= 0 ? ex + e.walk : nullptr;
    rc = psa_xattn_layer_map(q, k, v, ws + p.est, kp, vp, cap, sim_thresholds, map, walk, B, Hq, Hkv, L, D, block, stride, chunk, mode, n_items,
                             item_level, item_lo, item_hi, special_blocks, causal, stream);
    if (rc != PSA_OK) return rc;
    if (walk != nullptr) {
      psa_sched::Geometry g;
      PSA_REQUIRE(psa_schedule_geometry(B, Hq, Hkv, L, D, block, block, g), PSA_ERR_UNSUPPORTED, "psa_build_schedule: shape out of range");
      rc = psa_walk_order(walk, g, stream);
      if (rc != PSA_OK) return rc;
      return psa_fwd_walk(q, nullptr, k, v, kp, vp, map, 1, walk, out, nullptr, B, Hq, Hkv, L, D, block, block, sm_scale, causal, stream);
    }
    return attn_run(p.attn, ws, kp, vp, q, nullptr, k, v, map, out, B, Hq, Hkv, L, D, block, block, sm_scale, causal, stream);
  }
  rc = psa_estimate_xattn(q, k, (float*)(ws + p.scores), ws + p.est, B, Hq, Hkv, L, L, D, block, stride, chunk, causal, stream);
  if (rc != PSA_OK) return rc;
  rc = psa_level_map_qwen((const float*)(ws + p.scores), map, 1, (int64_t)B * Hq, S, mode, n_items, item_level, item_lo, item_hi,
                          special_blocks, causal, stream);
  if (rc != PSA_OK) return rc;
  rc = psa_ksim(k, cap, B, Hkv, L, D, block, sim_thresholds[0], sim_thresholds[1], sim_thresholds[2], stream);
  if (rc != PSA_OK) return rc;
  rc = psa_map_min_cap_heads(map, 1, cap, B, Hq, Hkv, S, S, stream);
  if (rc != PSA_OK) return rc;
  rc = psa_pool_kv(k, v, ws + p.attn.kp, ws + p.attn.vp, B, Hkv, L, D, block, stream);
  if (rc != PSA_OK) return rc;
  return attn_run(p.attn, ws, ws + p.attn.kp, ws + p.attn.vp, q, nullptr, k, v, map, out, B, Hq, Hkv, L, D, block, block, sm_scale, causal, stream);
}
