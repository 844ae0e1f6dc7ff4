// Pyramid sparse attention forward on fp32 tensors: fp32 operands and fp32 arithmetic throughout, products on the matrix
// cores' fp32 instruction (v_mfma_f32_16x16x4_f32: a k-ordered chain of fp32 multiply-adds).  Same walk as the 16-bit kernels
// (psa_tiles.h: the map row is compacted into tiles of 64 pooled keys of one level), same softmax (base 2, +log2(level)
// bias, online), same masks.
//
// One workgroup of 4 waves per QR = 64 / KS query rows; the K and V tile goes straight into LDS and is shared by the waves:
// wave w works on row group w / KS (16 rows) and the w % KS -th share of the tile's four 16-key blocks, with a softmax state
// of its own; the KS shares of a row meet once, at the end.  KS = 1, 2 or 4: the smallest that still gives the launch two
// workgroups per CU (the small layers this path serves have few rows: 2 heads of 4096 tokens are 128 q-blocks of 64).
// The transposed products S^T = K Q^T and O^T += V^T P^T leave a lane 4 keys of one query in the accumulator, and with
// k-index g of the i-th PV step taken to be key 4 g + i that register IS the step's B operand: nothing crosses lanes
// between the two products, and a row maximum is two lane exchanges.  Channels are dealt so that a lane's operands of four
// steps are 16 consecutive bytes (one ds_read_b128); rows are XOR-swizzled by 16-byte chunks: conflict-free.
// 2 heads of 4096 tokens x 64, 64-key blocks, 80 % sparse: 109 us on the vector units (two LDS operands per 4 FMAs), 36 us here.
#include <type_traits>

#include "psa_common.h"
#include "psa_tiles.h"

namespace {

constexpr int TK32 = 64;

// V rows of slots that hold no key: their probabilities are 0, which only a finite value leaves 0
__device__ __align__(16) const float f32_zero_chunk[4] = {};

struct F32Params {
  const float *q, *k, *v, *kp, *vp;
  float* o;
  float* lse;
  const void* map;
  int map_elem;
  int64_t q_sb, q_sh, q_sl, k_sb, k_sh, k_sl, v_sb, v_sh, v_sl, o_sb, o_sh, o_sl;
  int B, Hq, Hkv, L, Mq, Nk, bn_log2, bm, parts;
  int64_t npad;
  float scale_log2;
  int causal, max_tiles;
  const int32_t* q_index;
};

template <int D>
struct F32Geom {
  static constexpr int CH = D / 4;            // 16-byte chunks per row
  static constexpr int RPB = 64 / CH;         // rows per copy instruction (1 KiB)
  static constexpr int ROW = D * 4;           // bytes per row
  static constexpr int TILE = TK32 * ROW;     // bytes of a K or V tile
  static constexpr int STAGES = D == 64 ? 2 : 1;  // (128 channels: two workgroups per CU instead of a second buffer)
};

template <int D, int KS>
__global__ __launch_bounds__(256, 2) void psa_fwd_f32_kernel(F32Params p) {
  using G = F32Geom<D>;
  constexpr int QR = 64 / KS, KBW = 4 / KS, SQ = D / 16, DB = D / 16;
  extern __shared__ __align__(16) unsigned char smem[];  // [STAGES][K, V] tiles, later the shares of the output
  u32x2* tdesc = (u32x2*)(smem + G::STAGES * 2 * G::TILE);
  uint16_t* ids = (uint16_t*)(tdesc + p.max_tiles);
  __shared__ int s_cnt[4], s_ioff[4], s_toff[5], s_wcnt[16];
  __shared__ float s_m[4][16], s_l[4][16];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, g4 = lane >> 4;
  const int rg = wave / KS, ks = wave % KS;
  const int unit = blockIdx.x;  // (b, h, q-block, part)
  const int part = unit % p.parts, logical = unit / p.parts;
  const int I = logical % p.Mq, bh = logical / p.Mq, h = bh % p.Hq, b = bh / p.Hq;
  const int hk = h / (p.Hq / p.Hkv);
  const int q0 = I * p.bm + part * QR;  // first query position of this workgroup
  const int q_idx = q0 + rg * 16 + l16;
  int jmax = p.Nk;
  if (p.causal) {
    const int ce = (int)((((int64_t)(I + 1) * p.bm) + (1 << p.bn_log2) - 1) >> p.bn_log2);
    jmax = ce < jmax ? ce : jmax;
  }
  // Q: B operand of step 4 s + j holds channel 16 s + 4 g + j (rows past the sequence replicate the last one)
  f32x4 qf[SQ];
  {
    int qr = q_idx < p.L ? q_idx : p.L - 1;
    if (p.q_index != nullptr) qr = clamp_row(p.q_index[qr], p.L);
    const float* qp = p.q + b * p.q_sb + h * p.q_sh + (int64_t)qr * p.q_sl + 4 * g4;
#pragma unroll
    for (int s = 0; s < SQ; ++s) qf[s] = *(const f32x4*)(qp + 16 * s);
  }
  const int T = psa_tiles::build_row_schedule<256>(p.map, p.map_elem, ((int64_t)bh * p.Mq + I) * p.Nk, p.Nk, jmax, p.bn_log2, p.L,
                                                  p.causal != 0, (int64_t)I * p.bm, ids, tdesc, s_cnt, s_ioff, s_toff, s_wcnt);
  const float* kb0 = p.k + b * p.k_sb + hk * p.k_sh;
  const float* vb0 = p.v + b * p.v_sb + hk * p.v_sh;
  const int64_t BHkv = (int64_t)p.B * p.Hkv, bhk = (int64_t)b * p.Hkv + hk;

  // Copies: this wave brings tile rows 16 wave .. 16 wave + 15 of K and V.  LDS position c of a row holds chunk c ^ (row % 16).
  // Slots past the last key: K replicates a retained row (their logits are masked), V is zero - a replicated row with an infinite
  // value would turn the infinity that it rightly gives its channel into 0 * inf.
  const uint32_t lds0 = psa_tiles::lds_addr_of(smem);
  auto issue_rows = [&](const psa_tiles::TileRef& tr, int stage, auto full_c) __attribute__((always_inline)) {
    constexpr bool FULL = decltype(full_c)::value;  // every slot holds a key (a select per copy otherwise)
    const float* kbase = tr.lv == 0 ? kb0 : p.kp + psa_tiles::pool_row_offset(tr.lv, BHkv, bhk, p.npad) * D;
    const float* vbase = tr.lv == 0 ? vb0 : p.vp + psa_tiles::pool_row_offset(tr.lv, BHkv, bhk, p.npad) * D;
    const int64_t kstr = tr.lv == 0 ? p.k_sl : D, vstr = tr.lv == 0 ? p.v_sl : D;
#pragma unroll
    for (int n = 0; n < 16 / G::RPB; ++n) {
      const int row16 = n * G::RPB + lane / G::CH;
      const int pos = (tr.lt << 6) + wave * 16 + row16;
      int bi = pos >> tr.sbs_log2;
      if constexpr (!FULL) bi = bi < tr.cnt - 1 ? bi : tr.cnt - 1;
      int src = ((int)tr.ids[bi] << tr.sbs_log2) + (pos & ((1 << tr.sbs_log2) - 1));
      if constexpr (!FULL)
        if (tr.lv == 0) src = src < p.L ? src : p.L - 1;
      const int chunk = (lane % G::CH) ^ row16;
      const uint32_t at = lds0 + (uint32_t)(stage * 2 * G::TILE + (wave * 16 + n * G::RPB) * G::ROW);
      psa_tiles::lds_copy16_addr((const char*)(kbase + (int64_t)src * kstr + chunk * 4), at);
      const float* vsrc = vbase + (int64_t)src * vstr + chunk * 4;
      if constexpr (!FULL) vsrc = wave * 16 + row16 < tr.nvalid ? vsrc : f32_zero_chunk;
      psa_tiles::lds_copy16_addr((const char*)vsrc, at + G::TILE);
    }
  };
  auto issue_tile = [&](int t, int stage) __attribute__((always_inline)) {
    const psa_tiles::TileRef tr = psa_tiles::tile_ref(tdesc, ids, t, p.bn_log2);
    if (tr.nvalid == TK32) issue_rows(tr, stage, std::true_type{});
    else issue_rows(tr, stage, std::false_type{});
  };
  // operand addresses: K row l16 of a 16-key block, chunk 4 s + g; V rows 4 g + i, chunk l16 (+ 16 for the upper channels)
  uint32_t k_off[4], v_off[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) k_off[s] = (uint32_t)(l16 * G::ROW + (((4 * s + g4) ^ l16) * 16));
#pragma unroll
  for (int i = 0; i < 4; ++i) v_off[i] = (uint32_t)(G::TILE + (4 * g4 + i) * G::ROW + ((l16 ^ (4 * g4 + i)) * 16));

  f32x4 acc[DB];  // acc[4 c + e][i]: channel 64 c + 16 g + 4 i + e of query l16
#pragma unroll
  for (int db = 0; db < DB; ++db) acc[db] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;  // the row's maximum over this wave's keys; this lane's part of its sum

  auto compute = [&](int t, int stage) __attribute__((always_inline)) {
    PSA_LDS(unsigned char) Ts = (PSA_LDS(unsigned char))(smem) + stage * 2 * G::TILE + ks * (KBW * 16 * G::ROW);
    f32x4 s[KBW];
#pragma unroll
    for (int x = 0; x < KBW; ++x) {
      s[x] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < SQ; ++c) {
        const f32x4 a = *(PSA_LDS(const f32x4))(Ts + k_off[c & 3] + (c >> 2) * 256 + x * (16 * G::ROW));
#pragma unroll
        for (int j = 0; j < 4; ++j) s[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], qf[c][j], s[x], 0, 0, 0);
      }
    }
    const psa_tiles::TileRef tr = psa_tiles::tile_ref(tdesc, ids, t, p.bn_log2);
    const float bias = (float)tr.lv;
#pragma unroll
    for (int x = 0; x < KBW; ++x)
#pragma unroll
      for (int i = 0; i < 4; ++i) s[x][i] = __builtin_fmaf(s[x][i], p.scale_log2, bias);
    if (tr.masked) {
      // valid slots are a prefix of the tile; a pooled key of level lv is visible to query i once its last token is:
      // src < (i + 1) >> lv.  Both cut each run of 4 consecutive slots after its first `keep` elements.
      const int qlim = (q_idx + 1) >> tr.lv;
#pragma unroll
      for (int x = 0; x < KBW; ++x) {
        const int r0 = (ks * KBW + x) * 16 + 4 * g4;
        int keep = tr.nvalid - r0;
        if (p.causal) {
          const int pos = (tr.lt << 6) + r0;
          int bi = pos >> tr.sbs_log2;
          bi = bi < tr.cnt - 1 ? bi : tr.cnt - 1;
          const int src0 = ((int)tr.ids[bi] << tr.sbs_log2) + (pos & ((1 << tr.sbs_log2) - 1));
          keep = keep < qlim - src0 ? keep : qlim - src0;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) s[x][i] = i < keep ? s[x][i] : -INFINITY;
      }
    }
    float mx = fmaxf(fmaxf(s[0][0], s[0][1]), fmaxf(s[0][2], s[0][3]));
#pragma unroll
    for (int x = 1; x < KBW; ++x) mx = fmaxf(mx, fmaxf(fmaxf(s[x][0], s[x][1]), fmaxf(s[x][2], s[x][3])));
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m_new = fmaxf(m_run, mx);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = fast_exp2(m_run - m_use);
    float sum = 0.f;
#pragma unroll
    for (int x = 0; x < KBW; ++x)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[x][i] = fast_exp2(s[x][i] - m_use);
        sum += s[x][i];
      }
    l_run = l_run * alpha + sum;
    m_run = m_new;
    if (__any(alpha != 1.0f)) {
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[db][i] *= alpha;
    }
#pragma unroll
    for (int x = 0; x < KBW; ++x)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int c = 0; c < DB / 4; ++c) {
          const f32x4 a = *(PSA_LDS(const f32x4))(Ts + v_off[i] + c * 256 + x * (16 * G::ROW));
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[4 * c + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], s[x][i], acc[4 * c + e], 0, 0, 0);
        }
  };
  if (T > 0) {
    if constexpr (G::STAGES == 2) {
      issue_tile(0, 0);
      __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
      __syncthreads();
      for (int t = 0; t < T; ++t) {
        if (t + 1 < T) issue_tile(t + 1, (t + 1) & 1);
        compute(t, t & 1);
        __builtin_amdgcn_s_waitcnt(0x0f70);
        __syncthreads();
      }
    } else {
      for (int t = 0; t < T; ++t) {
        issue_tile(t, 0);
        __builtin_amdgcn_s_waitcnt(0x0f70);
        __syncthreads();
        compute(t, 0);
        __syncthreads();  // the tile's readers are done
      }
    }
  }

  // ---- the KS shares of a row meet in LDS; results leave as rows ---------------------------------------------------
  constexpr int OP = D + 4;  // padded row of the staging area (floats)
  float l_tot = l_run + __shfl_xor(l_run, 16, 64);
  l_tot += __shfl_xor(l_tot, 32, 64);
  float* os = (float*)smem + wave * 16 * OP;
#pragma unroll
  for (int c = 0; c < DB / 4; ++c)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *(f32x4*)(os + l16 * OP + 64 * c + 16 * g4 + 4 * i) = f32x4{acc[4 * c][i], acc[4 * c + 1][i], acc[4 * c + 2][i], acc[4 * c + 3][i]};
  if (g4 == 0) {
    s_m[wave][l16] = m_run;
    s_l[wave][l16] = l_tot;
  }
  __syncthreads();
  for (int u = tid; u < QR * G::CH; u += 256) {
    const int r = u / G::CH, c4 = u % G::CH, w0 = (r >> 4) * KS, r16 = r & 15;
    const int qi = q0 + r;
    if (qi >= p.L) continue;
    const int orow = p.q_index != nullptr ? p.q_index[qi] : qi;
    if ((unsigned)orow >= (unsigned)p.L) continue;
    float m = s_m[w0][r16];
#pragma unroll
    for (int w = 1; w < KS; ++w) m = fmaxf(m, s_m[w0 + w][r16]);
    const float m_use = m == -INFINITY ? 0.f : m;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    float l = 0.f;
#pragma unroll
    for (int w = 0; w < KS; ++w) {
      const float f = fast_exp2(s_m[w0 + w][r16] - m_use);
      const f32x4 x = *(const f32x4*)((const float*)smem + ((w0 + w) * 16 + r16) * OP + c4 * 4);
      l = __builtin_fmaf(s_l[w0 + w][r16], f, l);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = __builtin_fmaf(x[e], f, o[e]);
    }
    const float l_safe = fmaxf(l, 1e-8f);
    const float inv = 1.0f / l_safe;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] *= inv;
    *(f32x4*)(p.o + b * p.o_sb + h * p.o_sh + (int64_t)orow * p.o_sl + c4 * 4) = o;
    if (p.lse != nullptr && c4 == 0) p.lse[((int64_t)b * p.Hq + h) * p.L + orow] = (m + fast_log2(l_safe)) * 0.6931471805599453f;
  }
}

template <int D, int KS>
int launch_f32(const F32Params& p, hipStream_t stream) {
  using G = F32Geom<D>;
  const size_t shmem = (size_t)G::STAGES * 2 * G::TILE + (size_t)p.max_tiles * 8 + (size_t)p.Nk * 2 + 16;
  if (shmem > 159 * 1024) return PSA_ERR_UNSUPPORTED;
  if (hipFuncSetAttribute((const void*)psa_fwd_f32_kernel<D, KS>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem) != hipSuccess)
    return PSA_ERR_LAUNCH;
  const int64_t units = (int64_t)p.B * p.Hq * p.Mq * p.parts;
  hipLaunchKernelGGL((psa_fwd_f32_kernel<D, KS>), dim3((unsigned)units), dim3(256), shmem, stream, p);
  return PSA_OK;
}

}  // namespace

int psa_fwd_f32(psa_tensor4 q, psa_tensor4 k, psa_tensor4 v, const void* k_pool, const void* v_pool, const void* map, int map_elem_bytes,
                psa_tensor4 out, float* lse, int B, int Hq, int Hkv, int L, int D, int block_m, int block_n, float sm_scale, int causal,
                psa_stream_t stream, const int32_t* q_index) {
  PSA_REQUIRE(q.ptr && k.ptr && v.ptr && out.ptr, PSA_ERR_ARG, "psa_fwd: null pointer");
  PSA_REQUIRE(map == nullptr || (k_pool && v_pool), PSA_ERR_ARG, "psa_fwd: pooled K/V required with a level map");
  PSA_REQUIRE(map_elem_bytes == 1 || map_elem_bytes == 4, PSA_ERR_ARG, "psa_fwd: map_elem_bytes must be 1 or 4");
  PSA_REQUIRE(Hq % Hkv == 0, PSA_ERR_ARG, "psa_fwd: Hq=%d must be a multiple of Hkv=%d", Hq, Hkv);
  PSA_REQUIRE(sm_scale > 0.f, PSA_ERR_ARG, "psa_fwd: sm_scale must be positive");
  PSA_REQUIRE(D == 64 || D == 128, PSA_ERR_UNSUPPORTED, "psa_fwd: head dim %d not in {64, 128}", D);
  PSA_REQUIRE(block_m == 64 || block_m == 128, PSA_ERR_UNSUPPORTED, "psa_fwd: block_m=%d not in {64, 128}", block_m);
  PSA_REQUIRE(block_n == 32 || block_n == 64 || block_n == 128, PSA_ERR_UNSUPPORTED, "psa_fwd: block_n=%d not in {32, 64, 128}", block_n);
  const psa_tensor4* ts[4] = {&q, &k, &v, &out};
  for (int i = 0; i < 4; ++i)
    PSA_REQUIRE(((uintptr_t)ts[i]->ptr % 16 == 0) && ts[i]->stride_b % 4 == 0 && ts[i]->stride_h % 4 == 0 && ts[i]->stride_l % 4 == 0,
                PSA_ERR_UNSUPPORTED, "psa_fwd: fp32 tensors must be 16-byte aligned with strides that are multiples of 4 elements");
  const int Mq = (L + block_m - 1) / block_m, Nk = (L + block_n - 1) / block_n;
  PSA_REQUIRE(Nk <= 65535, PSA_ERR_UNSUPPORTED, "psa_fwd: more than 65535 kv-blocks");
  PSA_REQUIRE((int64_t)B * Hq * Mq * 8 < (1ll << 31), PSA_ERR_UNSUPPORTED, "psa_fwd: too many workgroups");
  F32Params p;
  p.q = (const float*)q.ptr; p.k = (const float*)k.ptr; p.v = (const float*)v.ptr; p.o = (float*)out.ptr;
  p.kp = (const float*)k_pool; p.vp = (const float*)v_pool;
  p.lse = lse; p.map = map; p.map_elem = map_elem_bytes;
  p.q_sb = q.stride_b; p.q_sh = q.stride_h; p.q_sl = q.stride_l;
  p.k_sb = k.stride_b; p.k_sh = k.stride_h; p.k_sl = k.stride_l;
  p.v_sb = v.stride_b; p.v_sh = v.stride_h; p.v_sl = v.stride_l;
  p.o_sb = out.stride_b; p.o_sh = out.stride_h; p.o_sl = out.stride_l;
  p.B = B; p.Hq = Hq; p.Hkv = Hkv; p.L = L; p.Mq = Mq; p.Nk = Nk;
  // rows per workgroup: 64, or 32 / 16 while the launch would have fewer than two workgroups per CU
  int ks = 1;
  while (ks < 4 && (int64_t)B * Hq * Mq * (block_m * ks / 64) < 512) ks *= 2;
  p.bn_log2 = psa_ilog2(block_n); p.bm = block_m; p.parts = block_m * ks / 64;
  p.npad = (int64_t)Nk * block_n;
  p.scale_log2 = sm_scale * 1.4426950408889634f;
  p.causal = causal ? 1 : 0;
  p.max_tiles = (block_n >= 64 ? Nk * (block_n / 64) : (Nk * block_n + 63) / 64) + 4;
  p.q_index = q_index;
  hipStream_t st = (hipStream_t)stream;
  int rc;
  if (D == 128) rc = ks == 1 ? launch_f32<128, 1>(p, st) : ks == 2 ? launch_f32<128, 2>(p, st) : launch_f32<128, 4>(p, st);
  else rc = ks == 1 ? launch_f32<64, 1>(p, st) : ks == 2 ? launch_f32<64, 2>(p, st) : launch_f32<64, 4>(p, st);
  PSA_REQUIRE(rc == PSA_OK, rc, "psa_fwd: sequence too long for the fp32 kernel's on-chip schedule (LDS)");
  return psa_check_launch("psa_fwd (fp32)");
}
