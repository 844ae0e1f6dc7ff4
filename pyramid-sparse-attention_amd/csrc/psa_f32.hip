// Pyramid sparse attention forward on fp32 tensors: fp32 operands and fp32 arithmetic throughout, products on the matrix
// cores' fp32 instruction (v_mfma_f32_16x16x4_f32: a k-ordered chain of fp32 multiply-adds).  Same walk as the 16-bit kernels
// (psa_tiles.h: the map row is compacted into tiles of 64 pooled keys of one level), same softmax (base 2, +log2(level)
// bias, online), same masks.
//
// A tile's four 16-key blocks go one to each wave of a workgroup (psa_fwd_f32_direct_kernel: 16 or 32 query rows; a softmax state per
// wave, joined once at the end) or all, or two, to every wave, which then has 16 rows of its own or with one other (psa_fwd_f32_kernel: 64 or
// 32 rows).  Which: launch_f32.
// The transposed products S^T = K Q^T and O^T += V^T P^T leave a lane 4 keys of one query in the accumulator, and with
// k-index g of the i-th PV step taken to be key 4 g + i that register IS the step's B operand: nothing crosses lanes
// between the two products, and a row maximum is two lane exchanges.  Channels are dealt so that a lane's operands of four
// steps are 16 consecutive bytes.
// Bound by the vector units: the fp32 matrix instruction runs on them, 32 cycles of a SIMD for 16 x 16 x 4, and nothing else issues beside
// it.  What helps is fewer instructions around it.
// 2 heads of 4096 tokens x 64, 64-key blocks, 80 % sparse: 109 us with plain multiply-adds (two LDS operands per 4 FMAs), 36 with tiles through
// LDS, 27 here (11 of them products).
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

// The KS shares of a row meet in LDS; results leave as rows.  smem: 64 rows of D + 4 floats.
template <int D, int KS>
__device__ __forceinline__ void f32_finish(const F32Params& p, int b, int h, int q0, int wave, int l16, int g4, int tid, const f32x4 (&acc)[D / 16],
                                           float m_run, float l_run, float* smem, float (*s_m)[16], float (*s_l)[16]) {
  using G = F32Geom<D>;
  constexpr int QR = 64 / KS, DB = D / 16;
  constexpr int OP = D + 4;  // padded row of the staging area (floats)
  float l_tot = l_run + __shfl_xor(l_run, 16, 64);
  l_tot += __shfl_xor(l_tot, 32, 64);
  float* os = smem + wave * 16 * OP;
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
      const f32x4 x = *(const f32x4*)(smem + ((w0 + w) * 16 + r16) * OP + c4 * 4);
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

// 64 / KS rows per workgroup; KS waves share a row's keys.  The K and V tile goes straight into LDS and is shared by the waves; rows are XOR-swizzled by 16-byte chunks (one ds_read_b128 per four steps): conflict-free.
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
  const int unit = blockIdx.x;  // (b, h, q-block, part)
  const int part = unit % p.parts, logical = unit / p.parts;
  const int I = logical % p.Mq, bh = logical / p.Mq, h = bh % p.Hq, b = bh / p.Hq;
  const int hk = h / (p.Hq / p.Hkv);
  const int q0 = I * p.bm + part * QR;  // first query position of this workgroup
  const int rg = wave / KS, ks = wave % KS;  // this wave's 16 rows and its share of a tile's keys
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
    mx = quarter_wave_max(mx);
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

  f32_finish<D, KS>(p, b, h, q0, wave, l16, g4, tid, acc, m_run, l_run, (float*)smem, s_m, s_l);
}

// 16 RG rows per workgroup, K and V rows straight into the registers of the wave that has their block: no LDS tiles and no barriers between
// the row's list and the end.  The next block's rows are requested before a block's products (two blocks ahead: more registers, fewer waves, 4 to
// 8 % slower).  Wave w has keys 16 w .. 16 w + 15 of every tile.  RG = 2 halves the row addresses per product and the number of workgroups.
// (RG = 2 at head dim 128 would take more than the 256 registers of two waves per SIMD.)
template <int D, int RG>
__global__ __launch_bounds__(256, 2) void psa_fwd_f32_direct_kernel(F32Params p) {
  constexpr int SQ = D / 16, DB = D / 16, NV = D / 16, NB = 2;
  extern __shared__ __align__(16) unsigned char smem[];  // the shares of the output, then the row's tiles
  u32x2* tdesc = (u32x2*)(smem + 64 * (D + 4) * 4);
  uint16_t* ids = (uint16_t*)(tdesc + p.max_tiles);
  __shared__ int s_cnt[4], s_ioff[4], s_toff[5], s_wcnt[16];
  __shared__ float s_m[4][16], s_l[4][16];
  __shared__ __align__(16) u32x4 s_base[4];  // first rows of K and V of every level

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, g4 = lane >> 4;
  const int unit = blockIdx.x;  // (b, h, q-block, part)
  const int part = unit % p.parts, logical = unit / p.parts;
  const int I = logical % p.Mq, bh = logical / p.Mq, h = bh % p.Hq, b = bh / p.Hq;
  const int hk = h / (p.Hq / p.Hkv);
  const int q0 = I * p.bm + part * (16 * RG);
  int jmax = p.Nk;
  if (p.causal) {
    const int ce = (int)((((int64_t)(I + 1) * p.bm) + (1 << p.bn_log2) - 1) >> p.bn_log2);
    jmax = ce < jmax ? ce : jmax;
  }
  f32x4 qf[RG][SQ];
#pragma unroll
  for (int r = 0; r < RG; ++r) {
    int qr = q0 + r * 16 + l16;
    qr = qr < p.L ? qr : p.L - 1;
    if (p.q_index != nullptr) qr = clamp_row(p.q_index[qr], p.L);
    const float* qp = p.q + b * p.q_sb + h * p.q_sh + (int64_t)qr * p.q_sl + 4 * g4;
#pragma unroll
    for (int s = 0; s < SQ; ++s) qf[r][s] = *(const f32x4*)(qp + 16 * s);
  }
  if (tid < 4) {
    const int64_t BHkv = (int64_t)p.B * p.Hkv, bhk = (int64_t)b * p.Hkv + hk, at = psa_tiles::pool_row_offset(tid, BHkv, bhk, p.npad) * D;
    const uint64_t kb = (uint64_t)(tid == 0 ? p.k + b * p.k_sb + hk * p.k_sh : p.kp + at), vb = (uint64_t)(tid == 0 ? p.v + b * p.v_sb + hk * p.v_sh : p.vp + at);
    s_base[tid] = u32x4{(uint32_t)kb, (uint32_t)(kb >> 32), (uint32_t)vb, (uint32_t)(vb >> 32)};
  }
  const int T = psa_tiles::build_row_schedule<256>(p.map, p.map_elem, ((int64_t)bh * p.Mq + I) * p.Nk, p.Nk, jmax, p.bn_log2, p.L,
                                                  p.causal != 0, (int64_t)I * p.bm, ids, tdesc, s_cnt, s_ioff, s_toff, s_wcnt);

  // Rows through buffer descriptors: 32-bit offsets (one 24-bit multiply-add per lane and tensor), the four V rows of a lane, which follow
  // each other in one block, by scalar offsets.
  auto rows_of = [](uint32_t lo, uint32_t hi) __attribute__((always_inline)) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane(hi) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane(lo)), 0, -1, 0x00020000);
  };

  // Two look-ups lead from a tile to its rows: its description, then the blocks of this lane's K row and V rows.
  struct Block {
    f32x4 k[SQ], v[NV];
    uint32_t d0, d1;
  };
  u32x2 d_next = {0u, 0u};
  uint32_t d0 = 0, d1 = 0;
  int k_id = 0, v_id = 0;
  u32x4 base = {0u, 0u, 0u, 0u};
  auto look_desc = [&](int t) __attribute__((always_inline)) { d_next = tdesc[t < T ? t : T - 1]; };
  auto look_ids = [&]() __attribute__((always_inline)) {
    d0 = __builtin_amdgcn_readfirstlane(d_next[0]);
    d1 = __builtin_amdgcn_readfirstlane(d_next[1]);
    const int sbs_log2 = p.bn_log2 - (int)(d0 & 3), last = (int)(d1 >> 16) - 1;
    const uint16_t* list = ids + (d1 & 0xffff);
    const int pos = ((int)(d0 >> 10) << 6) + wave * 16;
    int kb = (pos + l16) >> sbs_log2, vb = (pos + 4 * g4) >> sbs_log2;
    kb = kb < last ? kb : last;
    vb = vb < last ? vb : last;
    k_id = list[kb];
    v_id = list[vb];
    base = s_base[d0 & 3];
  };
  auto load = [&](Block& w) __attribute__((always_inline)) {
    const int lv = d0 & 3, sbs_log2 = p.bn_log2 - lv, mask = (1 << sbs_log2) - 1, pos = ((int)(d0 >> 10) << 6) + wave * 16;
    const uint32_t kstr = lv == 0 ? (uint32_t)p.k_sl * 4u : D * 4u, vstr = lv == 0 ? (uint32_t)p.v_sl * 4u : D * 4u;
    const auto kr = rows_of(base[0], base[1]), vr = rows_of(base[2], base[3]);
    const int last = (lv == 0 ? p.L : (int)(p.npad >> lv)) - 1;
    int ks = (k_id << sbs_log2) + ((pos + l16) & mask);
    ks = ks < last ? ks : last;
    const int at = (int)__umul24(ks, kstr) + 16 * g4;
#pragma unroll
    for (int s = 0; s < SQ; ++s) w.k[s] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(kr, at + 64 * s, 0, 0));
    const int vs = (v_id << sbs_log2) + ((pos + 4 * g4) & mask);
    if (lv == 0 && (d0 >> 3 & 127) < TK32) {  // (the sequence may end among the four rows)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int vat = (int)__umul24(vs + i < last ? vs + i : last, vstr) + 16 * l16;
#pragma unroll
        for (int c = 0; c < DB / 4; ++c) w.v[i * (DB / 4) + c] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(vr, vat + 256 * c, 0, 0));
      }
    } else {
      const int vat = (int)__umul24(vs, vstr) + 16 * l16;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int c = 0; c < DB / 4; ++c)
          w.v[i * (DB / 4) + c] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(vr, vat + 256 * c, (int)(i * vstr), 0));
    }
    w.d0 = d0;
    w.d1 = d1;
  };

  f32x4 acc[RG][DB];
  float m_run[RG], l_run[RG];
#pragma unroll
  for (int r = 0; r < RG; ++r) {
#pragma unroll
    for (int db = 0; db < DB; ++db) acc[r][db] = f32x4{0.f, 0.f, 0.f, 0.f};
    m_run[r] = -INFINITY;
    l_run[r] = 0.f;
  }

  auto compute = [&](Block& w) __attribute__((always_inline)) {
    const int lv = w.d0 & 3, nvalid = (w.d0 >> 3) & 127;
    if (wave * 16 >= nvalid) return;
    f32x4 s[RG];
#pragma unroll
    for (int r = 0; r < RG; ++r) s[r] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < SQ; ++c)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < RG; ++r) s[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(w.k[c][j], qf[r][c][j], s[r], 0, 0, 0);
    const float bias = (float)lv;
#pragma unroll
    for (int r = 0; r < RG; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) s[r][i] = __builtin_fmaf(s[r][i], p.scale_log2, bias);
    if (w.d0 & 4) {
      // (as above; V rows of slots that hold no key are some row of the sequence and become zero)
      const int r0 = wave * 16 + 4 * g4, full = nvalid - r0;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int c = 0; c < DB / 4; ++c)
#pragma unroll
          for (int e = 0; e < 4; ++e) w.v[i * (DB / 4) + c][e] = i < full ? w.v[i * (DB / 4) + c][e] : 0.f;
      int src0 = 0;
      if (p.causal) {
        const int pos = ((int)(w.d0 >> 10) << 6) + r0, sbs_log2 = p.bn_log2 - lv, last = (int)(w.d1 >> 16) - 1;
        int bi = pos >> sbs_log2;
        bi = bi < last ? bi : last;
        src0 = ((int)ids[(w.d1 & 0xffff) + bi] << sbs_log2) + (pos & ((1 << sbs_log2) - 1));
      }
#pragma unroll
      for (int r = 0; r < RG; ++r) {
        const int qlim = (q0 + r * 16 + l16 + 1) >> lv;
        const int keep = p.causal && qlim - src0 < full ? qlim - src0 : full;
#pragma unroll
        for (int i = 0; i < 4; ++i) s[r][i] = i < keep ? s[r][i] : -INFINITY;
      }
    }
#pragma unroll
    for (int r = 0; r < RG; ++r) {
      const float mx = quarter_wave_max(fmaxf(fmaxf(s[r][0], s[r][1]), fmaxf(s[r][2], s[r][3])));
      const float m_new = fmaxf(m_run[r], mx);
      const float m_use = m_new == -INFINITY ? 0.f : m_new;
      const float alpha = fast_exp2(m_run[r] - m_use);
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[r][i] = fast_exp2(s[r][i] - m_use);
        sum += s[r][i];
      }
      l_run[r] = l_run[r] * alpha + sum;
      m_run[r] = m_new;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[r][db][i] *= alpha;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int c = 0; c < DB / 4; ++c)
#pragma unroll
        for (int r = 0; r < RG; ++r)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            acc[r][4 * c + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(w.v[i * (DB / 4) + c][e], s[r][i], acc[r][4 * c + e], 0, 0, 0);
  };
  if (T > 0) {
    Block w[NB];
    look_desc(0);
    look_ids();
    look_desc(1);
#pragma unroll
    for (int n = 0; n < NB - 1; ++n) {
      load(w[n]);
      look_ids();
      look_desc(n + 2);
    }
    auto step = [&](int t, Block& next, Block& w) __attribute__((always_inline)) {
      load(next);  // tile t + NB - 1, or the last again
      look_ids();
      look_desc(t + NB + 1);
      __builtin_amdgcn_sched_barrier(0);
      compute(w);
      __builtin_amdgcn_sched_barrier(0);
    };
    for (int t = 0;;) {
      step(t, w[NB - 1], w[0]);
      if (++t >= T) break;
      step(t, w[0], w[1]);
      if (++t >= T) break;
    }
  }
#pragma unroll
  for (int r = 0; r < RG; ++r) {
    if (r > 0) __syncthreads();  // the staging area's readers are done
    f32_finish<D, 4>(p, b, h, q0 + 16 * r, wave, l16, g4, tid, acc[r], m_run[r], l_run[r], (float*)smem, s_m, s_l);
  }
}

size_t f32_list_bytes(const F32Params& p) { return (size_t)p.max_tiles * 8 + (size_t)p.Nk * 2 + 16; }

template <class K>
int launch_f32(K kernel, size_t tiles, int64_t grid, const F32Params& p, hipStream_t stream) {
  const size_t shmem = tiles + f32_list_bytes(p);
  if (shmem > 48 * 1024 && hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem) != hipSuccess)
    return PSA_ERR_LAUNCH;
  hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(256), shmem, stream, p);
  return PSA_OK;
}
// Workgroups of 16 or 32 rows without LDS tiles, or of 32 or 64 rows with them.  The former list a row's tiles two to four times as often and
// fetch K and V as often again; the latter wait at a barrier for every tile and, with 64 rows, leave small launches with too few workgroups.
// Layers, us, tiles in LDS (16 rows below 1024 blocks of 16 rows, 32 below 2048, 64 from there on) / without (RG = 1 up to 1280 blocks, 2 above;
// head dim 128: 1) / as chosen here, on keys with a common part, topk (head dim 64: 128-key blocks, and where marked 64):
//   head dim 64   8 heads x 1000  32 / 29 / 28   12 x 2048  49 / 41 / 41   17 x 2000  63 / 54 / 55   24 x 1536  55 / 51 / 51   12 x 4000  106 / 98 / 99
//                 8 x 8000  229 / 224 / 223   1 x 30000  449 / 390 / 388.   Short rows in one or two full rounds of 64-row workgroups: 16 x 2000  50 / 54 / 49
//                 32 x 1000 (64)  46 / 47 / 43   200 x 300 (64)  59 / 66 / 59   512 x 128  59 / 65 / 59
//   head dim 128  2 x 4096  63 / 56 / 56   8 x 1000  40 / 36 / 35   24 x 640 (960)  44 / 45 / 46   3 x 7000  195 / 183 / 183   1 x 20000  458 / 377 / 377   3 x 9000 (1704 blocks)  298 / 266 / 265
//                 6 x 4600 (1728)  160 / 152 / 151.   Short rows: 12 x 2048 (1536)  75 / 80 / 71   24 x 1152 (1728)  84 / 92 / 84.   More rows: 16 x 2000 (2000)
//                 78 / 99 / 76   12 x 4000 (3072)  194 / 220 / 191   8 x 6000 (3008)  270 / 297 / 264   96 x 500 (3072)  88 / 117 / 86.   K and V of a head beyond 20 MiB,
//                 which rows of 16 fetch from memory: 1 x 24000  567 / 511 / 537   1 x 30000 (1880)  830 / 793 / 830 (forward on a random map of 80 % 726 / 890 / 726)
// Rounding (relative to float64, random maps): 12 x 1400 x 128 4.3e-7 / 4.0e-7 / 4.3e-7, 32 x 1000 x 64 3.6e-7 / 2.8e-7 / 3.6e-7; without tiles a row's
// keys are added up in four parts.
template <int D>
int launch_f32(F32Params p, hipStream_t stream) {
  const int64_t rows16 = (int64_t)p.B * p.Hq * p.Mq * (p.bm / 16);
  // (sizes in elements: a row's offset in bytes below 2^31, its factors below 2^24)
  auto near = [&](int64_t stride, int64_t rows) { return stride >= 0 && stride < (1 << 22) && rows < (1 << 24) && rows * (stride > D ? stride : D) < (1ll << 29); };
  const bool direct = near(p.k_sl, p.L) && near(p.v_sl, p.L) && near(D, p.npad);
  // workgroups of 64 rows in one or two full rounds of the chip's 512 places
  const bool full_rounds = rows16 >= 2048 && rows16 <= 4096 && (rows16 - 1) % 2048 >= 1840;
  const bool wins = D == 64 ? p.L > 2048 || !full_rounds : rows16 < 1024 || (rows16 <= 1728 && p.L >= 4096 && p.L <= 20480);
  if (direct && wins) {
    const int rg = D == 64 && rows16 > 1280 ? 2 : 1;
    p.parts = p.bm / (16 * rg);
    const size_t stage = (size_t)64 * (D + 4) * 4;
    if constexpr (D == 64)
      if (rg == 2) return launch_f32(psa_fwd_f32_direct_kernel<D, 2>, stage, rows16 / rg, p, stream);
    return launch_f32(psa_fwd_f32_direct_kernel<D, 1>, stage, rows16 / rg, p, stream);
  }
  const size_t tiles = (size_t)F32Geom<D>::STAGES * 2 * F32Geom<D>::TILE;
  const int ks = rows16 < 2048 ? 2 : 1;
  p.parts = p.bm * ks / 64;
  if (ks == 2) return launch_f32(psa_fwd_f32_kernel<D, 2>, tiles, rows16 / 2, p, stream);
  return launch_f32(psa_fwd_f32_kernel<D, 1>, tiles, rows16 / 4, p, stream);
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
  p.bn_log2 = psa_ilog2(block_n); p.bm = block_m;
  p.npad = (int64_t)Nk * block_n;
  p.scale_log2 = sm_scale * 1.4426950408889634f;
  p.causal = causal ? 1 : 0;
  p.max_tiles = (block_n >= 64 ? Nk * (block_n / 64) : (Nk * block_n + 63) / 64) + 4;
  p.q_index = q_index;
  hipStream_t st = (hipStream_t)stream;
  PSA_REQUIRE(64 * 1024 + f32_list_bytes(p) <= 159 * 1024, PSA_ERR_UNSUPPORTED, "psa_fwd: sequence too long for the fp32 kernel's on-chip schedule (LDS)");
  const int rc = D == 128 ? launch_f32<128>(p, st) : launch_f32<64>(p, st);
  PSA_REQUIRE(rc == PSA_OK, rc, "psa_fwd: cannot reserve the fp32 kernel's LDS");
  return psa_check_launch("psa_fwd (fp32)");
}
