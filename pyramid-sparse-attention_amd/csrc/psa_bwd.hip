// Backward of the pyramid sparse attention w.r.t. Q, K, V.
//
//   delta_i = sum_d O_id dO_id
//   p_it    = exp2(scale*log2e * q_i.K_l[t] + log2(l) - lse_i*log2e)     (one value per retained pooled key)
//   dV_l[t] += sum_i p_it dO_i          dP_it = dO_i . V_l[t]          dS_it = p_it (dP_it - delta_i)
//   dQ_i    += scale sum_t dS_it K_l[t]                                dK_l[t] += scale sum_i dS_it q_i
//   dK[n]    = dK_1[n] + sum_{l=2,4,8} dK_l[n/l] / l, the part of replicate-pad rows n >= L added to row L-1
//
// Kernels:
//   psa_bwd_cost_kernel    row and column costs of the walks, whose issue orders psa_order.h sorts
//   psa_bwd_delta_kernel   HBM-bound: -delta and -lse in log2 units (rows without keys get -inf so p = 0)
//   psa_bwd_dq_lds_kernel  MFMA-bound row walk: the forward's tile schedule; per tile S^T = K Q^T,
//                          dP^T = V dO^T, dQ^T += K^T dS^T on bf16 / fp16 MFMA, operands pooled K/V read directly
//   psa_bwd_dkdv_lds_kernel MFMA-bound column walk: one workgroup per (kv head, kv-block, level slot) keeps
//                          its pooled keys (128 at most) in registers and streams the q-blocks that retain this block at
//                          this level; dK_l, dV_l go to an fp32 workspace (every row written exactly once)
//   psa_bwd_unpool_kernel  HBM-bound: sums the levels, spreads pooled gradients, folds the pad tail, -> the tensors' type
#include "psa_tiles.h"
#include "psa_order.h"

namespace {

using namespace psa_tiles;

struct BwdParams {
  const bf16_t *q, *k, *v, *o, *dout;
  int64_t q_sb, q_sh, q_sl, k_sb, k_sh, k_sl, v_sb, v_sh, v_sl, o_sb, o_sh, o_sl, do_sb, do_sh, do_sl;
  bf16_t *dq, *dk, *dv;
  int64_t dq_sb, dq_sh, dq_sl, dk_sb, dk_sh, dk_sl, dv_sb, dv_sh, dv_sl;
  const bf16_t *kp, *vp;
  const void* map;
  int map_elem;
  const float* lse;
  float *ndelta, *nlse2;  // workspace [B*Hq*L] each: -delta, -lse in log2 units
  float *wk, *wv;       // workspace: per-level fp32 dK / dV, levels back to back: [BHkv, npad >> lv, D]
  int B, Hq, Hkv, L, Mq, Nk, bn_log2, bm;
  int64_t npad;
  float scale, scale_log2;
  int causal;
  int max_tiles;
};

// ------------------------------------------------------------------------------------------------------
// delta and log2-domain lse
// ------------------------------------------------------------------------------------------------------
template <int D, class ET>
__global__ __launch_bounds__(256) void psa_bwd_delta_kernel(BwdParams p) {
  constexpr int LPR = D / 8;  // lanes per row
  const int bh = blockIdx.y, b = bh / p.Hq, h = bh % p.Hq;
  const int64_t row = (int64_t)blockIdx.x * (256 / LPR) + threadIdx.x / LPR;
  const int c = threadIdx.x % LPR;
  float acc = 0.f;
  if (row < p.L) {
    const u32x4 ow = *(const u32x4*)(p.o + b * p.o_sb + h * p.o_sh + row * p.o_sl + c * 8);
    const u32x4 dw = *(const u32x4*)(p.dout + b * p.do_sb + h * p.do_sh + row * p.do_sl + c * 8);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      acc += ET::from_bits(ow[j] & 0xffffu) * ET::from_bits(dw[j] & 0xffffu);
      acc += ET::from_bits(ow[j] >> 16) * ET::from_bits(dw[j] >> 16);
    }
  }
#pragma unroll
  for (int o = LPR / 2; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
  if (c == 0 && row < p.L) {
    const float l = p.lse[(int64_t)bh * p.L + row];
    p.ndelta[(int64_t)bh * p.L + row] = -acc;
    // rows that saw no key have lse = -inf and zero gradient: -inf makes every p vanish
    p.nlse2[(int64_t)bh * p.L + row] = (l == -INFINITY) ? -INFINITY : l * -1.4426950408889634f;
  }
}

// ------------------------------------------------------------------------------------------------------
// dQ row walk.  K and V tiles are copied from global memory straight into double-buffered LDS tiles (layout: psa_tiles.h), one
// barrier per tile; S^T = K Q^T and dP^T = V dO^T read them row-wise (128-bit reads), dQ^T += K^T dS^T reads the K tile
// through the transposing LDS load.  dP's accumulators start from -delta.
// Bound by the board's power and by the instruction port, as the forward at head dim 128 is, whence the same measures: 16 x 16 x 32
// MFMAs, which sustain 2.1 PFLOP/s on random operands where 32 x 32 x 16 ones sustain 1.8, and the vector instructions of one half
// of a tile between the MFMAs of another product (they came after all of a tile's logits).  12 heads of 32760 x 128 at 85 %
// sparsity 1374 -> 1181 us, 48 heads of 8776 x 64 262 -> 215 us; training steps 4752 -> 4613 us, 1121 -> 1098 us.
// ------------------------------------------------------------------------------------------------------
template <int D, int NW, class ET>
__global__ __launch_bounds__(NW * 64, 2) void psa_bwd_dq_lds_kernel(BwdParams p, int chunk, const int32_t* order) {
  using G = LtGeom<D>;
  using x8 = typename ET::x8;
  constexpr int LT_TILE = G::TILE;
  constexpr int NT = NW * 64, BM = NW * 32, CH = D / 8, KK = D / 32, DB = D / 16;
  constexpr int G16 = 4 / NW;
  constexpr int OST = D * 2 + 16;
  static_assert(BM * OST <= 4 * LT_TILE, "dQ staging must fit the tile buffers");

  extern __shared__ __align__(16) unsigned char smem[];
  // K tiles at 0 and LT_TILE, V tiles at 2*LT_TILE and 3*LT_TILE
  u32x2* tdesc = (u32x2*)(smem + 4 * LT_TILE);
  uint16_t* ids = (uint16_t*)(tdesc + p.max_tiles);
  __shared__ int s_cnt[4], s_ioff[4], s_toff[5], s_wcnt[4 * NW];

  // the workgroup's row (b, h, q-block): shares of rows per XCD, longest rows first (see psa_order.h)
  int row = psa_order::dealt_entry((int)blockIdx.x, chunk);
  if (order != nullptr) row = order[row];
  if (row < 0 || row >= p.B * p.Hq * p.Mq) return;
  const int I = row % p.Mq;
  const int bh = row / p.Mq;
  const int h = bh % p.Hq, b = bh / p.Hq;
  const int hk = h / (p.Hq / p.Hkv);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lg = lane >> 4;
  const int L = p.L, bn_log2 = p.bn_log2, causal = p.causal;
  const float scale_log2 = p.scale_log2;

  int jmax = p.Nk;
  if (causal) {
    const int ce = (int)((((int64_t)(I + 1) * p.bm) + (1 << bn_log2) - 1) >> bn_log2);
    jmax = ce < jmax ? ce : jmax;
  }
  // Q and dO fragments (B operands) of this wave's 32 rows, two blocks of 16: lane holds row l16, channels 32 * kk + 8 * lg .. + 7;
  // per-row delta and lse
  const int q_idx = I * BM + wave * 32 + l16;  // block qb: + 16 * qb
  x8 qf[2][KK], dof[2][KK];
  float ndelta[2], nlse2[2];
#pragma unroll
  for (int qb = 0; qb < 2; ++qb) {
    const int qi = q_idx + 16 * qb, qr = qi < L ? qi : L - 1;
    const bf16_t* qp = p.q + b * p.q_sb + h * p.q_sh + (int64_t)qr * p.q_sl + lg * 8;
    const bf16_t* dp_ = p.dout + b * p.do_sb + h * p.do_sh + (int64_t)qr * p.do_sl + lg * 8;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      qf[qb][kk] = *(const x8*)(qp + kk * 32);
      dof[qb][kk] = *(const x8*)(dp_ + kk * 32);
    }
    ndelta[qb] = qi < L ? p.ndelta[(int64_t)bh * L + qi] : 0.f;
    nlse2[qb] = qi < L ? p.nlse2[(int64_t)bh * L + qi] : -INFINITY;
  }

  const int T = build_row_schedule<NT>(p.map, p.map_elem, ((int64_t)bh * p.Mq + I) * p.Nk, p.Nk, jmax, bn_log2, L, causal != 0,
                                       (int64_t)I * p.bm, ids, tdesc, s_cnt, s_ioff, s_toff, s_wcnt);

  KvSource kvs;
  kvs.k0 = (const char*)(p.k + b * p.k_sb + hk * p.k_sh);
  kvs.v0 = (const char*)(p.v + b * p.v_sb + hk * p.v_sh);
  kvs.kp = (const char*)p.kp; kvs.vp = (const char*)p.vp;
  kvs.k_strb = (uint32_t)p.k_sl * 2u; kvs.v_strb = (uint32_t)p.v_sl * 2u;
  kvs.BHkv = (int64_t)p.B * p.Hkv; kvs.bhk = (int64_t)b * p.Hkv + hk; kvs.npad = p.npad;
  kvs.bn_log2 = bn_log2; kvs.L = L;
  const uint32_t f_chunk = lt_fetch_chunk<D>(lane);
  const uint32_t r_off = lt_row_operand16<D>(l16, lg);
  uint32_t t_off[2];
  lt_tr_operand16<D>(lane, t_off);

  auto issue_tile = [&](int t, int stage) __attribute__((always_inline)) {
    TileSrc<G16> ts;
    lt_tile_src<D, G16>(kvs, tdesc, ids, t, wave, lane, ts);
    lt_issue_rows<D, G16>(smem + stage * LT_TILE, ts.kbase, ts.kstr, ts.lim, ts.src0, wave, f_chunk);
    lt_issue_rows<D, G16>(smem + (2 + stage) * LT_TILE, ts.vbase, ts.vstr, ts.lim, ts.src0, wave, f_chunk);
  };

  f32x4 acc[2][DB];
#pragma unroll
  for (int qb = 0; qb < 2; ++qb)
#pragma unroll
    for (int db = 0; db < DB; ++db) acc[qb][db] = f32x4{0.f, 0.f, 0.f, 0.f};

  // A tile is worked on in six runs of MFMAs, with the vector instructions of one half (32 keys) between the MFMAs of another run:
  //   S(0) | dP(0) + p(0) | S(1) + dS(0) | dP(1) + p(1) | dQ(0) + dS(1) | dQ(1)
  // Every A operand feeds two MFMAs (the query blocks) and is read PD pairs ahead.
  constexpr int NM = 4 * KK, NO = NM / 2, PD = 4;  // MFMAs and operands of a run
  static_assert(NO == DB, "");
  constexpr int VPS = 16 / NM;  // logits of a lane per MFMA
  auto compute_tile = [&](int t, auto stage_c) __attribute__((always_inline)) {
    constexpr int ST = decltype(stage_c)::value;
    const uint32_t d = __builtin_amdgcn_readfirstlane(tdesc[t][0]);
    const int lv = d & 3;
    PSA_LDS(unsigned char) Ks = (PSA_LDS(unsigned char))(smem) + ST * LT_TILE;
    PSA_LDS(unsigned char) Vs = (PSA_LDS(unsigned char))(smem) + (2 + ST) * LT_TILE;
    f32x4 s[2][2][2], dp[2][2][2];  // [half][query block][16-key block]
    u32x4 ds[2][2];                 // [half][query block]: B operand of dQ^T += K^T dS^T
    x8 op[6 * NO];
    auto fetch = [&](auto n_c) __attribute__((always_inline)) {
      constexpr int n = decltype(n_c)::value, run = n / NO, i = n % NO;
      if constexpr (run < 4) {  // operand i = 2 * k-step + key block
        op[n] = *(PSA_LDS(const x8))((run & 1 ? Vs : Ks) + r_off + (run >> 1) * G::HALF + (i >> 1) * 64 + (i & 1) * G::GROUP);
      } else if constexpr (run < 6) {
        PSA_LDS(unsigned char) a = Ks + t_off[i & 1] + (run - 4) * G::HALF + (i >> 1) * 64;
        const u32x2 lo = ET::read_tr(a), hi = ET::read_tr(a + G::GROUP);
        op[n] = __builtin_bit_cast(x8, u32x4{lo[0], lo[1], hi[0], hi[1]});
      }
    };
    const float nb[2] = {(float)lv + nlse2[0], (float)lv + nlse2[1]};
    // logit v (0..15) of a lane, in the order in which a run completes them: key block v >> 3, query block (v >> 2) & 1
    auto prob = [&](auto half_c, auto v_c) __attribute__((always_inline)) {
      constexpr int c = decltype(half_c)::value, v = decltype(v_c)::value, kb = v >> 3, qb = (v >> 2) & 1, e = v & 3;
      s[c][qb][kb][e] = fast_exp2(__builtin_fmaf(s[c][qb][kb][e], scale_log2, nb[qb]));
    };
    auto dsv = [&](auto half_c, auto v_c) __attribute__((always_inline)) {
      constexpr int c = decltype(half_c)::value, v = decltype(v_c)::value, kb = v >> 3, qb = (v >> 2) & 1, e = v & 3;
      dp[c][qb][kb][e] *= s[c][qb][kb][e];
      if constexpr (e & 1) ds[c][qb][kb * 2 + (e >> 1)] = ET::pack2(dp[c][qb][kb][e - 1], dp[c][qb][kb][e]);
    };
    auto mask_half = [&](auto half_c) __attribute__((always_inline)) {
      constexpr int c = decltype(half_c)::value;
      if (!(d & 4)) return;
      // Partly empty tile and/or causal diagonal: valid slots are a prefix of the tile (nvalid); a pooled key of
      // level lv is visible to query i iff src < (i + 1) >> lv.  Each run of 4 slots keeps its first `keep`.
      const int nvalid = (int)((d >> 3) & 127);
      const uint32_t d1 = __builtin_amdgcn_readfirstlane(tdesc[t][1]);
      const int cnt = (int)(d1 >> 16), lt = (int)(d >> 10), sbs_log2 = bn_log2 - lv;
      const uint16_t* lids = ids + (d1 & 0xffff);
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const int r0 = c * 32 + kb * 16 + lg * 4;
        int src0 = 0;
        if (causal) {
          const int gpos = (lt << 6) + r0;
          int bi = gpos >> sbs_log2;
          bi = bi < cnt - 1 ? bi : cnt - 1;
          src0 = ((int)lids[bi] << sbs_log2) + (gpos & ((1 << sbs_log2) - 1));
        }
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) {
          int keep = nvalid - r0;
          if (causal) {
            const int vis = ((q_idx + 16 * qb + 1) >> lv) - src0;
            keep = keep < vis ? keep : vis;
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) s[c][qb][kb][e] = e < keep ? s[c][qb][kb][e] : -INFINITY;
        }
      }
    };
    static_for<PD>([&](auto n) __attribute__((always_inline)) { fetch(n); });
    static_for<6>([&](auto run_c) __attribute__((always_inline)) {
      constexpr int run = decltype(run_c)::value;
      if constexpr (run < 4) {
        auto& x = run & 1 ? dp[run >> 1] : s[run >> 1];
#pragma unroll
        for (int qb = 0; qb < 2; ++qb)
#pragma unroll
          for (int kb = 0; kb < 2; ++kb) {
            const float v = run & 1 ? ndelta[qb] : 0.f;
            x[qb][kb] = f32x4{v, v, v, v};
          }
      }
      __builtin_amdgcn_sched_barrier(0);
      static_for<NM>([&](auto st_c) __attribute__((always_inline)) {
        constexpr int st = decltype(st_c)::value, i = st >> 1, qb = st & 1, kb = i & 1, n = run * NO + i;
        if constexpr (run < 4) {
          constexpr int c = run >> 1;
          if constexpr (run & 1) dp[c][qb][kb] = ET::mfma16(op[n], dof[qb][i >> 1], dp[c][qb][kb]);
          else s[c][qb][kb] = ET::mfma16(op[n], qf[qb][i >> 1], s[c][qb][kb]);
        } else {
          acc[qb][i] = ET::mfma16(op[n], __builtin_bit_cast(x8, ds[run - 4][qb]), acc[qb][i]);
        }
        if constexpr (qb == 1) fetch(IC<n + PD>{});
        static_for<VPS>([&](auto j) __attribute__((always_inline)) {
          constexpr int v = st * VPS + decltype(j)::value;
          if constexpr (run == 1 || run == 3) prob(IC<(run >> 1)>{}, IC<v>{});
          if constexpr (run == 2) dsv(IC<0>{}, IC<v>{});
          if constexpr (run == 4) dsv(IC<1>{}, IC<v>{});
        });
        __builtin_amdgcn_sched_barrier(0);
      });
      if constexpr (run == 0 || run == 2) mask_half(IC<(run >> 1)>{});
    });
  };

  if (T > 0) {
    // the Q / dO fragments must have arrived before the first copy is issued (a pending ordinary load would make
    // the compiler wait for all copies in flight inside the loop)
    __builtin_amdgcn_s_waitcnt(0x0f70);
    issue_tile(0, 0);
    __builtin_amdgcn_s_waitcnt(0x0f70);
    __syncthreads();
    const std::integral_constant<int, 0> S0;
    const std::integral_constant<int, 1> S1;
    for (int t = 0; t < T; t += 2) {
      // invariant: stage t&1 holds tile t, the other stage is free
      if (t + 1 < T) issue_tile(t + 1, 1);
      compute_tile(t, S0);
      __builtin_amdgcn_s_waitcnt(0x0f70);
      __syncthreads();
      if (t + 1 < T) {
        if (t + 2 < T) issue_tile(t + 2, 0);
        compute_tile(t + 1, S1);
        __builtin_amdgcn_s_waitcnt(0x0f70);
        __syncthreads();
      }
    }
  }

  __syncthreads();
  unsigned char* Os = smem;
  const float scale = p.scale;
#pragma unroll
  for (int qb = 0; qb < 2; ++qb)
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const f32x4 a = acc[qb][db];
      *(u32x2*)(Os + (wave * 32 + qb * 16 + l16) * OST + (db * 16 + lg * 4) * 2) =
          u32x2{ET::pack2(a[0] * scale, a[1] * scale), ET::pack2(a[2] * scale, a[3] * scale)};
    }
  __syncthreads();
  bf16_t* ob = p.dq + b * p.dq_sb + h * p.dq_sh;
  for (int u = tid; u < BM * CH; u += NT) {
    const int rr = u / CH, ch = u % CH;
    const int row = I * BM + rr;
    if (row < L) *(u32x4*)(ob + (int64_t)row * p.dq_sl + ch * 8) = *(const u32x4*)(Os + rr * OST + ch * 16);
  }
}

// slots of a kv-block in the dK/dV walk: one per level (a level-0 block of 128 keys is one slot of 128 keys)
constexpr int DKDV_SLOTS = 4;

// ------------------------------------------------------------------------------------------------------
// Longest-columns-first order for the dK/dV walk.  A workgroup's work is the number of q-blocks that retain its
// kv-block at its level, which varies a lot (a few key blocks are kept by every query block); issuing the
// workgroups by decreasing work removes the tail of the launch.  Results do not depend on the order.
// ------------------------------------------------------------------------------------------------------
constexpr int COL_BINS = psa_order::COST_BINS;

// cost of a 128-key slot of n q-blocks: exact, or the octave of its length (classes, issued head by head)
__device__ __forceinline__ int wide_cost(int n, bool octaves) {
  if (octaves) return 32 - __builtin_clz(n | 1);
  return n < COL_BINS - 1 ? n : COL_BINS - 1;
}

// Costs of every walk in one launch, their sorts in another: both are latency-bound (a sort is one workgroup per share, 8 to 16
// per list) and two cost launches and three sorts one after the other left the chip nearly idle.  Measured now 9 + 12.5 us;
// training step of 48 heads x 8776 x 64 1208 -> 1198 us, of 12 heads x 32760 x 128 4549 -> 4543 us.  The first row_wgs workgroups: four rows each, costs of the dQ walk.  The others, one per
// (kv head, kv-block): per-level counts over the column -> cost of each of its slots.  The
// costs of the slots slot_lo .. of all blocks form one list per dK/dV launch; with a 128-key slot 0 that slot's costs are a list of their
// own (cost0): one cost per slot, or (halve > 0) one per half, 0 for the second one of a slot of fewer than halve q-blocks.
__global__ __launch_bounds__(256) void psa_bwd_cost_kernel(BwdParams p, int row_wgs, int32_t* cost_row, int wide0, bool octaves, int halve, int32_t* cost0, int32_t* cost) {
  __shared__ int s_n[4];
  if ((int)blockIdx.x < row_wgs) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= p.B * p.Hq * p.Mq) return;
    const int c = psa_order::row_cost(p.map, p.map_elem, row, p.Mq, p.Nk, p.bn_log2, p.bm, p.causal);
    if ((threadIdx.x & 63) == 0) cost_row[row] = c;
    return;
  }
  const int64_t blk = (int)blockIdx.x - row_wgs;
  const int J = (int)(blk % p.Nk), bhk = (int)(blk / p.Nk), b = bhk / p.Hkv, hk = bhk % p.Hkv;
  const int n_rep = p.Hq / p.Hkv, Mq = p.Mq, bn_log2 = p.bn_log2;
  if (threadIdx.x < 4) s_n[threadIdx.x] = 0;
  __syncthreads();
  int n[4] = {0, 0, 0, 0};
  for (int e = threadIdx.x; e < n_rep * Mq; e += 256) {
    const int hl = e / Mq, I = e % Mq;
    const int h = hk * n_rep + hl;
    int level = load_map(p.map, (((int64_t)b * p.Hq + h) * Mq + I) * p.Nk + J, p.map_elem);
    if (p.causal) {
      const int ce = (int)((((int64_t)(I + 1) * p.bm) + (1 << bn_log2) - 1) >> bn_log2);
      if (J >= ce) level = 0;
    }
#pragma unroll
    for (int lv = 0; lv < 4; ++lv) n[lv] += level == (1 << lv);
  }
#pragma unroll
  for (int lv = 0; lv < 4; ++lv)
    if (n[lv]) atomicAdd(&s_n[lv], n[lv]);
  __syncthreads();
  if ((int)threadIdx.x < DKDV_SLOTS) {
    const int lv = (int)threadIdx.x;
    const int c = s_n[lv] < COL_BINS - 1 ? s_n[lv] : COL_BINS - 1;
    if (!wide0) cost[blk * DKDV_SLOTS + lv] = c;
    else if (lv == 0) {
      const int n = s_n[0];
      if (halve > 0) {
        const bool cut = n >= halve;
        cost0[2 * blk] = wide_cost(cut ? (n + 1) / 2 : n, octaves);
        cost0[2 * blk + 1] = cut ? wide_cost((n + 1) / 2, octaves) : 0;
      } else {
        cost0[blk] = wide_cost(n, octaves);
      }
    }
    else cost[blk * (DKDV_SLOTS - 1) + (lv - 1)] = c;
  }
}

// ------------------------------------------------------------------------------------------------------
// 128-key slots in halves.  A few key blocks are kept by nearly every q-block, others by one or two, and a launch that the chip holds in
// one round or little more takes as long as its longest slot (16 heads of 3484 x 128 114 us beside a dQ walk of 55).  There a slot that a
// quarter of the q-blocks and more keep goes to two workgroups of 64 keys each, 16 per wave, which walk the whole list: a key's products are
// added in the same order wherever it is worked on, so a head's gradients have the same bits in any launch.
// Which launches: the whole backward with whole / halved slots, us, fixed quotas and thresholds, by the longest possible list (q-blocks of the kv head):
//   head dim 128   16 q-blocks, 384 slots 148 / 133 and 155 / 141, 640 slots 169 / 156 and 195 / 214;   26, 650 slots 213 / 194 and 242 / 250;
//                  32, 512 slots 218 / 192 and 230 / 211, 768 slots 243 / 222 and 292 / 293, 1024 slots 284 / 277 and 357 / 386;   48, 384 slots
//                  273 / 238 and 274 / 246, 768 slots 318 / 290 and 360 / 342, 960 slots 354 / 327 and 416 / 442;   71, 852 slots 449 / 408 and
//                  478 / 518;   8, 384 slots 82 / 102 and 110 / 108
//   head dim 64    16, 384 slots 103 / 97 and 107 / 103 (steps that the host bounds);   32, 768 slots 172 / 157 and 185 / 177;   48, 768 slots 232 / 210
//                  and 234 / 222, 1008 slots 227 / 210 and 261 / 262, 1200 slots 257 / 240 and 301 / 310;   125, 1000 slots 428 / 402 and 423 / 416
// In larger launches the lists of threshold maps, of which many are that long, lose more by half-filled workgroups than the tail gives.  Cut from a half
// or an eighth of the q-blocks on: 8 x 9000 x 128 350 and 326 us for 320; elsewhere within 2 %.
// (Lists cut along the q-blocks with fp32 sums in memory end sooner, 48 q-blocks of 384 slots 186 and 240, but the sums' order is then the launch's
// business, or, in the order of the parts everywhere, 1 to 12 % of large launches with fixed quotas: 48 x 2583 x 128 240 -> 270.)
// ------------------------------------------------------------------------------------------------------
int halved_slots(int D, int64_t slots, int64_t list) {  // shortest list of a halved slot; 0: none.  (The chip holds 512 / 768 workgroups of the walk at once)
  const int64_t most = D == 128 ? 768 : 1024;
  if (list < (D == 128 ? 16 : 32) || slots > (24 * list < most ? 24 * list : most)) return 0;
  return (int)(list / 4);
}

// ------------------------------------------------------------------------------------------------------
// dK/dV column walk: Q and dO rows are copied from global memory straight into LDS (double buffered, one barrier per step of 64
// query rows) in the padded + swizzled row-major tile layout of the forward kernel; the row operands (S = Q K^T, dP = dO V^T) are
// 128-bit LDS reads and the transposed operands (dV^T += dO^T P, dK^T += Q^T dS) come from the same tiles through the transposing
// LDS load.
// The 128-key slots are bound by power and the instruction port like the dQ walk, the others by the Q / dO rows that they fetch.
// At head dim 128 the accumulators and the K / V fragments take 192 of 256 registers, so that nothing of a neighbouring
// pass fits beside them; 16 x 16 x 32 MFMAs in runs by 16-row groups leave the room for the vector instructions to lie between
// the MFMAs all the same (compute_step).  Kernel before (32 x 32 x 16 MFMAs, all of a pass's exponentials between its products) and
// now: 12 heads of 32760 x 128 at 85 % sparsity, 128-key slots 1840 -> 1515 us, the others 809 -> 677 us; 48 heads of 8776 x 64
// 381 -> 262, 338 -> 280 us; training steps, with the dQ walk, 4601 -> 4196 us and 1193 -> 1071 us.
// The four waves of a workgroup split its keys and the 64 query rows of a step: 128 keys (level 0 of a 128-key
// block) = 4 key quarters, every wave takes both query halves one after the other ("wide": each Q / dO tile that is
// fetched feeds twice the arithmetic); <= 64 keys = 2 key halves x 2 query halves, combined through LDS at the end.  A wave works on 32 keys,
// two blocks of 16, in slots of more than 32 keys and on one block in smaller ones and in halves of 128: all four waves of a 32-key slot have work,
// and those of a 16-key slot compute nothing for keys that are not there.  The walk is there twice in the kernel for that, one branch at its
// start: 14 to 48 scalars are spilled before the walk and come back behind it, few of them in a step (a branch around each step spills there).  With 32 keys per wave throughout / now, the launch of the pooled levels, us: 48 heads of 17043 x
// 128, fixed quotas, 1677 / 1488, 24 of 21613 x 64 693 / 606, 48 of 8776 x 64 282 / 250, 12 of 32760 x 128, thresholds, 660 / 621.
// ------------------------------------------------------------------------------------------------------
constexpr int B_ISTR = LT_ISTR;  // bytes between the blocks of a tile

// Gradients of the replicate-pad rows L .. npad - 1, which land on the last real token: over the pooled rows behind it, each counted
// with its share of pad tokens.  By the 256 threads of the workgroup that owns that token (barriers inside), dK to fold[0 .. D) and dV to
// fold[D .. 2 D); part: 2048 floats of LDS.  One lane that walks the pad tokens of its channels, three loads each, holds up the whole
// launch: 16 heads of 3484 x 128 (100 pad tokens) 223 us, 114 without that.
template <int D>
__device__ __forceinline__ void fold_pad_rows(const BwdParams& p, int bhk, int tid, float* part, float* fold) {
  constexpr int CH = D / 4, NG = 256 / CH;
  const int c = tid % CH, g = tid / CH;
  const int64_t BH = (int64_t)p.B * p.Hkv;
  f32x4 k = {0.f, 0.f, 0.f, 0.f}, v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int l = 1; l < 4; ++l) {
    const int64_t rows = BH * p.npad + pool_row_offset(l, BH, bhk, p.npad);
    const int t0 = p.L >> l, t1 = (int)(p.npad >> l);
#pragma unroll 2
    for (int t = t0 + g; t < t1; t += NG) {
      const f32x4 x = *(const f32x4*)(p.wk + (rows + t) * D + c * 4), y = *(const f32x4*)(p.wv + (rows + t) * D + c * 4);
      const float share = t == t0 ? (float)(((t0 + 1) << l) - p.L) / (float)(1 << l) : 1.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        k[e] = __builtin_fmaf(x[e], share, k[e]);
        v[e] = __builtin_fmaf(y[e], share, v[e]);
      }
    }
  }
  f32x4* const sums = (f32x4*)part;  // [tensor][group][chunk]
  sums[tid] = k;
  sums[256 + tid] = v;
  __syncthreads();
  if (tid < 2 * CH) {
    f32x4 a = sums[(tid / CH) * 256 + tid % CH];
    for (int i = 1; i < NG; ++i) {
      const f32x4 x = sums[(tid / CH) * 256 + i * CH + tid % CH];
#pragma unroll
      for (int e = 0; e < 4; ++e) a[e] += x[e];
    }
    ((f32x4*)fold)[tid] = a;
  }
  __syncthreads();
}

// One instantiation per kind of slot (WIDE: the 128-key level-0 slot; else the slots slot_lo .. slot_lo + slot_cnt - 1 of
// every kv-block); workgroup id = ((b * Hkv + kv head) * Nk + kv-block) * slot_cnt + (slot - slot_lo), or (WIDE, halves: the halves' costs)
// ((b * Hkv + kv head) * Nk + kv-block) * 2 + half, optionally re-ordered.
// HALVES: launches with halved slots; the others keep a kernel with the one walk.
template <int D, bool WIDE, bool CAUSAL, class ET, bool HALVES = false>
__global__ __launch_bounds__(256, 2) void psa_bwd_dkdv_lds_kernel(BwdParams p, int slot_lo, int slot_cnt, int n_wg, int chunk,
                                                                 const int32_t* order, const int32_t* halves) {
  using G = LtGeom<D>;
  using x8 = typename ET::x8;
  constexpr int KK = D / 32, DB = D / 16, RPL = G::RPL;
  constexpr int B_TILE = G::TILE;
  extern __shared__ __align__(16) unsigned char smem[];
  // stage s: Q tile at 2*s*B_TILE, dO tile at (2*s + 1)*B_TILE
  PSA_LDS(float) const s_lse = (PSA_LDS(float))((PSA_LDS(unsigned char))smem + 4 * B_TILE);  // [2 stages][64]
  PSA_LDS(float) const s_del = s_lse + 128;                                                  // [2 stages][64]
  PSA_LDS(uint32_t) const qlist = (PSA_LDS(uint32_t))(s_del + 128);                          // [n_rep * Mq]  (head in group << 16 | q-block)
  const uint32_t lds0 = (uint32_t)(uintptr_t)(PSA_LDS(unsigned char))smem;
  __shared__ int s_nq;

  int wg = psa_order::dealt_entry((int)blockIdx.x, chunk);  // shares of slots per XCD, longest lists first (psa_order.h)
  if (order != nullptr) wg = order[wg];
  if (wg < 0 || wg >= n_wg) return;
  const int slot = slot_lo + wg % slot_cnt;
  int blk = wg / slot_cnt, half = 0;
  bool halved = false;
  if constexpr (HALVES) {
    blk = wg >> 1;
    half = wg & 1;
    halved = __builtin_amdgcn_readfirstlane(halves[wg | 1]) > 0;
    if (half > 0 && !halved) return;
  }
  const int J = blk % p.Nk, bhk = blk / p.Nk;
  const int b = bhk / p.Hkv, hk = bhk % p.Hkv;
  const int n_rep = p.Hq / p.Hkv;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lg = lane >> 4;
  const int L = p.L, bn_log2 = p.bn_log2, causal = p.causal, bm = p.bm, Mq = p.Mq;

  const int lv = slot;
  const int sbs = 1 << (bn_log2 - lv);            // pooled keys of this block at this level
  constexpr bool wide = WIDE;                     // 128 keys (the host launches this instantiation for such slots only)
  const int nkeys = sbs;
  const int64_t key_row0 = (int64_t)J << (bn_log2 - lv);  // first pooled row of this workgroup
  int key_valid = nkeys;                          // level 0: rows past L do not exist
  if (lv == 0) {
    const int64_t rem = (int64_t)L - key_row0;
    key_valid = rem < nkeys ? (rem > 0 ? (int)rem : 0) : nkeys;
  }
  // <= 64 keys: waves = 2 key halves x 2 query halves.  With 16 keys only one key half works: alternate
  // which pair of waves that is from workgroup to workgroup, so that all four SIMDs of a CU get work.
  // 128 keys: waves = 4 key quarters.
  const int flip = nkeys <= 16 ? (int)((blockIdx.x >> 3) & 1) : 0;
  const int kh = wide ? wave : ((wave & 1) ^ flip), qh = wide ? 0 : wave >> 1;
  const bool narrow = wide ? halved : nkeys <= 32;  // 16 keys per wave
  const int wave_key0 = (narrow ? kh * 16 : kh * 32) + half * 64;
  const bool wave_active = key_valid > wave_key0;

  // ---- list of (head in group, q-block) that retain block J at this level -------------------------
  if (wave == 0) {
    int n = 0;
    const int total = n_rep * Mq;
    for (int e0 = 0; e0 < total; e0 += 64) {
      const int e = e0 + lane;
      bool on = false;
      if (e < total) {
        const int hl = e / Mq, I = e % Mq;
        const int h = hk * n_rep + hl;
        int level = p.map ? load_map(p.map, (((int64_t)b * p.Hq + h) * Mq + I) * p.Nk + J, p.map_elem) : 1;
        if (causal) {
          const int ce = (int)((((int64_t)(I + 1) * bm) + (1 << bn_log2) - 1) >> bn_log2);
          if (J >= ce) level = 0;
        }
        on = level == (1 << lv);
      }
      const uint64_t bal = __ballot(on);
      if (on) qlist[n + __popcll(bal & ((1ull << lane) - 1ull))] = ((uint32_t)(e / Mq) << 16) | (uint32_t)(e % Mq);
      n += __popcll(bal);
    }
    if (lane == 0) s_nq = n;
  }

  auto walk = [&](auto kb_c) __attribute__((always_inline)) {
  constexpr int KB = decltype(kb_c)::value;
  // ---- this wave's keys, KB blocks of 16: K and V fragments (B operands), lane = key l16, channels 32 * kk + 8 * lg .. + 7 -----
  const int key_local = wave_key0 + l16;  // block kb: + 16 * kb
  x8 kf[KB][KK], vf[KB][KK];
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    const int key = key_local + 16 * kb;
    int64_t row = key_row0 + (key < key_valid ? key : 0);
    if (key_valid == 0) row = 0;
    const bf16_t *kp_, *vp_;
    if (lv == 0 || p.kp == nullptr) {
      // without a level map there are no pooled buffers: the workgroups of the pooled levels have an empty
      // q-block list and only write zeros, whatever they load here
      kp_ = p.k + b * p.k_sb + hk * p.k_sh + (lv == 0 ? row : 0) * p.k_sl;
      vp_ = p.v + b * p.v_sb + hk * p.v_sh + (lv == 0 ? row : 0) * p.v_sl;
    } else {
      const int64_t off = (pool_row_offset(lv, (int64_t)p.B * p.Hkv, bhk, p.npad) + row) * D;
      kp_ = p.kp + off;
      vp_ = p.vp + off;
    }
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      kf[kb][kk] = *(const x8*)(kp_ + kk * 32 + lg * 8);
      vf[kb][kk] = *(const x8*)(vp_ + kk * 32 + lg * 8);
    }
  }
  // last token that the pooled key covers (< npad); block kb: + 16 << lv
  const int key_up = (int)(((key_row0 + key_local + 1) << lv) - 1);
  __syncthreads();
  const int nq = s_nq;

  // ---- lane-invariant LDS addressing (tile layout: see the forward kernel) ---------------------------
  // copy: wave w fills the 16-row group w of both tiles; lane (fq = lane / CH, pos = lane % CH) of block n writes
  // row fq of that block, i.e. tile row 16w + RPL * fq + n, chunk pos ^ lt_key(fq)
  // (recomputed from the lane id at every use - see issue_step - instead of living in registers across the matrix work:
  // this kernel has no register to spare, and a spilled value comes back through a vmcnt wait that would also wait
  // for the tile copies in flight)
  // (qh = 0 in a wide workgroup, whose passes add HALF * query half as an immediate)
  uint32_t r_off = lt_row_operand16<D>(l16, lg) + (uint32_t)(qh * G::HALF);  // row operand: + 64 * kk + GROUP * (16-row group)
  uint32_t t_off[2];
  lt_tr_operand16<D>(lane, t_off);  // transposed operand of channel block db: t_off[db & 1] + 64 * (db >> 1)
#pragma unroll
  for (int i = 0; i < 2; ++i) t_off[i] += (uint32_t)(qh * G::HALF);

  f32x4 dk[KB][DB], dv[KB][DB];  // [key block][channel block]
#pragma unroll
  for (int kb = 0; kb < KB; ++kb)
#pragma unroll
    for (int db = 0; db < DB; ++db) dk[kb][db] = dv[kb][db] = f32x4{0.f, 0.f, 0.f, 0.f};
  const float scale_log2 = p.scale_log2;
  const float bias = (float)lv;
  const int spb_log2 = bm >> 7;      // steps of 64 query rows per q-block: 1 (block_m 64) or 2 (128)
  const int n_steps = key_valid > 0 ? nq << spb_log2 : 0;
  const uint32_t q_strb = (uint32_t)p.q_sl * 2u, do_strb = (uint32_t)p.do_sl * 2u;

  // step i -> (head, q-block, first query row)
  auto step_of = [&](int i, int& h, int& I, int& q0) __attribute__((always_inline)) {
    const uint32_t ent = qlist[i >> spb_log2];
    h = hk * n_rep + (int)(ent >> 16);
    I = (int)(ent & 0xffff);
    q0 = I * bm + (i & ((1 << spb_log2) - 1)) * 64;
  };
  // rows of step i and their -lse / -delta -> stage
  auto issue_step = [&](int i, int stage) __attribute__((always_inline)) {
    int h, I, q0;
    step_of(i, h, I, q0);
    h = __builtin_amdgcn_readfirstlane(h);
    q0 = __builtin_amdgcn_readfirstlane(q0);
    const int ln = lane_id();  // (not kept over the matrix work)
    if (wave == 0) {
      const int64_t at = ((int64_t)b * p.Hq + h) * L + q0;
      if (q0 + ln < L) {
        psa_tiles::lds_copy4((const char*)(p.nlse2 + at), (uint32_t)ln * 4u, lds0 + (uint32_t)(4 * B_TILE + stage * 256));
        psa_tiles::lds_copy4((const char*)(p.ndelta + at), (uint32_t)ln * 4u, lds0 + (uint32_t)(4 * B_TILE + 512 + stage * 256));
      } else {  // rows past L: -lse = -inf makes every p vanish
        s_lse[stage * 64 + ln] = -INFINITY;
        s_del[stage * 64 + ln] = 0.f;
      }
    }
    const char* qb = (const char*)(p.q + b * p.q_sb + h * p.q_sh);
    const char* ob = (const char*)(p.dout + b * p.do_sb + h * p.do_sh);
    const uint32_t f_chunk = lt_fetch_chunk<D>(ln);
    const int f_row = wave * 16 + lt_fetch_row<D>(ln);
    const int r0 = q0 + f_row;
    if (q0 + 64 <= L) {
      const uint32_t qo = (uint32_t)r0 * q_strb + f_chunk, oo = (uint32_t)r0 * do_strb + f_chunk;
#pragma unroll
      for (int n = 0; n < RPL; ++n) {
        psa_tiles::lds_copy16(qb + (uint64_t)(n * q_strb), qo, lds0 + (uint32_t)(2 * stage * B_TILE + (wave * RPL + n) * B_ISTR));
        psa_tiles::lds_copy16(ob + (uint64_t)(n * do_strb), oo, lds0 + (uint32_t)((2 * stage + 1) * B_TILE + (wave * RPL + n) * B_ISTR));
      }
    } else {
#pragma unroll
      for (int n = 0; n < RPL; ++n) {
        int row = r0 + n;
        row = row < L ? row : L - 1;
        row = row > 0 ? row : 0;
        psa_tiles::lds_copy16(qb, (uint32_t)row * q_strb + f_chunk, lds0 + (uint32_t)(2 * stage * B_TILE + (wave * RPL + n) * B_ISTR));
        psa_tiles::lds_copy16(ob, (uint32_t)row * do_strb + f_chunk, lds0 + (uint32_t)((2 * stage + 1) * B_TILE + (wave * RPL + n) * B_ISTR));
      }
    }
  };
  // 32 query rows x 32 keys are worked on in four runs of MFMAs, S = Q K^T | dP = dO V^T | dV^T += dO^T P | dK^T += Q^T dS.  The
  // first two go by 16-row groups, and the vector instructions of a group lie between the MFMAs half a run (p) and one and
  // a half (dS) behind its logits: of S, dP, P and dS at most 28 registers are live.  Every A operand feeds two MFMAs
  // (the key blocks) and is read PD pairs ahead: two are what the registers allow without spilling (one where the causal mask takes
  // two more; one everywhere 1646 us where two take 1583).
  PSA_LDS(const float) rows_base = (PSA_LDS(const float))(smem + 4 * B_TILE) + (qh * 32 + lg * 4);
  constexpr int PD = D == 128 && WIDE && CAUSAL ? 1 : 2;
  constexpr int NO = 2 * KK;  // operands of a run
  static_assert(NO == DB, "");
  constexpr int VPS = 4 / KK;  // logits of a lane per MFMA
  constexpr int NM = NO * KB, NV = 8 * KB;  // MFMAs of a run, logits of a lane
  auto compute_step = [&](int i) __attribute__((always_inline)) {
    int h, I, q0;
    step_of(i, h, I, q0);
    I = __builtin_amdgcn_readfirstlane(I);
    q0 = __builtin_amdgcn_readfirstlane(q0);
    const bool diag = causal && ((((int64_t)J + 1) << bn_log2) - 1 > (int64_t)I * bm);
    static_for<WIDE ? 2 : 1>([&](auto qi_c) __attribute__((always_inline)) {
      constexpr int qi = decltype(qi_c)::value;
      const int qhv = WIDE ? qi : qh;  // the query half of this pass (the lane offsets already hold qh)
      PSA_LDS(unsigned char) Qs = (PSA_LDS(unsigned char))(smem) + qi * G::HALF;
      PSA_LDS(unsigned char) Os = (PSA_LDS(unsigned char))(smem) + B_TILE + qi * G::HALF;
      PSA_LDS(const float) rows = rows_base + qi * 32;  // one lane base + immediates (group, lse / delta array)
      // lane = key column, registers = query rows: [16-row group][key block]
      f32x4 s[2][KB], dp[2][KB], l4[2];
      u32x4 pk[KB], dsk[KB];  // [key block]: P and dS, the B operands of the last two runs
      x8 op[4 * NO];
      auto fetch = [&](auto n_c) __attribute__((always_inline)) {
        constexpr int n = decltype(n_c)::value, run = n / NO, j = n % NO;
        if constexpr (run < 2) {  // operand j = KK * 16-row group + k-step
          op[n] = *(PSA_LDS(const x8))((run ? Os : Qs) + r_off + (j % KK) * 64 + (j / KK) * G::GROUP);
        } else if constexpr (run < 4) {
          PSA_LDS(unsigned char) a = (run == 2 ? Os : Qs) + t_off[j & 1] + (j >> 1) * 64;
          const u32x2 lo = ET::read_tr(a), hi = ET::read_tr(a + G::GROUP);
          op[n] = __builtin_bit_cast(x8, u32x4{lo[0], lo[1], hi[0], hi[1]});
        }
      };
      // Only the causal diagonal needs a mask: keys behind the query get p = 0 (thr: first query row of this pass, relative to
      // the lane's rows, that sees the lane's key).  Lanes whose key does not exist (the ragged end of the sequence at level 0;
      // lanes beyond the 16 keys of a level-8 block) work on a copy of the block's first key: the columns of dK^T / dV^T are
      // independent of each other and those lanes' columns are never read.
      int thr[KB] = {};
      if constexpr (CAUSAL)
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) thr[kb] = diag ? key_up + ((16 * kb) << lv) - (q0 + qhv * 32 + lg * 4) : -0x40000000;
      // logit v of a lane, in the order in which a run completes them: p = exp2(scale * s + bias - lse)
      auto prob = [&](auto v_c) __attribute__((always_inline)) {
        constexpr int v = decltype(v_c)::value, qg = v / (4 * KB), kb = (v >> 2) % KB, e = v & 3;
        float pe = fast_exp2(__builtin_fmaf(s[qg][kb][e], scale_log2, l4[qg][e]));
        if constexpr (CAUSAL) pe = thr[kb] <= qg * 16 + e ? pe : 0.f;
        s[qg][kb][e] = pe;
        if constexpr (e & 1) pk[kb][qg * 2 + (e >> 1)] = ET::pack2(s[qg][kb][e - 1], pe);
      };
      // dS = p (dP - delta)
      auto dsv = [&](auto v_c) __attribute__((always_inline)) {
        constexpr int v = decltype(v_c)::value, qg = v / (4 * KB), kb = (v >> 2) % KB, e = v & 3;
        dp[qg][kb][e] *= s[qg][kb][e];
        if constexpr (e & 1) dsk[kb][qg * 2 + (e >> 1)] = ET::pack2(dp[qg][kb][e - 1], dp[qg][kb][e]);
      };
      static_for<PD>([&](auto n) __attribute__((always_inline)) { fetch(n); });
      static_for<4>([&](auto run_c) __attribute__((always_inline)) {
        constexpr int run = decltype(run_c)::value;
        __builtin_amdgcn_sched_barrier(0);
        static_for<NM>([&](auto st_c) __attribute__((always_inline)) {
          constexpr int st = decltype(st_c)::value, j = st / KB, kb = st % KB, qg = j / KK, kk = j % KK, n = run * NO + j;
          if constexpr (run < 2 && kk == 0 && kb == 0) {
            if constexpr (run == 0) {
              static_for<KB>([&](auto x) __attribute__((always_inline)) { s[qg][decltype(x)::value] = f32x4{0.f, 0.f, 0.f, 0.f}; });
              l4[qg] = *(PSA_LDS(const f32x4))(rows + qg * 16);
              if constexpr (!WIDE)
#pragma unroll
                for (int e = 0; e < 4; ++e) l4[qg][e] += bias;
            } else {
              const f32x4 d4 = *(PSA_LDS(const f32x4))(rows + 128 + qg * 16);
              static_for<KB>([&](auto x) __attribute__((always_inline)) { dp[qg][decltype(x)::value] = d4; });
            }
          }
          if constexpr (run == 0) s[qg][kb] = ET::mfma16(op[n], kf[kb][kk], s[qg][kb]);
          if constexpr (run == 1) dp[qg][kb] = ET::mfma16(op[n], vf[kb][kk], dp[qg][kb]);
          if constexpr (run == 2) dv[kb][j] = ET::mfma16(op[n], __builtin_bit_cast(x8, pk[kb]), dv[kb][j]);
          if constexpr (run == 3) dk[kb][j] = ET::mfma16(op[n], __builtin_bit_cast(x8, dsk[kb]), dk[kb][j]);
          if constexpr (kb == KB - 1) fetch(IC<n + PD>{});
          static_for<VPS>([&](auto u) __attribute__((always_inline)) {
            constexpr int v = (run * NM + st - NM / 2) * VPS + decltype(u)::value;
            if constexpr (v >= 0 && v < NV) prob(IC<v>{});
            if constexpr (v >= NV && v < 2 * NV) dsv(IC<v - NV>{});
          });
          __builtin_amdgcn_sched_barrier(0);
        });
      });
    });
  };

  if (n_steps > 0) {
    issue_step(0, 0);
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the rows have landed
    __syncthreads();
    // One body for both stages, the lane offsets step between them: with a body per stage the last tile is out of reach of the
    // LDS reads' immediate offsets and takes further base registers.
    for (int i = 0, stage = 0; i < n_steps; ++i, stage ^= 1) {
      // invariant: the stage holds step i, the other one is free
      if (i + 1 < n_steps) issue_step(i + 1, stage ^ 1);
      if (wave_active) compute_step(i);
      __builtin_amdgcn_s_waitcnt(0x0f70);
      __syncthreads();
      const int to = stage ? -1 : 1;
      r_off += to * (2 * B_TILE);
      t_off[0] += to * (2 * B_TILE);
      t_off[1] += to * (2 * B_TILE);
      rows_base += to * 64;
    }
  }

  const int ln = lane_id();
  // ---- 128-key level-0 slot: this workgroup owns 128 tokens of dK / dV outright.  The pooled levels' launch has
  // finished, so the tokens' shares of the pooled gradients (1/l of pooled row n >> level; for the last real token
  // also those of the replicate-pad tokens behind it) are added here and dK, dV leave in the tensors' 16-bit type: no fp32 level-0
  // buffer, no separate pass.
  if constexpr (WIDE) {
    float* const fold = (float*)smem;
    const int64_t key_end = key_row0 + (half > 0 || !halved ? 128 : 64);
    const bool folds = key_end >= L && p.npad > L;  // (this workgroup owns the last token, and there are pad rows)
    if (folds) {
      __syncthreads();
      fold_pad_rows<D>(p, bhk, wave * 64 + ln, fold + 2 * D, fold);
    }
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      const int64_t n = key_row0 + wave_key0 + (ln & 15) + 16 * kb;
      if (n >= L) continue;
      const int64_t BH = (int64_t)p.B * p.Hkv, npad = p.npad;
      const float* lk[3];
      const float* lvv[3];
#pragma unroll
      for (int l = 1; l < 4; ++l) {
        const int64_t rows = BH * npad + pool_row_offset(l, BH, bhk, npad);
        lk[l - 1] = p.wk + rows * D;
        lvv[l - 1] = p.wv + rows * D;
      }
      bf16_t* dkp = p.dk + b * p.dk_sb + hk * p.dk_sh + n * p.dk_sl;
      bf16_t* dvp = p.dv + b * p.dv_sb + hk * p.dv_sh + n * p.dv_sl;
      const float scale = p.scale;
      auto contrib = [&](const float* const (&w)[3], int64_t row, int col) __attribute__((always_inline)) {
        f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int l = 1; l < 4; ++l) {
          const f32x4 x = *(const f32x4*)(w[l - 1] + (row >> l) * D + col);
          const float inv = 1.0f / (float)(1 << l);
#pragma unroll
          for (int e = 0; e < 4; ++e) a[e] += x[e] * inv;
        }
        return a;
      };
#pragma unroll
      for (int db = 0; db < DB; ++db) {
          const int col = db * 16 + (ln >> 4) * 4;
          f32x4 gk, gv = dv[kb][db];
#pragma unroll
          for (int e = 0; e < 4; ++e) gk[e] = dk[kb][db][e] * scale;
          {
            const f32x4 ak = contrib(lk, n, col), av = contrib(lvv, n, col);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              gk[e] += ak[e];
              gv[e] += av[e];
            }
          }
          if (folds && n == L - 1) {
            const f32x4 ak = *(const f32x4*)(fold + col), av = *(const f32x4*)(fold + D + col);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              gk[e] += ak[e];
              gv[e] += av[e];
            }
          }
          u32x2 ok_, ov_;
          ok_[0] = ET::pack2(gk[0], gk[1]);
          ok_[1] = ET::pack2(gk[2], gk[3]);
          ov_[0] = ET::pack2(gv[0], gv[1]);
          ov_[1] = ET::pack2(gv[2], gv[3]);
          *(u32x2*)(dkp + col) = ok_;
          *(u32x2*)(dvp + col) = ov_;
        }
    }
    return;
  }
  // ---- combine the two query halves (<= 64 keys) and write this workgroup's rows of the level buffers ----
  __syncthreads();
  f32x4* red = (f32x4*)smem;  // [2 key halves][2 tensors][KB key blocks][DB][64 lanes]
  auto red_at = [&](int tensor, int kb, int db) __attribute__((always_inline)) { return red + (((kh * 2 + tensor) * KB + kb) * DB + db) * 64 + ln; };
  if (qh == 1) {
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        *red_at(0, kb, db) = dk[kb][db];
        *red_at(1, kb, db) = dv[kb][db];
      }
  }
  __syncthreads();
  if (qh != 0) return;
  const int64_t lvl_off = pool_row_offset(lv, (int64_t)p.B * p.Hkv, bhk, p.npad);
  // level buffers: level 0 first ([BHkv, npad, D]), then levels 1..3 like the pooled K/V buffers
  const int64_t base_rows = lv == 0 ? bhk * p.npad : (int64_t)p.B * p.Hkv * p.npad + lvl_off;
  const float scale = p.scale;
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    const int key = wave_key0 + (ln & 15) + 16 * kb;
    if (key >= nkeys) continue;
    float* wk = p.wk + (base_rows + key_row0 + key) * D;
    float* wv = p.wv + (base_rows + key_row0 + key) * D;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const f32x4 rk = *red_at(0, kb, db), rv = *red_at(1, kb, db);
      f32x4 a, c2;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        a[e] = (dk[kb][db][e] + rk[e]) * scale;
        c2[e] = dv[kb][db][e] + rv[e];
      }
      *(f32x4*)(wk + db * 16 + (ln >> 4) * 4) = a;
      *(f32x4*)(wv + db * 16 + (ln >> 4) * 4) = c2;
    }
  }
  };
  if constexpr (!WIDE || HALVES) {
    if (narrow) return walk(IC<1>{});
  }
  walk(IC<2>{});
}

// ------------------------------------------------------------------------------------------------------
// un-pool: levels -> dK, dV (the tensors' 16-bit type)
// ------------------------------------------------------------------------------------------------------
template <class ET>
__global__ __launch_bounds__(256) void psa_bwd_unpool_kernel(BwdParams p, int D) {
  const int which = blockIdx.z;  // 0: dK, 1: dV
  const int bhk = blockIdx.y, b = bhk / p.Hkv, hk = bhk % p.Hkv;
  const int chunks = D >> 2;  // float4 chunks per row
  const int64_t unit = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t n = unit / chunks;
  const int c = (int)(unit % chunks);
  if (n >= p.L) return;
  const float* w = which == 0 ? p.wk : p.wv;
  const int64_t BH = (int64_t)p.B * p.Hkv, npad = p.npad;
  const float* w0 = w + (bhk * npad) * D;
  const float* wl[3];
#pragma unroll
  for (int lv = 1; lv < 4; ++lv) wl[lv - 1] = w + (BH * npad + pool_row_offset(lv, BH, bhk, npad)) * D;
  auto contrib = [&](int64_t row) {
    f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int lv = 1; lv < 4; ++lv) {
      const f32x4 x = *(const f32x4*)(wl[lv - 1] + (row >> lv) * D + c * 4);
      const float inv = 1.0f / (float)(1 << lv);
#pragma unroll
      for (int e = 0; e < 4; ++e) a[e] += x[e] * inv;
    }
    return a;
  };
  f32x4 g = *(const f32x4*)(w0 + n * D + c * 4);
  {
    const f32x4 a = contrib(n);
#pragma unroll
    for (int e = 0; e < 4; ++e) g[e] += a[e];
  }
  if (n == p.L - 1) {  // gradient of the replicate-pad rows lands on the last real token (fold_pad_rows)
#pragma unroll
    for (int lv = 1; lv < 4; ++lv) {
      const int t0 = p.L >> lv, t1 = (int)(npad >> lv);
#pragma unroll 4
      for (int t = t0; t < t1; ++t) {
        const f32x4 x = *(const f32x4*)(wl[lv - 1] + (int64_t)t * D + c * 4);
        const float share = t == t0 ? (float)(((t0 + 1) << lv) - p.L) / (float)(1 << lv) : 1.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) g[e] = __builtin_fmaf(x[e], share, g[e]);
      }
    }
  }
  bf16_t* dst = which == 0 ? p.dk + b * p.dk_sb + hk * p.dk_sh + n * p.dk_sl : p.dv + b * p.dv_sb + hk * p.dv_sh + n * p.dv_sl;
  u32x2 o;
  o[0] = ET::pack2(g[0], g[1]);
  o[1] = ET::pack2(g[2], g[3]);
  *(u32x2*)(dst + c * 4) = o;
}


}  // namespace

extern "C" int64_t psa_bwd_workspace_bytes(int B, int Hq, int Hkv, int L, int D, int block_n) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || L <= 0 || D <= 0 || block_n <= 0) return 0;
  const int64_t npad = (int64_t)((L + block_n - 1) / block_n) * block_n;
  const int64_t levels = (int64_t)B * Hkv * D * (npad + npad / 2 + npad / 4 + npad / 8);
  // + cost and issue order of the dQ rows (block_m >= 64) and of the dK/dV slots (4 per kv-block, or 3 and two halves), padded to whole shares
  const int64_t pad = 16 * psa_order::MAX_PHASES;
  const int64_t n_rows = (int64_t)B * Hq * ((L + 63) / 64), n_blocks = (int64_t)B * Hkv * ((L + block_n - 1) / block_n);
  return (2 * levels + 2 * (int64_t)B * Hq * L + 2 * (n_rows + pad) + 2 * (5 * n_blocks + 2 * pad)) * (int64_t)sizeof(float);
}

extern "C" int psa_bwd(psa_tensor4 q, psa_tensor4 k, psa_tensor4 v, const void* k_pool, const void* v_pool, const void* map,
                       int map_elem_bytes, psa_tensor4 out, psa_tensor4 dout, const float* lse, psa_tensor4 dq, psa_tensor4 dk,
                       psa_tensor4 dv, void* workspace, int B, int Hq, int Hkv, int L, int D, int block_m, int block_n,
                       float sm_scale, int causal, psa_stream_t stream) {
  PSA_REQUIRE(q.ptr && k.ptr && v.ptr && out.ptr && dout.ptr && lse && dq.ptr && dk.ptr && dv.ptr && workspace, PSA_ERR_ARG,
              "psa_bwd: null pointer");
  PSA_REQUIRE(map == nullptr || (k_pool && v_pool), PSA_ERR_ARG, "psa_bwd: pooled K/V required with a level map");
  PSA_REQUIRE(map_elem_bytes == 1 || map_elem_bytes == 4, PSA_ERR_ARG, "psa_bwd: map_elem_bytes must be 1 or 4");
  PSA_REQUIRE(B > 0 && Hq > 0 && Hkv > 0 && L > 0, PSA_ERR_ARG, "psa_bwd: B, H, L must be positive");
  PSA_REQUIRE(Hq % Hkv == 0, PSA_ERR_ARG, "psa_bwd: Hq=%d must be a multiple of Hkv=%d", Hq, Hkv);
  PSA_REQUIRE(sm_scale > 0.f, PSA_ERR_ARG, "psa_bwd: sm_scale must be positive");
  PSA_REQUIRE(D == 64 || D == 128, PSA_ERR_UNSUPPORTED, "psa_bwd: head dim %d not in {64, 128}", D);
  PSA_REQUIRE(block_m == 64 || block_m == 128, PSA_ERR_UNSUPPORTED, "psa_bwd: block_m=%d not in {64, 128}", block_m);
  PSA_REQUIRE(block_n == 32 || block_n == 64 || block_n == 128, PSA_ERR_UNSUPPORTED, "psa_bwd: block_n=%d not in {32, 64, 128}", block_n);
  const psa_tensor4* ts[8] = {&q, &k, &v, &out, &dout, &dq, &dk, &dv};
  for (int i = 0; i < 8; ++i)
    PSA_REQUIRE(((uintptr_t)ts[i]->ptr % 16 == 0) && ts[i]->stride_b % 8 == 0 && ts[i]->stride_h % 8 == 0 && ts[i]->stride_l % 8 == 0,
                PSA_ERR_UNSUPPORTED, "psa_bwd: tensors must be 16-byte aligned with strides that are multiples of 8 elements");
  PSA_REQUIRE((int64_t)L * k.stride_l * 2 < (1ll << 32) && (int64_t)L * v.stride_l * 2 < (1ll << 32), PSA_ERR_UNSUPPORTED,
              "psa_bwd: one (batch, head) slice of K/V must span less than 4 GiB");
  PSA_REQUIRE((int64_t)L * q.stride_l * 2 < (1ll << 32) && (int64_t)L * dout.stride_l * 2 < (1ll << 32), PSA_ERR_UNSUPPORTED,
              "psa_bwd: one (batch, head) slice of q / dout must span less than 4 GiB");
  const int Mq = (L + block_m - 1) / block_m, Nk = (L + block_n - 1) / block_n;
  PSA_REQUIRE(Nk <= 65535 && Mq <= 65535, PSA_ERR_UNSUPPORTED, "psa_bwd: more than 65535 blocks");
  PSA_REQUIRE((int64_t)B * Hq <= 65535, PSA_ERR_UNSUPPORTED, "psa_bwd: B*Hq too large");
  for (int i = 1; i < 8; ++i)
    PSA_REQUIRE(ts[i]->dtype == q.dtype, PSA_ERR_ARG, "psa_bwd: q, k, v, out, dout, dq, dk, dv must share one element type");
  PSA_REQUIRE(q.dtype == PSA_DTYPE_BF16 || q.dtype == PSA_DTYPE_F16, PSA_ERR_UNSUPPORTED,
              "psa_bwd: element type must be bf16 or fp16 (the pooled buffers in the same type)");
  BwdParams p;
  p.q = (const bf16_t*)q.ptr; p.k = (const bf16_t*)k.ptr; p.v = (const bf16_t*)v.ptr;
  p.o = (const bf16_t*)out.ptr; p.dout = (const bf16_t*)dout.ptr;
  p.q_sb = q.stride_b; p.q_sh = q.stride_h; p.q_sl = q.stride_l;
  p.k_sb = k.stride_b; p.k_sh = k.stride_h; p.k_sl = k.stride_l;
  p.v_sb = v.stride_b; p.v_sh = v.stride_h; p.v_sl = v.stride_l;
  p.o_sb = out.stride_b; p.o_sh = out.stride_h; p.o_sl = out.stride_l;
  p.do_sb = dout.stride_b; p.do_sh = dout.stride_h; p.do_sl = dout.stride_l;
  p.dq = (bf16_t*)dq.ptr; p.dk = (bf16_t*)dk.ptr; p.dv = (bf16_t*)dv.ptr;
  p.dq_sb = dq.stride_b; p.dq_sh = dq.stride_h; p.dq_sl = dq.stride_l;
  p.dk_sb = dk.stride_b; p.dk_sh = dk.stride_h; p.dk_sl = dk.stride_l;
  p.dv_sb = dv.stride_b; p.dv_sh = dv.stride_h; p.dv_sl = dv.stride_l;
  p.kp = (const bf16_t*)k_pool; p.vp = (const bf16_t*)v_pool;
  p.map = map; p.map_elem = map_elem_bytes; p.lse = lse;
  p.B = B; p.Hq = Hq; p.Hkv = Hkv; p.L = L; p.Mq = Mq; p.Nk = Nk;
  p.bn_log2 = psa_ilog2(block_n); p.bm = block_m;
  p.npad = (int64_t)Nk * block_n;
  p.scale = sm_scale;
  p.scale_log2 = sm_scale * 1.4426950408889634f;
  p.causal = causal ? 1 : 0;
  p.max_tiles = psa_tiles::max_tiles(Nk, block_n);
  const int64_t levels = (int64_t)B * Hkv * D * (p.npad + p.npad / 2 + p.npad / 4 + p.npad / 8);
  p.wk = (float*)workspace;
  p.wv = p.wk + levels;
  p.ndelta = p.wv + levels;
  p.nlse2 = p.ndelta + (int64_t)B * Hq * L;
  hipStream_t st = (hipStream_t)stream;

  auto run = [&](auto et) -> int {
  using ET = decltype(et);
  // 1. -delta, -lse2
  {
    const int rows_per_wg = 256 / (D / 8);
    dim3 grid((unsigned)((L + rows_per_wg - 1) / rows_per_wg), (unsigned)(B * Hq));
    if (D == 128) hipLaunchKernelGGL((psa_bwd_delta_kernel<128, ET>), grid, dim3(256), 0, st, p);
    else hipLaunchKernelGGL((psa_bwd_delta_kernel<64, ET>), grid, dim3(256), 0, st, p);
    const int rc = psa_check_launch("psa_bwd (delta)");
    if (rc != PSA_OK) return rc;
  }
  // 2. issue orders of the dQ rows and of the two lists of dK/dV slots: one launch for the costs, one for the sorts.  (Costs and
  // orders live behind nlse2 in the workspace; every list is padded to whole shares.)  The dK/dV slots are the 128-key level-0 slots
  // (if block_n = 128) and the other slots.
  const int64_t total = (int64_t)B * Hq * Mq, n_blocks = (int64_t)B * Hkv * Nk;
  const bool wide0 = block_n > 64;
  const bool cols_ordered = map != nullptr && n_blocks > 8;
  const int halve = cols_ordered && wide0 ? halved_slots(D, n_blocks, (int64_t)(Hq / Hkv) * Mq) : 0;
  const int64_t n_wide = wide0 ? (halve > 0 ? 2 * n_blocks : n_blocks) : 0, n_rest = n_blocks * (wide0 ? DKDV_SLOTS - 1 : DKDV_SLOTS);
  PSA_REQUIRE(total < (1ll << 28) && 4 * n_blocks < (1ll << 28), PSA_ERR_UNSUPPORTED, "psa_bwd: too many workgroups");
  // shares by the K/V rows (dQ) and the Q/dO rows (dK/dV) that the walks stream
  const double kv_bytes = 2.0 * B * Hkv * (double)p.npad * D * 2.0 * (map != nullptr ? 1.875 : 1.0);
  const double qdo_bytes = 2.0 * B * Hq * (double)L * D * 2.0;
  int chunk, groups, chunk_w = 1, groups_w = 8, chunk_r, groups_r;
  psa_order::deal(total, kv_bytes, B * Hkv, chunk, groups);
  if (wide0) psa_order::deal(n_wide, qdo_bytes, B * Hkv, chunk_w, groups_w);
  psa_order::deal(n_rest, qdo_bytes, B * Hkv, chunk_r, groups_r);
  const int32_t *order = nullptr, *order_wide = nullptr, *order_rest = nullptr;
  const int32_t* halves = nullptr;
  const bool rows_ordered = map != nullptr && total > 8 * 32;
  if (rows_ordered || cols_ordered) {
    int32_t* cost = (int32_t*)(p.nlse2 + (int64_t)B * Hq * L);
    int32_t* ord = cost + total;
    int32_t* cost_r = cost + 2 * total + 16 * psa_order::MAX_PHASES;
    int32_t* cost_w = cost_r + n_rest;
    int32_t* ord_w = cost_w + n_wide;
    int32_t* ord_r = ord_w + (wide0 ? (int64_t)chunk_w * groups_w : 0);
    const int row_wgs = rows_ordered ? (int)((total + 3) / 4) : 0;
    // Where the Q / dO rows of a head group are about the size of an XCD's L2 (4 MiB), the 128-key slots of a share are issued in
    // classes, an octave of their list's length each, head by head inside a class (the sort is stable): an XCD then works on one
    // or two heads at a time and finds their rows in L2, where the exact longest-first order mixes all heads of the share; the
    // few long columns still go first, and what is left for the end is short.  The launch in classes of a quarter of the longest possible list /
    // of an octave, us: 24 x 21613 x 64 580 / 533, 24 x 12001 x 64 224 / 213 and 312 / 303 (fixed quotas, thresholds), 48 x 8776 x 64 236 / 235
    // and 380 / 365, 12 x 10700 x 128 302 / 275.  In exact order / classes of a quarter, training steps: 48 heads x 8776 x 64 1195 / 1160 us,
    // 24 x 12001 x 64 1028 / 999, 24 x 9000 x 128 1640 / 1601 (4.4 MiB), 12 x 10700 x 128 1013 / 983 (5.2 MiB).  Past the line the
    // rows do not fit (the launch, exact / octaves): 24 x 23000 x 64 (5.6 MiB) 655 / 669, 24 x 30000 x 64 (7.3 MiB) 962 / 982 and 1118 / 1173,
    // 16 x 16000 x 128 (7.8 MiB) 404 / 410 and 542 / 557.  With fewer slots than the
    // chip holds at once (512 or 768) only the tail counts: 12 x 4000 x 64 311 / 319; columns of fewer than 32
    // q-blocks leave classes of a few: 48 x 3000 x 128 727 / 740.
    // (shares of about one round, which also keep an XCD on one head, lose 3-5 % at 24 x 12001 x 64 and 32 x 6000 x 128)
    const bool by_head = wide0 && qdo_bytes / (B * Hkv) <= 5.5 * 1024 * 1024 && n_blocks > 768 && Hq / Hkv * Mq >= 32;
    hipLaunchKernelGGL(psa_bwd_cost_kernel, dim3((unsigned)(row_wgs + (cols_ordered ? n_blocks : 0))), dim3(256), 0, st, p, row_wgs, cost,
                       wide0 ? 1 : 0, by_head, halve, cost_w, cost_r);
    if (int e = psa_check_launch("psa_bwd (cost)")) return e;
    if (halve > 0) halves = cost_w;
    psa_order::sort_lists<3>({{{cost, ord, (int)total, chunk, rows_ordered ? groups : 0},
                               {cost_w, ord_w, (int)n_wide, chunk_w, cols_ordered && wide0 ? groups_w : 0},
                               {cost_r, ord_r, (int)n_rest, chunk_r, cols_ordered ? groups_r : 0}}}, st);
    if (int e = psa_check_launch("psa_bwd (order)")) return e;
    if (rows_ordered) order = ord;
    if (cols_ordered) {
      if (wide0) order_wide = ord_w;
      order_rest = ord_r;
    }
  }
  // 3. dQ
  {
    auto launch = [&](auto kern, size_t tile_bytes, int nw) -> int {
      const size_t shmem = tile_bytes + (size_t)p.max_tiles * 8 + (size_t)Nk * 2;
      if (shmem > 160 * 1024) return PSA_ERR_UNSUPPORTED;
      if (shmem > 48 * 1024 && hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem) != hipSuccess)
        return PSA_ERR_LAUNCH;
      hipLaunchKernelGGL(kern, dim3((unsigned)(chunk * groups)), dim3(nw * 64), shmem, st, p, chunk, order);
      return PSA_OK;
    };
    int rc;
    if (D == 128 && block_m == 128) rc = launch(psa_bwd_dq_lds_kernel<128, 4, ET>, (size_t)4 * LtGeom<128>::TILE, 4);
    else if (D == 128) rc = launch(psa_bwd_dq_lds_kernel<128, 2, ET>, (size_t)4 * LtGeom<128>::TILE, 2);
    else if (block_m == 128) rc = launch(psa_bwd_dq_lds_kernel<64, 4, ET>, (size_t)4 * LtGeom<64>::TILE, 4);
    else rc = launch(psa_bwd_dq_lds_kernel<64, 2, ET>, (size_t)4 * LtGeom<64>::TILE, 2);
    PSA_REQUIRE(rc == PSA_OK, rc, "psa_bwd: sequence too long for the on-chip schedule (LDS)");
    rc = psa_check_launch("psa_bwd (dQ)");
    if (rc != PSA_OK) return rc;
  }
  // 4. dK, dV per level: the 128-key level-0 slots (if block_n = 128) in one launch, the other slots in a second one
  {
    const int n_rep = Hq / Hkv;
    size_t shmem = (size_t)4 * (D == 128 ? LtGeom<128>::TILE : LtGeom<64>::TILE) + 256 * sizeof(float) + (size_t)n_rep * Mq * 4;
    const size_t red = (size_t)2 * 2 * (D / 32) * 16 * 64 * sizeof(float);
    if (shmem < red) shmem = red;
    PSA_REQUIRE(shmem <= 160 * 1024, PSA_ERR_UNSUPPORTED, "psa_bwd: too many q-blocks for the on-chip lists (LDS)");
    auto launch = [&](auto kern, int64_t n_wg, int chunk, int groups, int slot_lo, int slot_cnt, const int32_t* order) -> int {
      if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem) != hipSuccess) return PSA_ERR_LAUNCH;
      hipLaunchKernelGGL(kern, dim3((unsigned)(chunk * groups)), dim3(256), shmem, st, p, slot_lo, slot_cnt, (int)n_wg, chunk, order, halves);
      return PSA_OK;
    };
    // the pooled levels first: the 128-key level-0 launch adds their rows to its own and writes dK, dV
    const int lo = wide0 ? 1 : 0;
    int rl;
    if (causal)
      rl = D == 128 ? launch(psa_bwd_dkdv_lds_kernel<128, false, true, ET>, n_rest, chunk_r, groups_r, lo, DKDV_SLOTS - lo, order_rest)
                    : launch(psa_bwd_dkdv_lds_kernel<64, false, true, ET>, n_rest, chunk_r, groups_r, lo, DKDV_SLOTS - lo, order_rest);
    else
      rl = D == 128 ? launch(psa_bwd_dkdv_lds_kernel<128, false, false, ET>, n_rest, chunk_r, groups_r, lo, DKDV_SLOTS - lo, order_rest)
                    : launch(psa_bwd_dkdv_lds_kernel<64, false, false, ET>, n_rest, chunk_r, groups_r, lo, DKDV_SLOTS - lo, order_rest);
    PSA_REQUIRE(rl == PSA_OK, rl, "psa_bwd: cannot reserve %zu bytes of LDS", shmem);
    if (int e = psa_check_launch("psa_bwd (dK/dV)")) return e;
    if (wide0) {
      auto launch_wide = [&](auto halves_c) {
        constexpr bool H = decltype(halves_c)::value;
        if (causal)
          return D == 128 ? launch(psa_bwd_dkdv_lds_kernel<128, true, true, ET, H>, n_wide, chunk_w, groups_w, 0, 1, order_wide)
                          : launch(psa_bwd_dkdv_lds_kernel<64, true, true, ET, H>, n_wide, chunk_w, groups_w, 0, 1, order_wide);
        return D == 128 ? launch(psa_bwd_dkdv_lds_kernel<128, true, false, ET, H>, n_wide, chunk_w, groups_w, 0, 1, order_wide)
                        : launch(psa_bwd_dkdv_lds_kernel<64, true, false, ET, H>, n_wide, chunk_w, groups_w, 0, 1, order_wide);
      };
      rl = halves != nullptr ? launch_wide(std::true_type{}) : launch_wide(std::false_type{});
      PSA_REQUIRE(rl == PSA_OK, rl, "psa_bwd: cannot reserve %zu bytes of LDS", shmem);
      return psa_check_launch("psa_bwd (dK/dV, 128-key slots)");
    }
  }
  // 5. un-pool (blocks of 64 or 32 keys: every level went to the fp32 buffers)
  {
    const int64_t units = (int64_t)L * (D / 4);
    dim3 grid((unsigned)((units + 255) / 256), (unsigned)(B * Hkv), 2);
    hipLaunchKernelGGL(psa_bwd_unpool_kernel<ET>, grid, dim3(256), 0, st, p, D);
  }
  return psa_check_launch("psa_bwd (un-pool)");
  };
  int rc = PSA_ERR_ARG;
  psa_dispatch16(q.dtype, [&](auto et) { rc = run(et); });
  return rc;
}
