// Antidiagonal ("xattn") block-importance estimator used by the causal Qwen2.5-VL path.
//
//   A[m, n]   = sum_{i < S} q[m S + S-1-i] . k[n S + i]                 (S = stride; m, n index groups of S tokens)
//   z[m, n]   = A[m, n] * log2(e) / (sqrt(D) * S);  causal: only n <= m + (Nr - Mr)
//   P[m, :]   = softmax_2(z[m, :])                                       (base-2 softmax over all strided keys)
//   Est[I, J] = sum_{m in I, n in J} P[m, n]                             (I, J: blocks of block/S strided rows)
//
// A is a plain NT GEMM of Q' [Mr, S*D] (the S rows of a group concatenated in reverse order) with
// K' [Nr, S*D] (K viewed with S rows per line), i.e. MFMA-bound: 2*Mr*Nr*S*D flops (half under causality).
// Kernel 1: 256 (m) x 256 (n) output tiles, 4 waves of 128 x 128 (small launches: 128 x 128 tiles, see xattn_small); both operands go
// from global memory straight into double-buffered LDS (buffer_load_dwordx4 .. lds, the padded + swizzled 64-row tile layout of
// psa_tiles.h) in stages of 64 contraction elements, i.e. half a head-dim row of one of the S interleaved
// tokens; the transposed product (rows = n, lanes = m) makes part of the reductions over n in-lane.  A 256 x 256 tile needs 32 bytes of
// copies per CU cycle at the full MFMA rate (the path delivers 64; a 128 x 128 tile would need all of it).
// What bounds it: MFMAs (0.57 of the cycles at 28 heads x 32768 tokens, stride 8) at the clock that the board's power leaves (1.63 - 1.86 GHz),
// the epilogue, 256 exponentials and about 1500 other vector instructions per lane and tile with nothing beside them (a fifth of a
// tile), and copies that are still in flight at a stage's barrier (a seventh).  A wave of 128 x 128 reads 0.25 operands from LDS per MFMA; the 8
// waves of 64 x 128 before it read 0.375, met at a barrier with no operand in registers (0.48 of the cycles), and each tile began
// with its first copies: contraction alone 512 -> 435, 561 -> 509 us by card (0.94 - 1.11 PFLOP/s of the products under the diagonal,
// 0.06 more with the tiles' padding), with the reduction 581 -> 490, 567 -> 511; 12001 tokens 107 -> 85, 8192 48 -> 43, 2345 21.8 -> 16.6, 16 heads x 12000 67 -> 53, 12 x 1500, stride 16, 32 -> 21.5.
// Taken back: the tiles of four tile rows column by column, so that an XCD works on a block of the output (32768 tokens 491 -> 484, 16384
// 126 -> 132).
// The epilogue reduces each (row m, key block J) to a pair
// (local max, sum of exp2(z - local max)) in an fp32 workspace laid out [J][m] - the logits never
// reach HBM.  Kernel 2 (HBM-bound): per row the global max and denominator from the pairs, then the
// block sums.  Rows / keys past the real length are zero vectors (zero padding to `chunk` tokens); padded
// keys are not masked (logit 0), padded query rows contribute 0.
#include <type_traits>

#include "psa_common.h"
#include "psa_level_map_row.h"
#include "psa_pool_rows.h"
#include "psa_schedule.h"
#include "psa_tiles.h"

namespace {

constexpr int KC = 64;                       // contraction chunk
using XG = psa_tiles::LtGeom<KC>;            // LDS tiles: 64 rows of KC values
constexpr int X_TILE = XG::TILE, X_ISTR = psa_tiles::LT_ISTR;
// A workgroup's output tile: 2 x 2 waves, each 16 * NC rows (m) x 16 * NA keys (n) in accumulators of 16 x 16.
template <int NA_, int NC_, int PER_CU_>
struct XTile {
  static constexpr int NA = NA_, NC = NC_, PER_CU = PER_CU_;       // PER_CU: workgroups per CU
  static constexpr int TM = 32 * NC, TN = 32 * NA;
  static constexpr int QT = TM / 64, KT = TN / 64;                 // Q and K tiles per stage
  static constexpr int STAGE = (QT + KT) * X_TILE;                 // bytes per stage
  static constexpr int GPW = QT + KT;                              // 16-row groups copied per wave
  static_assert(QT == KT && NA % 4 == 0 && NC % 4 == 0, "two waves copy Q, two K");
};
using XLarge = XTile<8, 8, 1>;  // 256 x 256, 256 accumulator registers per lane, one wave per SIMD
using XSmall = XTile<4, 4, 2>;  // 128 x 128
constexpr int X_BUFS = 2;    // stages in LDS
constexpr int X_CUS_PER_XCD = 32;

struct XParams {
  const bf16_t *q, *k;
  int64_t q_sb, q_sh, q_sl, k_sb, k_sh, k_sl;
  float* ws;      // [B*Hq][NB][Mr][2]
  float* est;     // [B*Hq][out_rows][out_cols]
  int Hq, Hkv, Lq, Lk, D, S_log2, rb_log2;
  int Mr, Nr, NB;  // strided rows / keys (padded), key blocks
  int off;         // causal offset in strided units (Nr - Mr)
  int causal;
  int real_rows;   // strided query rows with real data
  int out_rows, out_cols;
  float scale2;
  int tiles_m, tiles_n, act_per_bh, n_active, per_xcd;  // output tiles; those with visible keys per (batch, head) / in all / per XCD
  int slots;  // workgroups per XCD
};

// output tiles of tile row tm that contain visible keys
template <class X>
__host__ __device__ inline int tiles_in_row(int tm, int tiles_n, int causal, int off) {
  if (!causal) return tiles_n;
  const int last_n = (tm + 1) * X::TM - 1 + off;  // last visible strided key of the row's last query
  const int n = last_n / X::TN + 1;
  return n < tiles_n ? n : tiles_n;
}

// Pooling (and similarity cap) as further workgroups of a contraction with small tiles: both only read K, the contraction leaves CUs
// idle there, and the launches of the two passes are as long as their work (28 heads x 2345 tokens: 18 + 4
// + 5 -> 19 us).
struct PoolPart {
  PoolParams p;
  int first, nx, heads;  // first workgroup; workgroups per (tensor, head); heads
};

// 16 bytes per lane of the buffer `desc` at byte offset voff + soff into LDS at lds + off + 16 * lane (bytes past its records: zeros).
__device__ __forceinline__ void lds_copy16_buffer(u32x4 desc, uint32_t voff, uint32_t soff, uint32_t lds, int off) {
#pragma unroll
  for (int i = 0; i < 4; ++i) desc[i] = __builtin_amdgcn_readfirstlane(desc[i]);
  lds = __builtin_amdgcn_readfirstlane(lds);
  soff = __builtin_amdgcn_readfirstlane(soff);
  uint32_t at;
  // (the offset in one vector register: the range check leaves a scalar one out)
  asm volatile("s_add_u32 m0, %1, %5\n\tv_add_u32 %0, %2, %3\n\tbuffer_load_dwordx4 %0, %4, 0 offen lds"
               : "=&v"(at)
               : "s"(lds), "s"(soff), "v"(voff), "s"(desc), "i"(off)
               : "memory", "scc", "m0");
}
// v_max3_f32 as such: of fmaxf the compiler makes the NaNs of an MFMA's results canonical first, an instruction per value
__device__ __forceinline__ float max3_raw(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// a of the lanes' own and of the neighbouring 16 lanes, b likewise: the even 16-lane rows return max / sum for a, the odd ones for b
template <bool SUM>
__device__ __forceinline__ float pair16(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), false, false);
  const uint32_t r0 = r[0], r1 = r[1];  // r0 = rows (a0, b0, a2, b2), r1 = (a1, b1, a3, b3)
  const float x = __builtin_bit_cast(float, r0), y = __builtin_bit_cast(float, r1);
  return SUM ? x + y : fmaxf(x, y);
}
// ... between the half-waves: lanes 0 - 31 return it for a, lanes 32 - 63 for b
template <bool SUM>
__device__ __forceinline__ float pair32(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), false, false);
  const uint32_t r0 = r[0], r1 = r[1];
  const float x = __builtin_bit_cast(float, r0), y = __builtin_bit_cast(float, r1);
  return SUM ? x + y : fmaxf(x, y);
}
// even: the even 16-lane row of each half-wave in both of its rows; odd: the odd one
__device__ __forceinline__ void spread16(float v, float& even, float& odd) {
  const uint32_t u = __builtin_bit_cast(uint32_t, v);
  const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const uint32_t r0 = r[0], r1 = r[1];
  even = __builtin_bit_cast(float, r0);
  odd = __builtin_bit_cast(float, r1);
}

// Pairs (maximum, sum of exp2(z - maximum)) of a wave's rows m0w .. and key blocks n0w .., from its accumulators:
// acc[a][c][i] = logit of key n0w + 16 a + 4 lg + i and row m0w + 16 c + l16.  Four pairs at a time, so that after the exchanges every
// 16-lane row holds a pair of its own to store.  MASK: some key is not visible.  Both variants and both tiles give the same bits.
template <int RBL, class X, bool MASK>
__device__ __forceinline__ void xattn_pairs(f32x4 (&acc)[X::NA][X::NC], float* ws, int Mr, int m0w, int n0w, int off, float scale2, int lane) {
  const int l16 = lane & 15, lg = lane >> 4;
  constexpr int KP = RBL == 3 ? X::NA : (16 * X::NA) >> (RBL + 1);  // groups of four pairs per two row blocks
#pragma unroll
  for (int cp = 0; cp < X::NC / 2; ++cp) {
#pragma unroll
    for (int kp = 0; kp < KP; ++kp) {
      // the four lists of logits that are reduced together: RBL 3: key blocks of accumulators (a, a + 1) of one row block, two per
      // accumulator; else key blocks (2 kp, 2 kp + 1) of two row blocks
      constexpr int GB = RBL == 3 ? 1 : 1 << (RBL - 4), NE = RBL == 3 ? 2 : 4;  // accumulators per list, lists
      float z[NE][4 * GB], mx[NE];
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        const int c = RBL == 3 ? 2 * cp + (kp & 1) : 2 * cp + (e >> 1);
        const int m = m0w + 16 * c + l16;
#pragma unroll
        for (int g = 0; g < GB; ++g) {
          const int a = RBL == 3 ? 2 * (kp >> 1) + e : (2 * kp + (e & 1)) * GB + g;
          if constexpr (X::PER_CU == 1) asm volatile("" : "+a"(acc[a][c]));  // (read here: ahead of the branch between the variants all of them would not fit)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            z[e][4 * g + i] = !MASK || n0w + 16 * a + 4 * lg + i <= m + off ? acc[a][c][i] : -INFINITY;
          }
        }
        mx[e] = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4 * GB; i += 2) mx[e] = max3_raw(z[e][i], z[e][i + 1], mx[e]);
      }
      float top, ref[NE];
      if constexpr (RBL == 3) {
        top = pair16<false>(mx[0], mx[1]);
      } else {
        top = pair32<false>(pair16<false>(mx[0], mx[1]), pair16<false>(mx[2], mx[3]));
      }
      top *= scale2;
      const float r = top == -INFINITY ? 0.f : -top;
      if constexpr (RBL == 3) {
        spread16(r, ref[0], ref[1]);
      } else {
        float lo, hi;
        half_wave_swap(r, lo, hi);
        spread16(lo, ref[0], ref[1]);
        spread16(hi, ref[2], ref[3]);
      }
      float sm[NE];
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        sm[e] = fast_exp2(__builtin_fmaf(z[e][0], scale2, ref[e]));
#pragma unroll
        for (int i = 1; i < 4 * GB; ++i) sm[e] += fast_exp2(__builtin_fmaf(z[e][i], scale2, ref[e]));  // (fused in words: the same bits whatever the variant)
      }
      f32x2 pr;
      pr[0] = top;
      int J, c;
      if constexpr (RBL == 3) {
        pr[1] = pair16<true>(sm[0], sm[1]);
        J = (n0w >> 3) + 2 * (2 * (kp >> 1) + (lg & 1)) + (lg >> 1);
        c = 2 * cp + (kp & 1);
      } else {
        pr[1] = pair32<true>(pair16<true>(sm[0], sm[1]), pair16<true>(sm[2], sm[3]));
        J = (n0w >> RBL) + 2 * kp + (lg & 1);
        c = 2 * cp + (lg >> 1);
      }
      *(f32x2*)(ws + ((int64_t)J * Mr + m0w + 16 * c + l16) * 2) = pr;
      if (X::PER_CU == 1 && (kp & 1)) __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// acc += a * b.  With 256 accumulator registers per lane the compiler has no spare one, and moves accumulators about between
// the MFMAs (about every second one, with the waits that go with it): there the instruction is written with its accumulator in place.
// What the compiler does not know then: nothing but these MFMAs may touch an accumulator between xattn_mfma_begin and _end.
template <class X>
__device__ __forceinline__ void xattn_mfma(f32x4& acc, const bf16x8& a, const bf16x8& b) {
  if constexpr (X::PER_CU > 1) acc = EtBf16::mfma16(a, b, acc);
  else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}
// Zeroes the accumulators; the MFMAs may read them behind this.  (A first k-step of its own, without the zeros, spills.)
template <class X>
__device__ __forceinline__ void xattn_mfma_begin(f32x4 (&acc)[X::NA][X::NC]) {
#pragma unroll
  for (int a = 0; a < X::NA; ++a)
#pragma unroll
    for (int c = 0; c < X::NC; ++c) {
      acc[a][c] = f32x4{0.f, 0.f, 0.f, 0.f};
      if constexpr (X::PER_CU == 1) asm volatile("" : "+a"(acc[a][c]));
    }
  if constexpr (X::PER_CU == 1) asm volatile("s_nop 7");
}
// The results may be read behind this: the last MFMA (4 passes) has been over for long.
template <class X>
__device__ __forceinline__ void xattn_mfma_end(f32x4 (&acc)[X::NA][X::NC]) {
  asm volatile("s_nop 15\n\ts_nop 15");
#pragma unroll
  for (int a = 0; a < X::NA; ++a)
#pragma unroll
    for (int c = 0; c < X::NC; ++c) {
      if constexpr (X::PER_CU == 1) asm volatile("" : "+a"(acc[a][c]));
      else asm volatile("" : "+v"(acc[a][c]));
    }
}
// RBL: log2 of the strided keys per block; ROWS: rows of Q or K overlap in memory (strides below the head dim)
template <int RBL, class X, bool POOL, bool ROWS>
__global__ __launch_bounds__(256, X::PER_CU) void psa_xattn_gemm_kernel(XParams p, PoolPart pool) {
  constexpr int TM = X::TM, TN = X::TN, X_QT = X::QT, X_STAGE = X::STAGE, GPW = X::GPW, NA = X::NA, NC = X::NC;
  extern __shared__ __align__(16) unsigned char smem[];  // X_BUFS stages of [Q tiles | K tiles]
  // Workgroup ids go round-robin over the 8 XCDs and every XCD runs its ids in order.  The output tiles with
  // visible keys are listed (batch-head, tile row, tile column) and the list is cut into 8 contiguous shares, one
  // per XCD: all tiles cost the same, so the XCDs finish together, and the ~32 tiles an XCD works on at a time
  // are neighbours that find each other's Q and K rows in its L2.  Workgroup `slot` of an XCD takes tiles slot, slot + slots, ..
  if constexpr (POOL) {
    if ((int)blockIdx.x >= pool.first) {
      const int u = (int)blockIdx.x - pool.first, w = u / pool.nx;
      pool_rows<false, true, Pool16<EtBf16>>(pool.p, u % pool.nx, w % pool.heads, w / pool.heads, pool.heads);
      return;
    }
  }
  const int xcd = blockIdx.x & 7, share0 = xcd * p.per_xcd;
  int share1 = share0 + p.per_xcd;
  share1 = share1 < p.n_active ? share1 : p.n_active;
  int idx = share0 + (int)(blockIdx.x >> 3);
  if (idx >= share1) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lg = lane >> 4;
  const int wn = wave & 1, wm = wave >> 1;  // wave tile: rows m0 + 16 * NC * wm .., keys n0 + 16 * NA * wn ..
  const int S = 1 << p.S_log2;
  const int dc_log2 = p.D == 2 * KC ? 1 : 0;  // 64-channel chunks per row: 1 (D = 64) or 2 (D = 128)
  const int real_stages = S << dc_log2, stages = real_stages < 2 ? 2 : real_stages;  // (a second one of zeros: a tile spans both buffers)

  // copies: waves 0, 1 move the Q rows of a stage, waves 2, 3 the K rows: GPW groups of 16 rows, of which a lane fetches the RPL
  // consecutive ones from frow on; a row is one strided index (S tokens apart in memory).  They go through a buffer descriptor of the
  // (batch, head) slice, whose range check answers rows past the real length with zeros: every tile takes the same path, and a copy is a
  // scalar and a vector instruction beside the load.
  constexpr int RPL = XG::RPL;
  const bool is_q = wave < 2;
  const uint32_t f_chunk = psa_tiles::lt_fetch_chunk<KC>(lane);
  const int frow = psa_tiles::lt_fetch_row<KC>(lane);
  const uint32_t strb = (uint32_t)(is_q ? p.q_sl : p.k_sl) * 2u, rstr = strb << p.S_log2;
  const int limit = is_q ? p.Lq : p.Lk;
  const uint32_t slice_bytes = (uint32_t)(limit - 1) * strb + (uint32_t)p.D * 2u;
  const uint32_t dst0 = psa_tiles::lds_addr_of(smem) + wave * GPW * XG::GROUP;  // (the tiles of a stage follow each other without a gap)

  // a tile, and what this wave's copies of it need
  struct Tile {
    int bh, m0, n0;
    u32x4 desc;     // the slice of Q or K; no records: nothing to copy
    uint32_t voff;  // byte offset of the lane's first row, token 0 of the S, contraction chunk 0
    int row0;       // its strided index (ROWS)
  };
  auto locate = [&](int at) __attribute__((always_inline)) {
    Tile t;
    t.bh = at / p.act_per_bh;
    int tn = at % p.act_per_bh, tm = 0;
    for (;; ++tm) {
      const int row_n = tiles_in_row<X>(tm, p.tiles_n, p.causal, p.off);
      if (tn < row_n) break;
      tn -= row_n;
    }
    t.m0 = tm * TM;
    t.n0 = tn * TN;
    const int h = t.bh % p.Hq, b = t.bh / p.Hq;
    const char* slice = is_q ? (const char*)(p.q + b * p.q_sb + h * p.q_sh) : (const char*)(p.k + b * p.k_sb + (h / (p.Hq / p.Hkv)) * p.k_sh);
    const uint64_t a = (uint64_t)(uintptr_t)psa_tiles::uniform_ptr(slice);
    t.desc = u32x4{(uint32_t)a, (uint32_t)(a >> 32) & 0xffffu, slice_bytes, 0x00020000u};  // raw buffer, no stride, 32-bit data format
    t.row0 = (is_q ? t.m0 : t.n0) + (wave & 1) * (GPW * 16) + frow;
    t.voff = ((uint32_t)t.row0 << p.S_log2) * strb + f_chunk;
    return t;
  };
  // what the copies of one stage need, in scalar registers but for the lane's part
  struct Cursor {
    u32x4 desc;
    uint32_t voff, soff, lds;
    int row0, tok0;
  };
  auto cursor = [&](const u32x4& desc, uint32_t voff, int row0, int st) __attribute__((always_inline)) {
    st = __builtin_amdgcn_readfirstlane(st);
    const int i = st >> dc_log2, dc = st & ((1 << dc_log2) - 1);
    Cursor c;
    c.tok0 = is_q ? S - 1 - i : i;  // token S-1-i of every query group, token i of every key group
    c.soff = __builtin_amdgcn_readfirstlane((uint32_t)c.tok0 * strb + (uint32_t)(dc * (KC * 2)));
    c.lds = __builtin_amdgcn_readfirstlane(dst0 + (st & 1) * X_STAGE);
    c.voff = voff;
    c.row0 = row0;
    uint32_t d0 = __builtin_amdgcn_readfirstlane(desc[0]), d1 = __builtin_amdgcn_readfirstlane(desc[1]);
    uint32_t d2 = __builtin_amdgcn_readfirstlane(st < real_stages ? desc[2] : 0u), d3 = desc[3];
    // (a scalar register that the vector unit wrote may be read by a load five cycles later; the compiler does not see the loads)
    asm volatile("s_nop 4" : "+s"(d0), "+s"(d1), "+s"(d2), "+s"(d3));
    c.desc = u32x4{d0, d1, d2, d3};
    return c;
  };
  const uint32_t rstep = __builtin_amdgcn_readfirstlane(rstr);
  auto copy = [&](const Cursor& t, int u) __attribute__((always_inline)) {  // u of GPW * RPL
    const int row = 16 * (u / RPL) + u % RPL;
    if constexpr (!ROWS) {
      lds_copy16_buffer(t.desc, t.voff, t.soff + (uint32_t)row * rstep, t.lds, u * X_ISTR);
    } else {
      // (token by token: the byte after a row may belong to the next)
      const bool real = ((int64_t)(t.row0 + row) << p.S_log2) + t.tok0 < limit;
      lds_copy16_buffer(t.desc, real ? t.voff + t.soff + (uint32_t)row * rstep : 0xfffffff0u, 0, t.lds, u * X_ISTR);
    }
  };
  const uint32_t r_off = psa_tiles::lt_row_operand16<KC>(l16, lg);
  PSA_LDS(const unsigned char) const Qs = (PSA_LDS(const unsigned char))(smem) + wm * NC * XG::GROUP + r_off;
  PSA_LDS(const unsigned char) const Ks = (PSA_LDS(const unsigned char))(smem) + X_QT * X_TILE + wn * NA * XG::GROUP + r_off;

  // Operands of the k-step at hand and of the next one.  A k-step (32 channels) is NA * NC MFMAs; the next one's operands are read and,
  // in the second k-step of a stage, the copies of the stage after the next issued between them.  The barrier lies between the k-steps of a
  // stage: what the MFMAs behind it need is in registers, and the buffer whose last operands were read before it can be filled.
  // The next k-step's operands are read into registers of their own, but for the first six K ones: theirs are free once the MFMAs
  // of the operand are issued, and what is read last has to be there at the barrier.
  constexpr int NA_IN = NA - 2;  // K operands that are replaced in place
  f32x4 acc[NA][NC];
  bf16x8 bq[2][NC], ak[NA_IN], al[2][2];
  auto read_q = [&](int st, int kk, int c) __attribute__((always_inline)) {
    bq[kk][c] = *(PSA_LDS(const bf16x8))(Qs + (st & 1) * X_STAGE + c * XG::GROUP + kk * 64);
  };
  auto read_k = [&](int st, int kk, int a) __attribute__((always_inline)) {
    const bf16x8 v = *(PSA_LDS(const bf16x8))(Ks + (st & 1) * X_STAGE + a * XG::GROUP + kk * 64);
    if (a < NA_IN) ak[a] = v;
    else al[kk][a - NA_IN] = v;
  };
  // MFMAs of k-step kk, one K operand after the other, and between them, one at a time so that the matrix pipe does not run dry, the reads
  // of the next k-step's operands (stage st_r) and the copies at t.  (One body for every stage: accumulators that several
  // variants of a step hand on are moved from register to register, and spilled.)
  auto step = [&](auto kk_c, int st_r, const Cursor& t) __attribute__((always_inline)) {
    constexpr int KK = decltype(kk_c)::value, NX = NA * NC, NCP = GPW * RPL, NR = NC + 2;
    constexpr int CPS = NX / NCP;  // MFMAs per copy
    static_assert(CPS >= 2, "copies fit");
#pragma unroll
    for (int x = 0; x < NX; ++x) {
      const int a = x / NC, c = x % NC;
      xattn_mfma<X>(acc[a][c], a < NA_IN ? ak[a] : al[KK][a - NA_IN], bq[KK][c]);
      // even MFMAs: Q operands and the last two K operands; the last MFMA of an operand: its successor
      if (x % 2 == 0 && x / 2 < NR) {
        if (x / 2 < NC) read_q(st_r, KK ^ 1, x / 2);
        else read_k(st_r, KK ^ 1, NA_IN + x / 2 - NC);
      }
      if (c == NC - 1 && a < NA_IN) read_k(st_r, KK ^ 1, a);
      if (KK == 1 && x % CPS == 1) copy(t, x / CPS);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  Tile cur = locate(idx);
#pragma unroll
  for (int st = 0; st < 2; ++st) {
    const Cursor c = cursor(cur.desc, cur.voff, cur.row0, st);
#pragma unroll
    for (int u = 0; u < GPW * RPL; ++u) copy(c, u);
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
  __syncthreads();
#pragma unroll
  for (int c = 0; c < NC; ++c) read_q(0, 0, c);
#pragma unroll
  for (int a = 0; a < NA; ++a) read_k(0, 0, a);
  for (;;) {
    // the first two stages of the next tile are copied in the last two of this one, and the operands of its first k-step read in the last
    // k-step: it begins with all that it needs (behind the last tile: zeros, that nothing uses)
    idx += p.slots;
    const bool more = idx < share1;
    Tile next = cur;
    if (more) next = locate(idx);
    else next.desc[2] = 0;
    xattn_mfma_begin<X>(acc);
    int st = 0;
    do {
      const bool here = st + 2 < stages;
      u32x4 desc;
#pragma unroll
      for (int i = 0; i < 4; ++i) desc[i] = here ? cur.desc[i] : next.desc[i];
      const Cursor ahead = cursor(desc, here ? cur.voff : next.voff, here ? cur.row0 : next.row0, here ? st + 2 : st + 2 - stages);
      step(std::integral_constant<int, 0>{}, st, ahead);
      __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the copies of stage st+1 were issued a stage ago
      __syncthreads();
      step(std::integral_constant<int, 1>{}, st + 1, ahead);
    } while (++st < stages);
    xattn_mfma_end<X>(acc);
    const int m0w = cur.m0 + wm * (16 * NC), n0w = cur.n0 + wn * (16 * NA);
    float* const ws = p.ws + (int64_t)cur.bh * p.NB * p.Mr * 2;
    if (m0w < p.Mr && n0w < p.Nr) {  // (Mr and Nr are multiples of 128)
      if (p.causal && n0w + 16 * NA - 1 > m0w + p.off) xattn_pairs<RBL, X, true>(acc, ws, p.Mr, m0w, n0w, p.off, p.scale2, lane);
      else xattn_pairs<RBL, X, false>(acc, ws, p.Mr, m0w, n0w, p.off, p.scale2, lane);
    }
    if (!more) break;
    cur = next;
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);  // no copy outlives the workgroup's LDS
}

// one workgroup per (b, h, q-block): 256 threads; thread t handles key blocks t, t+256, ...
// cached != 0: the (maximum, sum) pairs of the workgroup's rows are read from the workspace once into dynamic LDS
// ([key block][row], NB * rb pairs) and the three passes below run on that copy instead of on memory.
// The row of block scores goes to dst.
__device__ __forceinline__ void xattn_reduce_row(const XParams& p, int cached, unsigned char* s_cache, int I, int bh, int tid, float* dst) {
  __shared__ float s_M[32], s_inv[32];
  __shared__ float s_big[256];
  const int rb = 1 << p.rb_log2;
  const int m0 = I * rb;
  const float* ws = p.ws + (int64_t)bh * p.NB * p.Mr * 2;
  int64_t row_stride = p.Mr;  // pairs between consecutive key blocks of one row
  int m_sub = 0;
  if (cached) {
    // a key block's rb pairs of this q-block are contiguous in the workspace: rb * 8 bytes per key block
    f32x2* c = (f32x2*)s_cache;
    const int jlim = p.causal ? (((m0 + rb - 1 + p.off) >> p.rb_log2) + 1) : p.NB;  // key blocks any row of the q-block sees
    const int jn = jlim < p.NB ? jlim : p.NB;
    // two pairs per load, four loads in flight per thread: one load after the other is a round trip to memory each (the map's
    // kernel, 28 heads x 32768 tokens, 150 -> 125 us)
    const int n2 = jn * rb >> 1, half_log2 = p.rb_log2 - 1;
    for (int u0 = tid; u0 < n2; u0 += 4 * 256) {
      f32x4 x[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        int u = u0 + e * 256;
        u = u < n2 ? u : n2 - 1;
        x[e] = *(const f32x4*)(ws + ((int64_t)(u >> half_log2) * p.Mr + m0 + 2 * (u & (rb / 2 - 1))) * 2);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int u = u0 + e * 256;
        if (u < n2) *(f32x4*)(c + 2 * u) = x[e];
      }
    }
    __syncthreads();
    ws = (const float*)s_cache;
    row_stride = rb;
    m_sub = m0;  // the copy starts at row m0: index (J * rb + (m - m0)) (never form a pointer below the array)
  }
  // pass 1: row max and denominator.  Thread (r = tid % rb, jl = tid / rb) strides over the key blocks
  // visible to row r (J <= (m + off) / rb under causality); partials are combined in a fixed order.
  const int r = tid & (rb - 1), jl = tid >> p.rb_log2, nj = 256 >> p.rb_log2;
  const int m = m0 + r;
  const int jmax = p.causal ? ((m + p.off) >> p.rb_log2) + 1 : p.NB;
  const int jend = jmax < p.NB ? jmax : p.NB;
  float M = -INFINITY;
  for (int J = jl; J < jend; J += nj) M = fmaxf(M, ws[((int64_t)J * row_stride + (m - m_sub)) * 2]);
  s_big[jl * rb + r] = M;
  __syncthreads();
  if (tid < rb) {
    float mm = -INFINITY;
    for (int j = 0; j < nj; ++j) mm = fmaxf(mm, s_big[j * rb + tid]);
    s_M[tid] = mm;
  }
  __syncthreads();
  const float Mref = s_M[r] == -INFINITY ? 0.f : s_M[r];
  float l = 0.f;
  for (int J = jl; J < jend; J += nj) {
    const f32x2 pr = *(const f32x2*)(ws + ((int64_t)J * row_stride + (m - m_sub)) * 2);
    l += pr[1] * fast_exp2(pr[0] - Mref);  // pr = (-inf, 0) for fully masked pairs: 0 * exp2(-inf) = 0
  }
  __syncthreads();
  s_big[jl * rb + r] = l;
  __syncthreads();
  if (tid < rb) {
    float ll = 0.f;
    for (int j = 0; j < nj; ++j) ll += s_big[j * rb + tid];
    const bool real = (m0 + tid) < p.real_rows;
    s_inv[tid] = (real && ll > 0.f) ? 1.0f / ll : 0.f;  // padded query rows contribute nothing
  }
  __syncthreads();
  // pass 2: Est[I, J] = sum_r sum[r, J] * exp2(max[r, J] - M_r) / l_r
  for (int J = tid; J < p.out_cols; J += 256) {
    float e = 0.f;
    for (int rr = 0; rr < rb; ++rr) {
      const int mm = m0 + rr;
      const int jm = p.causal ? ((mm + p.off) >> p.rb_log2) + 1 : p.NB;
      if (J < jm) {
        const f32x2 pr = *(const f32x2*)(ws + ((int64_t)J * row_stride + (mm - m_sub)) * 2);
        const float Mx = s_M[rr] == -INFINITY ? 0.f : s_M[rr];
        e += pr[1] * fast_exp2(pr[0] - Mx) * s_inv[rr];
      }
    }
    dst[J] = e;
  }
}

__global__ __launch_bounds__(256) void psa_xattn_reduce_kernel(XParams p, int cached) {
  extern __shared__ __align__(16) unsigned char s_cache[];
  const int I = blockIdx.x, bh = blockIdx.y;
  xattn_reduce_row(p, cached, s_cache, I, bh, (int)threadIdx.x, p.est + ((int64_t)bh * p.out_rows + I) * p.out_cols);
}

// The same, followed by the causal layer's level map of the row while its scores are in LDS, and by what ends a map row (similarity cap,
// map, tile records): one launch instead of reduction, map, cap and list, and a causal row ranks only the columns that it
// sees (a third of the comparisons).  LDS: [pairs, then scratch of the map: scratch bytes][S scores][S levels].
// 28 heads x 32768 tokens 69 + 65 + 8 + 18 -> 125 us, x 2345 tokens 5 + 5 + 4 + 4 -> 10.
__global__ __launch_bounds__(256) void psa_xattn_map_kernel(XParams p, int cached, int scratch, QwenMapParams mp, psa_sched::MapEnd end) {
  extern __shared__ __align__(16) unsigned char s_cache[];
  __shared__ int s_lists[16];
  const int I = blockIdx.x, bh = blockIdx.y, tid = threadIdx.x, S = mp.S;
  float* s_e = (float*)(s_cache + scratch);
  uint8_t* s_lv = (uint8_t*)(s_e + S);
  xattn_reduce_row(p, cached, s_cache, I, bh, tid, s_e);
  __syncthreads();
  int n = S;
  if (mp.causal && p.off == 0) {
    // (scores above the diagonal are 0; NaNs, whose place in the order depends on their sign, are ranked among all columns)
    bool nan = false;
    for (int j = tid; j <= I; j += 256) nan |= s_e[j] != s_e[j];
    if (!__syncthreads_or(nan)) n = I + 1;
  }
  qwen_map_row(mp, s_e, I, n, s_cache, tid, 256, [&](int col, int lv) __attribute__((always_inline)) { s_lv[col] = (uint8_t)lv; });
  psa_sched::end_map_row(end, s_lv, S, (int64_t)bh * S + I, bh, I, (uint16_t*)s_cache, s_lists, tid);
}

// output tiles of one (batch, head) that hold visible keys of rows below rows_used; sets the tile counts of p
template <class X>
int active_tiles(XParams& p, int rows_used) {
  p.tiles_m = (rows_used + X::TM - 1) / X::TM;
  p.tiles_n = (p.Nr + X::TN - 1) / X::TN;
  int n = 0;
  for (int tm = 0; tm < p.tiles_m; ++tm) n += tiles_in_row<X>(tm, p.tiles_n, p.causal, p.off);
  return n;
}
// Output tile of the launch.  A 128 x 128 tile is a quarter of the products at five sixths of the rate of a 256 x 256 one or less
// (copies and LDS operands per product): it pays where the large tiles leave CUs idle.  Large tiles cost by rounds of the chip (256), small
// ones, two workgroups per CU that end one by one, 0.6 of that per 512 and half a round for the end.  Contraction + reduction, 28 heads,
// stride 8, large / small in us: 2345 tokens 32 / 16.5, 6000 35 / 35, 8192 62 / 42, 12001 92 / 85, 16384 126 / 137, 32768 490 / 611; 16 heads x 12000
// 62 / 52.
bool xattn_small(int64_t n_large, int64_t n_small) {
  return (n_small + 256) * 3 < (n_large + 255) / 256 * 2560;
}

struct XGeom {
  int Lq_pad, Lk_pad, Mr, Nr, NB, MB;
};
XGeom xgeom(int Lq, int Lk, int block, int stride, int chunk) {
  XGeom g;
  g.Lq_pad = (Lq + chunk - 1) / chunk * chunk;
  g.Lk_pad = (Lk + chunk - 1) / chunk * chunk;
  g.Mr = g.Lq_pad / stride;
  g.Nr = g.Lk_pad / stride;
  g.NB = g.Lk_pad / block;
  g.MB = g.Lq_pad / block;
  return g;
}

}  // namespace

extern "C" int64_t psa_estimate_xattn_workspace_bytes(int B, int Hq, int Lq, int Lk, int block_size, int stride, int chunk_size) {
  if (B <= 0 || Hq <= 0 || Lq <= 0 || Lk <= 0 || block_size <= 0 || stride <= 0 || chunk_size <= 0) return 0;
  const XGeom g = xgeom(Lq, Lk, block_size, stride, chunk_size);
  return (int64_t)B * Hq * g.NB * g.Mr * 2 * (int64_t)sizeof(float);
}

// What psa_xattn_layer_map adds to an estimate: the level map of the layer in place of the scores
struct XattnMap {
  QwenMapParams mp;
  psa_sched::MapEnd end;
  PoolParams* pool;  // pooling and cap of the layer, run beside the contraction (pool_blocks, pool_heads) or before it by the caller
  int pool_nx, pool_heads;
};

static int xattn_run(psa_tensor4 q, psa_tensor4 k, float* est, void* workspace, int B, int Hq, int Hkv, int Lq,
                     int Lk, int D, int block_size, int stride, int chunk_size, int causal, psa_stream_t stream, XattnMap* xm) {
  PSA_REQUIRE(q.ptr && k.ptr && (est || xm) && workspace, PSA_ERR_ARG, "psa_estimate_xattn: null pointer");
  PSA_REQUIRE(B > 0 && Hq > 0 && Hkv > 0 && Lq > 0 && Lk > 0, PSA_ERR_ARG, "psa_estimate_xattn: sizes must be positive");
  PSA_REQUIRE(Hq % Hkv == 0, PSA_ERR_ARG, "psa_estimate_xattn: Hq must be a multiple of Hkv");
  PSA_REQUIRE(D == 64 || D == 128, PSA_ERR_UNSUPPORTED, "psa_estimate_xattn: head dim %d not in {64, 128}", D);
  PSA_REQUIRE(psa_is_pow2(stride) && stride <= 16, PSA_ERR_UNSUPPORTED, "psa_estimate_xattn: stride=%d must be a power of two <= 16", stride);
  PSA_REQUIRE(psa_is_pow2(block_size) && block_size % stride == 0, PSA_ERR_UNSUPPORTED, "psa_estimate_xattn: bad block_size");
  const int rb = block_size / stride;
  PSA_REQUIRE(rb == 8 || rb == 16 || rb == 32, PSA_ERR_UNSUPPORTED, "psa_estimate_xattn: block_size/stride=%d not in {8,16,32}", rb);
  PSA_REQUIRE(chunk_size % (128 * stride) == 0, PSA_ERR_UNSUPPORTED, "psa_estimate_xattn: chunk_size must be a multiple of 128*stride");
  PSA_REQUIRE(((int64_t)Lq + chunk_size) * q.stride_l * 2 < (1ll << 32) && ((int64_t)Lk + chunk_size) * k.stride_l * 2 < (1ll << 32),
              PSA_ERR_UNSUPPORTED, "psa_estimate_xattn: one (batch, head) slice of Q/K must span less than 4 GiB");
  PSA_REQUIRE(Lk >= Lq, PSA_ERR_ARG, "psa_estimate_xattn: Lk must not be shorter than Lq");
  PSA_REQUIRE(((uintptr_t)q.ptr % 16 == 0) && ((uintptr_t)k.ptr % 16 == 0) && q.stride_l % 8 == 0 && k.stride_l % 8 == 0 &&
                  q.stride_h % 8 == 0 && k.stride_h % 8 == 0 && q.stride_b % 8 == 0 && k.stride_b % 8 == 0,
              PSA_ERR_UNSUPPORTED, "psa_estimate_xattn: tensors must be 16-byte aligned with strides multiple of 8");
  PSA_REQUIRE((int64_t)B * Hq <= 65535, PSA_ERR_UNSUPPORTED, "psa_estimate_xattn: B*Hq too large");
  PSA_REQUIRE(q.dtype == PSA_DTYPE_BF16 && k.dtype == PSA_DTYPE_BF16, PSA_ERR_UNSUPPORTED,
              "psa_estimate_xattn: bf16 tensors only (element type %d / %d)", q.dtype, k.dtype);
  const XGeom g = xgeom(Lq, Lk, block_size, stride, chunk_size);
  XParams p;
  p.q = (const bf16_t*)q.ptr; p.k = (const bf16_t*)k.ptr;
  p.q_sb = q.stride_b; p.q_sh = q.stride_h; p.q_sl = q.stride_l;
  p.k_sb = k.stride_b; p.k_sh = k.stride_h; p.k_sl = k.stride_l;
  if (Lq == 1) p.q_sl = D;  // (a single row's stride may be anything, and says where the padding begins)
  if (Lk == 1) p.k_sl = D;
  p.ws = (float*)workspace; p.est = est;
  p.Hq = Hq; p.Hkv = Hkv; p.Lq = Lq; p.Lk = Lk; p.D = D;
  p.S_log2 = psa_ilog2(stride); p.rb_log2 = psa_ilog2(rb);
  p.Mr = g.Mr; p.Nr = g.Nr; p.NB = g.NB;
  p.off = g.Nr - g.Mr;
  p.causal = causal ? 1 : 0;
  // the reference zeroes rows at or past (real key length)/stride in the key-aligned numbering
  p.real_rows = (Lk + stride - 1) / stride - p.off;
  p.out_rows = (Lq + block_size - 1) / block_size;
  p.out_cols = (Lk + block_size - 1) / block_size;
  p.scale2 = 1.4426950408889634f / sqrtf((float)D) / (float)stride;
  hipStream_t st = (hipStream_t)stream;
  const int64_t heads = (int64_t)B * Hq;
  // (every pair that the reduction reads is written: the tile rows end with the last q-block's, the rest is padding)
  const int rows_used = p.out_rows * rb < g.Mr ? p.out_rows * rb : g.Mr;
  const int64_t n_large = heads * active_tiles<XLarge>(p, rows_used), n_small = heads * active_tiles<XSmall>(p, rows_used);
  // rows that overlap (expanded tensors) take the kernel that checks every row, which has small tiles only
  const bool overlap = (Lq > 1 && q.stride_l < D) || (Lk > 1 && k.stride_l < D);
  const bool small = overlap || xattn_small(n_large, n_small);
  const int64_t n_active = small ? n_small : n_large;
  PSA_REQUIRE(n_active < (1ll << 28), PSA_ERR_UNSUPPORTED, "psa_estimate_xattn: too many output tiles");
  p.n_active = (int)n_active;
  p.per_xcd = (int)((n_active + 7) / 8);
  PoolPart pool = {};
  auto launch = [&](auto x) -> int {
    using X = decltype(x);
    constexpr bool SMALL = std::is_same_v<X, XSmall>;
    p.act_per_bh = active_tiles<X>(p, rows_used);
    const size_t shmem = X_BUFS * (size_t)X::STAGE;
    auto pick = [&](auto pool_c, auto rows_c) {
      constexpr bool P = decltype(pool_c)::value, R = decltype(rows_c)::value;
      return rb == 8 ? psa_xattn_gemm_kernel<3, X, P, R> : rb == 16 ? psa_xattn_gemm_kernel<4, X, P, R> : psa_xattn_gemm_kernel<5, X, P, R>;
    };
    auto kern = pick(std::false_type{}, std::false_type{});
    // large tiles: one workgroup per CU, which takes a tile after the other and copies ahead; small ones: one each
    p.slots = SMALL || p.per_xcd < X_CUS_PER_XCD ? p.per_xcd : X_CUS_PER_XCD;
    int64_t blocks = (int64_t)p.slots * 8;
    if constexpr (SMALL) {
      if (xm != nullptr && xm->pool != nullptr) {
        kern = overlap ? pick(std::true_type{}, std::true_type{}) : pick(std::true_type{}, std::false_type{});
        pool.p = *xm->pool;
        pool.first = (int)blocks;
        pool.nx = xm->pool_nx;
        pool.heads = xm->pool_heads;
        blocks += (int64_t)xm->pool_nx * xm->pool_heads * 2;
      } else if (overlap) {
        kern = pick(std::false_type{}, std::true_type{});
      }
    }
    if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem) != hipSuccess) return PSA_ERR_LAUNCH;
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(256), shmem, st, p, pool);
    return PSA_OK;
  };
  if (!small && xm != nullptr && xm->pool != nullptr) psa_pool_launch_cap(*xm->pool, xm->pool_nx, xm->pool_heads, st);
  int rc = small ? launch(XSmall{}) : launch(XLarge{});
  PSA_REQUIRE(rc == PSA_OK, rc, "psa_estimate_xattn: cannot reserve LDS");
  rc = psa_check_launch("psa_estimate_xattn (contraction)");
  if (rc != PSA_OK) return rc;
  // the pairs of one q-block: NB * rb * 8 bytes; cached in LDS when that leaves room for several workgroups per CU
  const size_t cache_bytes = (size_t)p.NB * ((size_t)1 << p.rb_log2) * 8;
  const int cached = cache_bytes <= 48 * 1024 ? 1 : 0;
  if (xm != nullptr) {
    const size_t map_bytes = qwen_row_lds_bytes(p.out_cols);  // (more than the 2 bytes per column of the lists' ids)
    size_t scratch = cached && cache_bytes > map_bytes ? cache_bytes : map_bytes;
    scratch = (scratch + 15) & ~(size_t)15;
    const size_t shmem = scratch + (size_t)p.out_cols * 5;
    if (shmem > 48 * 1024) {
      hipError_t e = hipFuncSetAttribute((const void*)psa_xattn_map_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);
      PSA_REQUIRE(e == hipSuccess, PSA_ERR_LAUNCH, "psa_level_map_qwen: cannot reserve %zu bytes of LDS", shmem);
    }
    hipLaunchKernelGGL(psa_xattn_map_kernel, dim3((unsigned)p.out_rows, (unsigned)(B * Hq)), dim3(256), shmem, st, p, cached, (int)scratch, xm->mp,
                       xm->end);
    return psa_check_launch("psa_estimate_xattn (reduction + level map)");
  }
  hipLaunchKernelGGL(psa_xattn_reduce_kernel, dim3((unsigned)p.out_rows, (unsigned)(B * Hq)), dim3(256), cached ? cache_bytes : 0, st, p, cached);
  return psa_check_launch("psa_estimate_xattn (reduction)");
}

extern "C" int psa_estimate_xattn(psa_tensor4 q, psa_tensor4 k, float* est, void* workspace, int B, int Hq, int Hkv, int Lq,
                                  int Lk, int D, int block_size, int stride, int chunk_size, int causal, psa_stream_t stream) {
  PSA_REQUIRE(est, PSA_ERR_ARG, "psa_estimate_xattn: null pointer");
  return xattn_run(q, k, est, workspace, B, Hq, Hkv, Lq, Lk, D, block_size, stride, chunk_size, causal, stream, nullptr);
}

// Pooling, similarity cap, estimate, level map, cap on the map and tile records (walk, null: none) of the causal layer (psa_layer.hip).
int psa_xattn_layer_map(psa_tensor4 q, psa_tensor4 k, psa_tensor4 v, void* workspace, void* k_pool, void* v_pool, int32_t* cap,
                        const float* thresholds, void* map, void* walk, int B, int Hq, int Hkv, int L, int D,
                        int block, int stride, int chunk, int mode, int n_items, const int32_t* item_level, const double* item_lo,
                        const double* item_hi, int special_blocks, int causal, psa_stream_t stream) {
  const int S = (L + block - 1) / block;
  XattnMap xm = {};
  int rc = qwen_map_fill_params(xm.mp, S, mode, n_items, item_level, item_lo, item_hi, special_blocks, causal);
  if (rc != PSA_OK) return rc;
  PoolParams pool;
  rc = psa_pool_params(pool, k, v, nullptr, nullptr, nullptr, k_pool, v_pool, B, Hkv, L, D, block, cap, thresholds);
  if (rc != PSA_OK) return rc;
  xm.end.map_out = map; xm.end.map_elem = 1;
  xm.end.cap = cap; xm.end.Hq = Hq; xm.end.n_rep = Hkv > 0 ? Hq / Hkv : 1;
  if (walk != nullptr) {
    psa_sched::Geometry g;
    PSA_REQUIRE(psa_schedule_geometry(B, Hq, Hkv, L, D, block, block, g), PSA_ERR_UNSUPPORTED, "psa_build_schedule: shape out of range");
    psa_walk_end(xm.end, walk, g, block, block, L, causal);
  }
  xm.pool = &pool;
  xm.pool_nx = (int)((pool.npad / 8 * (D / 8) + 255) / 256);
  xm.pool_heads = B * Hkv;
  return xattn_run(q, k, nullptr, workspace, B, Hq, Hkv, L, L, D, block, stride, chunk, causal, stream, &xm);
}
