// Tile schedule of the row-walking attention kernels, built once per level map and kept in device memory.
//
// A (batch, head, q-block) row of the level map is walked as a sequence of TILES of 64 pooled keys of one level
// (psa_tiles.h).  The schedule stores that sequence per row so that the attention kernels neither compact the map
// row nor look block ids up per lane: with 128-key blocks every 16-key quarter of a tile lies inside ONE kv-block
// (the smallest pooled block holds 16 keys), so a tile is fully described by the source row of each quarter.
// With 64- and 32-key blocks the same holds for the pooled blocks of at least 16 keys; the tiles of smaller ones
// (FINE tiles: 8 or 4 keys per block) also have a list of block ids, one per 4 tile rows.
//
// Layout of the schedule buffer (all offsets from its start, `rows` = B * Hq * Mq):
//   reserved                                           64 bytes
//   order   int32 [order_entries]                      issue order of the rows (dealt to the XCDs, longest first), -1 = none
//   cost    int32 [rows]                               tiles per row, clamped to the sorter's range
//   tiles   int32 [rows]                               T: number of tiles of the row
//   records u32x4 [rows][rec_stride]                   one record per tile (+ 3), rec_stride = 2 * Nk + 4 for 128-key blocks
//   fine    uint16 [rows][fine_stride][16]             kv-block id of every 4-row run of a fine tile (64- / 32-key blocks)
//
// Record of a tile: four words, word g for the wave that copies tile rows 16g .. 16g+15 - each word is complete in
// itself, so a wave fetches one word per tile:
//   bits  0..19  first source row of that quarter, in the row numbering of the tile's level
//                (level 0: token index; level l: pooled row index of the level's [Npad >> l] rows)
//   bits 20..22  level code: 0..3 = pooling by 1, 2, 4, 8; 4 = a level-0 tile whose source rows run past the last
//                token (ragged: lanes clamp their rows to L - 1); 4 + level (6, 7) = a fine tile: bits 0..19 hold its
//                index in the row's part of `fine`
//   bit  23      masked: some slots are empty and / or the tile touches the causal diagonal
//   bits 24..30  nvalid: the first nvalid slots of the tile hold keys (0..64)
// Quarters past the end of a level's list point at the level's last retained block (any readable rows: masked).
// The last record of a row is repeated three times behind it (the kernels fetch records up to three tiles ahead).
#pragma once

#include "psa_common.h"

namespace psa_sched {

constexpr int REC_SRC_BITS = 20, REC_CODE_SHIFT = 20, REC_MASKED_BIT = 23, REC_NVALID_SHIFT = 24, REC_PAD = 3;
constexpr uint32_t REC_SRC_MASK = (1u << REC_SRC_BITS) - 1u;
constexpr uint32_t REC_CODE_RAGGED = 4, REC_CODE_FINE = 5;  // (codes from REC_CODE_FINE on are fine tiles)
constexpr int FINE_RUNS = 16;                                // 4-row runs per tile
constexpr int COST_LIMIT = 2047;                             // costs are clamped to the sorter's range (psa_order.h)

struct Layout {
  int64_t order_off, cost_off, tiles_off, rec_off, fine_off, bytes;
  int64_t order_entries;
  int rec_stride, fine_stride;
};

// Most records / fine tiles of a row.  A row of 128- or 64-key blocks has at most 2 * Nk / Nk tiles (every block at level
// 0: a partly filled tile of another level stands for at least one block), a row of 32-key blocks Nk / 2 and one partly
// filled tile per level.
static inline int rec_stride_of(int Nk, int block_n) { return block_n == 128 ? 2 * Nk + 4 : block_n == 64 ? Nk + 4 : (Nk + 1) / 2 + 8; }
static inline int fine_stride_of(int Nk, int block_n) { return block_n == 128 ? 0 : Nk / 8 + 2; }

// byte offsets of the parts for `rows` rows; order_entries bounds any dealing of the rows (psa_order::deal)
static inline Layout layout(int64_t rows, int Nk, int block_n, int64_t order_entries) {
  Layout l;
  l.rec_stride = rec_stride_of(Nk, block_n);
  l.fine_stride = fine_stride_of(Nk, block_n);
  l.order_entries = order_entries;
  l.order_off = 64;
  l.cost_off = l.order_off + ((order_entries * 4 + 63) & ~(int64_t)63);
  l.tiles_off = l.cost_off + ((rows * 4 + 63) & ~(int64_t)63);
  l.rec_off = l.tiles_off + ((rows * 4 + 63) & ~(int64_t)63);
  l.fine_off = l.rec_off + rows * (int64_t)l.rec_stride * 16;
  l.bytes = l.fine_off + rows * (int64_t)l.fine_stride * (FINE_RUNS * 2);
  return l;
}

// everything the host derives from a call's shape arguments (the buffer carries no header: nothing is read back)
struct Geometry {
  int64_t rows;
  int Mq, Nk;
  int wg_chunk, wg_groups;  // dealing of the rows: wg_groups shares of wg_chunk entries of order[]
  Layout lay;
};

__device__ __forceinline__ uint32_t rec_code(uint32_t w) { return (w >> REC_CODE_SHIFT) & 7u; }
__device__ __forceinline__ int rec_level(uint32_t w) { return (int)((w >> REC_CODE_SHIFT) & 3u); }
__device__ __forceinline__ bool rec_masked(uint32_t w) { return ((w >> REC_MASKED_BIT) & 1u) != 0; }
__device__ __forceinline__ int rec_nvalid(uint32_t w) { return (int)((w >> REC_NVALID_SHIFT) & 127u); }
__device__ __forceinline__ int rec_src(uint32_t w) { return (int)(w & REC_SRC_MASK); }

// The tiles of a row from its kv-blocks grouped by level: cnt[l] blocks of level l, ids[io[l] ..) ascending.
struct RowLists {
  int cnt[4], io[4], to[5];  // to[l]: first tile of level l
};
__device__ __forceinline__ void row_offsets(RowLists& r, int bn_log2) {
  int i = 0, t = 0;
#pragma unroll
  for (int lv = 0; lv < 4; ++lv) {
    r.io[lv] = i;
    r.to[lv] = t;
    i += r.cnt[lv];
    t += ((r.cnt[lv] << (bn_log2 - lv)) + 63) >> 6;
  }
  r.to[4] = t;
}
// Writes the records of tiles first, first + step, ..
__device__ __forceinline__ void write_records(const RowLists& rl, const uint16_t* ids, int first, int step, int bn_log2, int L, bool causal,
                                              int64_t q_first_row, u32x4* out, u32x4* fine) {
  const int T = rl.to[4], to1 = rl.to[1], to2 = rl.to[2], to3 = rl.to[3];
  const int c0 = rl.cnt[0], c1 = rl.cnt[1], c2 = rl.cnt[2], c3 = rl.cnt[3], i0 = rl.io[0], i1 = rl.io[1], i2 = rl.io[2], i3 = rl.io[3];
  for (int t = first; t < T; t += step) {
    const int lv = (t >= to1) + (t >= to2) + (t >= to3);
    const int lt = t - (lv == 0 ? 0 : lv == 1 ? to1 : lv == 2 ? to2 : to3);
    const int c_lv = lv == 0 ? c0 : lv == 1 ? c1 : lv == 2 ? c2 : c3, io_lv = lv == 0 ? i0 : lv == 1 ? i1 : lv == 2 ? i2 : i3;
    const int sbs_log2 = bn_log2 - lv;
    int nvalid = (c_lv << sbs_log2) - (lt << 6);
    nvalid = nvalid < 64 ? nvalid : 64;
    const int last_blk = ids[io_lv + (((lt << 6) + nvalid - 1) >> sbs_log2)];
    if (lv == 0) {
      const int over = (((lt << 6) + nvalid - 1) & ((1 << sbs_log2) - 1)) + 1 - (L - (last_blk << sbs_log2));
      if (over > 0) nvalid = nvalid - over > 0 ? nvalid - over : 0;
    }
    const bool diag = causal && ((((int64_t)last_blk + 1) << bn_log2) - 1 > q_first_row);
    u32x4 r;
    bool ragged = false;
    const bool is_fine = sbs_log2 < 4;
    // fine tiles are the last ones of a row (the levels come in ascending order): their index counts from the first
    const int fine_at = t - (bn_log2 - 2 < 4 ? to2 : to3);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      if (is_fine) {
        r[g] = (uint32_t)fine_at;
        continue;
      }
      const int gpos = (lt << 6) + 16 * g;
      int bi = gpos >> sbs_log2;
      bi = bi < c_lv - 1 ? bi : c_lv - 1;
      const int src = ((int)ids[io_lv + bi] << sbs_log2) + (gpos & ((1 << sbs_log2) - 1));
      ragged |= lv == 0 && src + 15 >= L;
      r[g] = (uint32_t)src;
    }
    if (is_fine) {
      u32x4* f = fine + (int64_t)fine_at * (FINE_RUNS * 2 / 16);
#pragma unroll
      for (int h8 = 0; h8 < FINE_RUNS / 8; ++h8) {
        u32x4 w;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          int bi = ((lt << 6) + 4 * (8 * h8 + e)) >> sbs_log2;
          bi = bi < c_lv - 1 ? bi : c_lv - 1;
          const uint32_t id = ids[io_lv + bi];
          w[e >> 1] = (e & 1) ? w[e >> 1] | (id << 16) : id;
        }
        f[h8] = w;
      }
    }
    const uint32_t code = ragged ? REC_CODE_RAGGED : is_fine ? 4u + (uint32_t)lv : (uint32_t)lv;
    const uint32_t hi = (code << REC_CODE_SHIFT) | ((uint32_t)(diag || nvalid < 64) << REC_MASKED_BIT) | ((uint32_t)nvalid << REC_NVALID_SHIFT);
#pragma unroll
    for (int g = 0; g < 4; ++g) r[g] |= hi;
    out[t] = r;
    if (t == T - 1) {
#pragma unroll
      for (int e = 1; e <= REC_PAD; ++e) out[t + e] = r;
    }
  }
}
// kv-blocks of a row (or of a row's columns j >= jmax: none) that a causal q-block I of bm rows reaches
__device__ __forceinline__ int reached_blocks(int Nk, int I, int bm, int bn_log2, bool causal) {
  if (!causal) return Nk;
  const int ce = (int)((((int64_t)(I + 1) * bm) + (1 << bn_log2) - 1) >> bn_log2);
  return ce < Nk ? ce : Nk;
}

// What is left to do for a row of the map once its levels are known.  The kernels that form maps keep the levels of a row in LDS, end
// them here - similarity cap, the map itself, tile records - and so spare a launch and a pass over the map each for the cap and for
// the list (psa_sched_build_kernel).  Reduction + map with and without, and what goes, us: 12 heads x 32760 tokens 60 for 52 + 9 + 5 (cap), with
// 32-key blocks 114 for 105 + 18, 48 heads x 45106 tokens of 32-key blocks 661 for 606 + 72.
struct MapEnd {
  void* map_out;
  int map_elem;
  const int32_t* cap;  // optional: [kv head][Nk]
  int Hq, n_rep;       // query heads per batch, per kv head
  // tile records (psa_schedule.h), null recs: none
  u32x4* recs;
  u32x4* fine;
  int32_t *tiles, *cost;
  int rec_stride, fine_stride;
  int bn_log2, bm, L, Mq, causal;
};

// Ends row `row` = bh * Mq + I (256 threads; a barrier comes first).  lv: its Nk levels in LDS; ids: 2 * Nk bytes of LDS; s_cnt: 16 ints.
__device__ __forceinline__ void end_map_row(const MapEnd& f, uint8_t* lv, int Nk, int64_t row, int bh, int I, uint16_t* ids, int* s_cnt, int tid) {
  constexpr int NT = 256, NW = NT / 64;
  const int lane = tid & 63, wave = tid >> 6;
  __syncthreads();
  const int32_t* cap = f.cap != nullptr ? f.cap + (int64_t)((bh / f.Hq) * (f.Hq / f.n_rep) + (bh % f.Hq) / f.n_rep) * Nk : nullptr;
  for (int j = tid; j < Nk; j += NT) {
    int l = lv[j];
    if (cap != nullptr) {
      const int c = cap[j];
      if (c < l) lv[j] = (uint8_t)(l = c);
    }
    store_map(f.map_out, row * Nk + j, f.map_elem, l);
  }
  if (f.recs == nullptr) return;
  __syncthreads();
  // wave w lists columns [w * share, (w + 1) * share): counts first, then, with those of the waves before it, the ids
  const int jmax = reached_blocks(Nk, I, f.bm, f.bn_log2, f.causal != 0);
  const int share = ((jmax + 64 * NW - 1) / (64 * NW)) * 64;
  const int j_lo = wave * share, j_hi = (wave + 1) * share < jmax ? (wave + 1) * share : jmax;
  RowLists rl;
#pragma unroll
  for (int l = 0; l < 4; ++l) rl.cnt[l] = 0;
  for (int j0 = j_lo; j0 < j_hi; j0 += 64) {
    const int lvl = j0 + lane < j_hi ? lv[j0 + lane] : 0;
#pragma unroll
    for (int l = 0; l < 4; ++l) rl.cnt[l] += __popcll(__ballot(lvl == (1 << l)));
  }
  if (lane == 0) {
#pragma unroll
    for (int l = 0; l < 4; ++l) s_cnt[wave * 4 + l] = rl.cnt[l];
  }
  __syncthreads();
  int run[4];
#pragma unroll
  for (int l = 0; l < 4; ++l) {
    run[l] = 0;
    rl.cnt[l] = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const int c = s_cnt[w * 4 + l];
      run[l] += w < wave ? c : 0;
      rl.cnt[l] += c;
    }
  }
  row_offsets(rl, f.bn_log2);
#pragma unroll
  for (int l = 0; l < 4; ++l) run[l] += rl.io[l];
  for (int j0 = j_lo; j0 < j_hi; j0 += 64) {
    const int lvl = j0 + lane < j_hi ? lv[j0 + lane] : 0;
#pragma unroll
    for (int l = 0; l < 4; ++l) {
      const uint64_t bal = __ballot(lvl == (1 << l));
      if (lvl == (1 << l)) ids[run[l] + __popcll(bal & ((1ull << lane) - 1ull))] = (uint16_t)(j0 + lane);
      run[l] += __popcll(bal);
    }
  }
  __syncthreads();
  const int T = rl.to[4];
  if (tid == 0) {
    f.tiles[row] = T;
    f.cost[row] = T < COST_LIMIT ? T : COST_LIMIT;
  }
  write_records(rl, ids, tid, NT, f.bn_log2, f.L, f.causal != 0, (int64_t)I * f.bm, f.recs + row * f.rec_stride,
                f.fine + row * f.fine_stride * (FINE_RUNS * 2 / 16));
}

}  // namespace psa_sched

// host side (psa_schedule.hip)
// Issue order of a walk whose records and costs are there already (psa_sched::MapEnd).
int psa_walk_order(void* walk, const psa_sched::Geometry& g, psa_stream_t stream);
// The parts of a walk buffer as the end of a map row writes them.
void psa_walk_end(psa_sched::MapEnd& e, void* walk, const psa_sched::Geometry& g, int block_m, int block_n, int L, int causal);

// shapes for which schedules exist (psa_schedule_*: 128-key blocks; psa_walk_*: every block_n)
bool psa_schedule_shape_ok(int D, int block_m, int block_n, int L);
bool psa_walk_shape_ok(int D, int block_m, int block_n, int L);
// geometry of the schedule of a shape (any block_n); false when the shape has none
bool psa_schedule_geometry(int B, int Hq, int Hkv, int L, int D, int block_m, int block_n, psa_sched::Geometry& g);
