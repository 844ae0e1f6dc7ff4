// Builds the tile schedule of a level map (psa_schedule.h): one pass over the map, one wave per (batch, head,
// q-block) row, followed by the longest-first issue order of the rows (psa_order.h).  HBM-bound on the map
// (rows * Nk bytes in, about 16 bytes per retained tile out); latency-bound at the usual sizes.
#include "psa_common.h"
#include "psa_order.h"
#include "psa_schedule.h"

namespace {

constexpr int ROWS_PER_WG = 4;

__global__ __launch_bounds__(64 * ROWS_PER_WG) void psa_sched_build_kernel(const void* map, int map_elem, int rows, int Mq, int Nk,
                                                                          int bn_log2, int bm, int L, int causal, int32_t* cost,
                                                                          int32_t* tiles, u32x4* recs, int rec_stride, u32x4* fine,
                                                                          int fine_stride) {
  extern __shared__ uint16_t s_ids[];  // [ROWS_PER_WG][Nk]: kv-block ids of a row, grouped by level, ascending inside a level
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row = blockIdx.x * ROWS_PER_WG + wave;
  const bool live = row < rows;
  uint16_t* ids = s_ids + wave * Nk;
  const int I = live ? row % Mq : 0;
  int jmax = live ? Nk : 0;
  if (causal) {
    const int ce = (int)((((int64_t)(I + 1) * bm) + (1 << bn_log2) - 1) >> bn_log2);
    jmax = ce < jmax ? ce : jmax;
  }
  const int64_t mrow = (int64_t)row * Nk;
  int cnt[4] = {0, 0, 0, 0};
  for (int j0 = 0; j0 < jmax; j0 += 64) {
    const int j = j0 + lane;
    const int lvl = j < jmax ? load_map(map, mrow + j, map_elem) : 0;
#pragma unroll
    for (int lv = 0; lv < 4; ++lv) cnt[lv] += __popcll(__ballot(lvl == (1 << lv)));
  }
  int io[4], to[5];
  {
    int i = 0, t = 0;
#pragma unroll
    for (int lv = 0; lv < 4; ++lv) {
      io[lv] = i;
      to[lv] = t;
      i += cnt[lv];
      t += ((cnt[lv] << (bn_log2 - lv)) + 63) >> 6;
    }
    to[4] = t;
  }
  {
    int run[4] = {io[0], io[1], io[2], io[3]};
    const uint64_t lt_mask = (1ull << lane) - 1ull;
    for (int j0 = 0; j0 < jmax; j0 += 64) {
      const int j = j0 + lane;
      const int lvl = j < jmax ? load_map(map, mrow + j, map_elem) : 0;
#pragma unroll
      for (int lv = 0; lv < 4; ++lv) {
        const uint64_t bal = __ballot(lvl == (1 << lv));
        if (lvl == (1 << lv)) ids[run[lv] + __popcll(bal & lt_mask)] = (uint16_t)j;
        run[lv] += __popcll(bal);
      }
    }
  }
  __syncthreads();  // (a wave only reads its own ids; the barrier orders the writes before the reads)
  const int T = to[4];
  u32x4* out = recs + (int64_t)row * rec_stride;
  if (live && lane == 0) {
    tiles[row] = T;
    cost[row] = T < psa_order::COST_BINS - 1 ? T : psa_order::COST_BINS - 1;
  }
  const int64_t q_first_row = (int64_t)I * bm;
  for (int t = lane; t < T; t += 64) {
    const int lv = (t >= to[1]) + (t >= to[2]) + (t >= to[3]);
    int lt = t, c_lv = cnt[0], io_lv = io[0];
#pragma unroll
    for (int l = 1; l < 4; ++l)
      if (lv == l) {
        lt = t - to[l];
        c_lv = cnt[l];
        io_lv = io[l];
      }
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
    const int fine_at = t - (bn_log2 - 2 < 4 ? to[2] : to[3]);
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
      u32x4* f = fine + ((int64_t)row * fine_stride + fine_at) * (psa_sched::FINE_RUNS * 2 / 16);
#pragma unroll
      for (int h8 = 0; h8 < psa_sched::FINE_RUNS / 8; ++h8) {
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
    const uint32_t code = ragged ? psa_sched::REC_CODE_RAGGED : is_fine ? 4u + (uint32_t)lv : (uint32_t)lv;
    const uint32_t hi = (code << psa_sched::REC_CODE_SHIFT) |
                        ((uint32_t)(diag || nvalid < 64) << psa_sched::REC_MASKED_BIT) | ((uint32_t)nvalid << psa_sched::REC_NVALID_SHIFT);
#pragma unroll
    for (int g = 0; g < 4; ++g) r[g] |= hi;
    out[t] = r;
    if (t == T - 1) {
#pragma unroll
      for (int e = 1; e <= psa_sched::REC_PAD; ++e) out[t + e] = r;
    }
  }
}

}  // namespace

// schedules of the public psa_schedule_* entry points
bool psa_schedule_shape_ok(int D, int block_m, int block_n, int L) {
  return (D == 128 || D == 64) && block_m == 128 && block_n == 128 && (int64_t)((L + 127) / 128) * 128 <= (1 << psa_sched::REC_SRC_BITS);
}
// schedules that the forward builds for itself (psa_walk_*); 8192 kv-blocks: the builder's LDS
bool psa_walk_shape_ok(int D, int block_m, int block_n, int L) {
  return (D == 128 || D == 64) && block_m == 128 && (block_n == 128 || block_n == 64 || block_n == 32) &&
         (int64_t)((L + 127) / 128) * 128 <= (1 << psa_sched::REC_SRC_BITS) && (L + block_n - 1) / block_n <= 8192;
}

bool psa_schedule_geometry(int B, int Hq, int Hkv, int L, int D, int block_m, int block_n, psa_sched::Geometry& g) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || L <= 0 || Hq % Hkv != 0 || !psa_walk_shape_ok(D, block_m, block_n, L)) return false;
  if (B >= 65536 || Hq >= 65536) return false;
  g.Mq = (L + block_m - 1) / block_m;
  g.Nk = (L + block_n - 1) / block_n;
  g.rows = (int64_t)B * Hq * g.Mq;
  if (g.rows >= (1ll << 28)) return false;
  // dealing of the rows to the XCDs, by the bytes of K, V and their pooled levels
  const double kv_bytes = 2.0 * B * Hkv * ((double)g.Nk * block_n) * D * 2.0 * 1.875;
  psa_order::deal(g.rows, kv_bytes, B * Hkv, g.wg_chunk, g.wg_groups);
  // Shares of even length: no walk needs them, but a caller may keep a schedule, and its layout follows from the share size.
  g.wg_chunk = (g.wg_chunk + 1) & ~1;
  g.lay = psa_sched::layout(g.rows, g.Nk, block_n, (int64_t)g.wg_chunk * g.wg_groups);
  return true;
}

static int build_schedule(const void* map, int map_elem_bytes, void* schedule, int B, int Hq, int Hkv, int L, int D, int block_m,
                          int block_n, int causal, psa_stream_t stream) {
  PSA_REQUIRE((uintptr_t)schedule % 16 == 0, PSA_ERR_ARG, "psa_build_schedule: schedule must be 16-byte aligned");
  psa_sched::Geometry g;
  PSA_REQUIRE(psa_schedule_geometry(B, Hq, Hkv, L, D, block_m, block_n, g), PSA_ERR_UNSUPPORTED, "psa_build_schedule: shape out of range");
  PSA_REQUIRE((size_t)ROWS_PER_WG * g.Nk * 2 <= 64 * 1024, PSA_ERR_UNSUPPORTED, "psa_build_schedule: more than 8192 kv-blocks");
  char* base = (char*)schedule;
  hipStream_t s = (hipStream_t)stream;
  int32_t* order = (int32_t*)(base + g.lay.order_off);
  int32_t* cost = (int32_t*)(base + g.lay.cost_off);
  int32_t* tiles = (int32_t*)(base + g.lay.tiles_off);
  u32x4* recs = (u32x4*)(base + g.lay.rec_off);
  hipLaunchKernelGGL(psa_sched_build_kernel, dim3((unsigned)((g.rows + ROWS_PER_WG - 1) / ROWS_PER_WG)), dim3(64 * ROWS_PER_WG),
                     (size_t)ROWS_PER_WG * g.Nk * 2, s, map, map_elem_bytes, (int)g.rows, g.Mq, g.Nk, psa_ilog2(block_n), block_m, L,
                     causal ? 1 : 0, cost, tiles, recs, g.lay.rec_stride, (u32x4*)(base + g.lay.fine_off), g.lay.fine_stride);
  if (int e = psa_check_launch("psa_build_schedule (tiles)")) return e;
  psa_order::sort_lists<1>({{{cost, order, (int)g.rows, g.wg_chunk, g.wg_groups}}}, s);
  return psa_check_launch("psa_build_schedule (order)");
}

extern "C" int64_t psa_schedule_bytes(int B, int Hq, int Hkv, int L, int D, int block_m, int block_n) {
  psa_sched::Geometry g;
  return psa_schedule_shape_ok(D, block_m, block_n, L) && psa_schedule_geometry(B, Hq, Hkv, L, D, block_m, block_n, g) ? g.lay.bytes : 0;
}

extern "C" int psa_build_schedule(const void* map, int map_elem_bytes, void* schedule, int B, int Hq, int Hkv, int L, int D,
                                  int block_m, int block_n, int causal, psa_stream_t stream) {
  PSA_REQUIRE(map != nullptr && schedule != nullptr, PSA_ERR_ARG, "psa_build_schedule: null pointer");
  PSA_REQUIRE(map_elem_bytes == 1 || map_elem_bytes == 4, PSA_ERR_ARG, "psa_build_schedule: map_elem_bytes must be 1 or 4");
  PSA_REQUIRE(B > 0 && Hq > 0 && Hkv > 0 && L > 0 && Hq % Hkv == 0, PSA_ERR_ARG, "psa_build_schedule: bad B / H / L");
  PSA_REQUIRE(psa_schedule_shape_ok(D, block_m, block_n, L), PSA_ERR_UNSUPPORTED,
              "psa_build_schedule: schedules exist for D = 64 or 128, block_m = block_n = 128 (got D=%d, block_m=%d, block_n=%d)", D, block_m, block_n);
  return build_schedule(map, map_elem_bytes, schedule, B, Hq, Hkv, L, D, block_m, block_n, causal, stream);
}

extern "C" int64_t psa_walk_bytes(int B, int Hq, int Hkv, int L, int D, int block_m, int block_n) {
  psa_sched::Geometry g;
  return psa_schedule_geometry(B, Hq, Hkv, L, D, block_m, block_n, g) ? g.lay.bytes : 0;
}

extern "C" int psa_build_walk(const void* map, int map_elem_bytes, void* walk, int B, int Hq, int Hkv, int L, int D, int block_m,
                              int block_n, int causal, psa_stream_t stream) {
  PSA_REQUIRE(map != nullptr && walk != nullptr, PSA_ERR_ARG, "psa_build_walk: null pointer");
  PSA_REQUIRE(map_elem_bytes == 1 || map_elem_bytes == 4, PSA_ERR_ARG, "psa_build_walk: map_elem_bytes must be 1 or 4");
  PSA_REQUIRE(B > 0 && Hq > 0 && Hkv > 0 && L > 0 && Hq % Hkv == 0, PSA_ERR_ARG, "psa_build_walk: bad B / H / L");
  return build_schedule(map, map_elem_bytes, walk, B, Hq, Hkv, L, D, block_m, block_n, causal, stream);
}
