// Builds the tile schedule of a level map (psa_schedule.h): one pass over the map, one wave per (batch, head,
// q-block) row, followed by the longest-first issue order of the rows (psa_order.h).  HBM-bound on the map
// (rows * Nk bytes in, about 16 bytes per retained tile out); latency-bound at the usual sizes.
#include "psa_common.h"
#include "psa_order.h"
#include "psa_schedule.h"

namespace {
using namespace psa_sched;
static_assert(COST_LIMIT == psa_order::COST_BINS - 1, "the last bin");

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
  const int jmax = live ? reached_blocks(Nk, I, bm, bn_log2, causal != 0) : 0;
  const int64_t mrow = (int64_t)row * Nk;
  RowLists rl;
#pragma unroll
  for (int lv = 0; lv < 4; ++lv) rl.cnt[lv] = 0;
  for (int j0 = 0; j0 < jmax; j0 += 64) {
    const int j = j0 + lane;
    const int lvl = j < jmax ? load_map(map, mrow + j, map_elem) : 0;
#pragma unroll
    for (int lv = 0; lv < 4; ++lv) rl.cnt[lv] += __popcll(__ballot(lvl == (1 << lv)));
  }
  row_offsets(rl, bn_log2);
  {
    int run[4] = {rl.io[0], rl.io[1], rl.io[2], rl.io[3]};
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
  const int T = rl.to[4];
  if (live && lane == 0) {
    tiles[row] = T;
    cost[row] = T < COST_LIMIT ? T : COST_LIMIT;
  }
  if (live)
    write_records(rl, ids, lane, 64, bn_log2, L, causal != 0, (int64_t)I * bm, recs + (int64_t)row * rec_stride,
                  fine + (int64_t)row * fine_stride * (FINE_RUNS * 2 / 16));
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

int psa_walk_order(void* walk, const psa_sched::Geometry& g, psa_stream_t stream) {
  char* base = (char*)walk;
  psa_order::sort_lists<1>({{{(const int32_t*)(base + g.lay.cost_off), (int32_t*)(base + g.lay.order_off), (int)g.rows, g.wg_chunk, g.wg_groups}}},
                           (hipStream_t)stream);
  return psa_check_launch("psa_build_schedule (order)");
}

void psa_walk_end(psa_sched::MapEnd& e, void* walk, const psa_sched::Geometry& g, int block_m, int block_n, int L, int causal) {
  char* base = (char*)walk;
  e.recs = (u32x4*)(base + g.lay.rec_off);
  e.fine = (u32x4*)(base + g.lay.fine_off);
  e.tiles = (int32_t*)(base + g.lay.tiles_off);
  e.cost = (int32_t*)(base + g.lay.cost_off);
  e.rec_stride = g.lay.rec_stride;
  e.fine_stride = g.lay.fine_stride;
  e.bn_log2 = psa_ilog2(block_n);
  e.bm = block_m;
  e.L = L;
  e.Mq = g.Mq;
  e.causal = causal ? 1 : 0;
}

static int build_schedule(const void* map, int map_elem_bytes, void* schedule, int B, int Hq, int Hkv, int L, int D, int block_m,
                          int block_n, int causal, psa_stream_t stream) {
  PSA_REQUIRE((uintptr_t)schedule % 16 == 0, PSA_ERR_ARG, "psa_build_schedule: schedule must be 16-byte aligned");
  psa_sched::Geometry g;
  PSA_REQUIRE(psa_schedule_geometry(B, Hq, Hkv, L, D, block_m, block_n, g), PSA_ERR_UNSUPPORTED, "psa_build_schedule: shape out of range");
  PSA_REQUIRE((size_t)ROWS_PER_WG * g.Nk * 2 <= 64 * 1024, PSA_ERR_UNSUPPORTED, "psa_build_schedule: more than 8192 kv-blocks");
  char* base = (char*)schedule;
  hipStream_t s = (hipStream_t)stream;
  int32_t* cost = (int32_t*)(base + g.lay.cost_off);
  int32_t* tiles = (int32_t*)(base + g.lay.tiles_off);
  u32x4* recs = (u32x4*)(base + g.lay.rec_off);
  hipLaunchKernelGGL(psa_sched_build_kernel, dim3((unsigned)((g.rows + ROWS_PER_WG - 1) / ROWS_PER_WG)), dim3(64 * ROWS_PER_WG),
                     (size_t)ROWS_PER_WG * g.Nk * 2, s, map, map_elem_bytes, (int)g.rows, g.Mq, g.Nk, psa_ilog2(block_n), block_m, L,
                     causal ? 1 : 0, cost, tiles, recs, g.lay.rec_stride, (u32x4*)(base + g.lay.fine_off), g.lay.fine_stride);
  if (int e = psa_check_launch("psa_build_schedule (tiles)")) return e;
  return psa_walk_order(schedule, g, stream);
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
