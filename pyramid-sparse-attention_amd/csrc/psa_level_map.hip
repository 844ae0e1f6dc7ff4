// Scores -> pyramid level map (and the index-list format), plus small map utilities.
//
// One workgroup per (b, h, q-block) row.  The row (<= a few thousand fp32 scores) lives in LDS:
//   1. stable descending order on a 64-bit key (inverted order-preserving score bits, then column
//      index) - keys are unique so ties resolve to the lower column (sort_row_desc);
//   2. thresholdbound only: sequential fp64 prefix sums rounded to fp32 (one lane walks the row,
//      which keeps the additions in exactly the order a serial CPU scan uses), r = c / c[last] with
//      an IEEE fp32 division, per-threshold counts of r <= thr;
//   3. integer interval logic per item (alignment of each level's count to ceil(level/align_div));
//   4. scatter of levels to their columns.
// Latency-bound: about 1 KB read and 0.25-1 KB written per row.
#include "psa_level_map_row.h"

__global__ __launch_bounds__(256) void psa_level_map_kernel(LevelMapParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ int s_cnt[PSA_MAX_LEVEL_ITEMS];
  __shared__ int s_iv[PSA_MAX_LEVEL_ITEMS][2];
  const int64_t row = blockIdx.x;
  level_map_row(p, p.scores + row * p.Nk, row, smem, s_cnt, s_iv, (int)threadIdx.x, (int)blockDim.x);
}

extern "C" int psa_level_map(const float* scores, void* map_out, int map_elem_bytes, int32_t* list_out, int64_t rows,
                             int Nk, int mode, int n_items, const int32_t* item_level, const double* item_hi,
                             int align_div, int text_blocks, double min_full_attn_ratio, psa_stream_t stream) {
  PSA_REQUIRE(scores && (map_out || list_out), PSA_ERR_ARG, "psa_level_map: null pointer");
  PSA_REQUIRE(map_elem_bytes == 1 || map_elem_bytes == 4, PSA_ERR_ARG, "psa_level_map: map_elem_bytes must be 1 or 4");
  PSA_REQUIRE(rows > 0 && rows < (1ll << 31), PSA_ERR_UNSUPPORTED, "psa_level_map: rows=%lld out of range", (long long)rows);
  LevelMapParams p;
  const int rc = level_map_fill_params(p, Nk, mode, n_items, item_level, item_hi, align_div, text_blocks, min_full_attn_ratio);
  if (rc != PSA_OK) return rc;
  p.scores = scores; p.map_out = map_out; p.list_out = list_out; p.map_elem = map_elem_bytes;
  size_t shmem = level_map_lds_bytes(p);
  if (shmem > 48 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void*)psa_level_map_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);
    PSA_REQUIRE(e == hipSuccess, PSA_ERR_LAUNCH, "psa_level_map: cannot reserve %zu bytes of LDS", shmem);
  }
  const int nt = Nk > RANK_SORT_MAX ? 256 : ((Nk + 63) / 64) * 64;  // one thread per score of a short row: idle waves only take up slots
  hipLaunchKernelGGL(psa_level_map_kernel, dim3((unsigned)rows), dim3(nt), shmem, (hipStream_t)stream, p);
  return psa_check_launch("psa_level_map");
}

// ---------------------------------------------------------------------------------------
// level map of the causal Qwen2.5-VL example: square map, per-row ratio windows, fix-ups
// ---------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void psa_level_map_qwen_kernel(QwenMapParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int64_t row = blockIdx.x;
  qwen_map_row(p, p.scores + row * p.S, (int)(row % p.S), p.S, smem, (int)threadIdx.x, (int)blockDim.x,
               [&](int col, int lv) __attribute__((always_inline)) { store_map(p.map_out, row * p.S + col, p.map_elem, lv); });
}

extern "C" int psa_level_map_qwen(const float* scores, void* map_out, int map_elem_bytes, int64_t bh, int S, int mode,
                                  int n_items, const int32_t* item_level, const double* item_lo, const double* item_hi,
                                  int special_blocks, int causal, psa_stream_t stream) {
  PSA_REQUIRE(scores && map_out && item_level && item_lo && item_hi, PSA_ERR_ARG, "psa_level_map_qwen: null pointer");
  PSA_REQUIRE(map_elem_bytes == 1 || map_elem_bytes == 4, PSA_ERR_ARG, "psa_level_map_qwen: map_elem_bytes must be 1 or 4");
  PSA_REQUIRE(bh > 0 && S > 0 && S <= 6144 && bh * S < (1ll << 31), PSA_ERR_UNSUPPORTED, "psa_level_map_qwen: sizes out of range");
  QwenMapParams p;
  const int rc = qwen_map_fill_params(p, S, mode, n_items, item_level, item_lo, item_hi, special_blocks, causal);
  if (rc != PSA_OK) return rc;
  p.scores = scores; p.map_out = map_out; p.map_elem = map_elem_bytes;
  const size_t shmem = qwen_row_lds_bytes(S);
  if (shmem > 48 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void*)psa_level_map_qwen_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);
    PSA_REQUIRE(e == hipSuccess, PSA_ERR_LAUNCH, "psa_level_map_qwen: cannot reserve %zu bytes of LDS", shmem);
  }
  const int nt = S > RANK_SORT_MAX ? 256 : ((S + 63) / 64) * 64;
  hipLaunchKernelGGL(psa_level_map_qwen_kernel, dim3((unsigned)(bh * S)), dim3(nt), shmem, (hipStream_t)stream, p);
  return psa_check_launch("psa_level_map_qwen");
}

// ---------------------------------------------------------------------------------------
// index list -> dense map
// ---------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void psa_map_from_list_kernel(const int32_t* list, void* map, int map_elem, int width, int Nk) {
  __shared__ int s_wave_sep[4];
  const int64_t row = blockIdx.x;
  const int32_t* src = list + row * width;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int j = tid; j < Nk; j += 256) store_map(map, row * Nk + j, map_elem, 0);
  __syncthreads();
  int seps_before = 0;  // separators in columns before the current chunk
  for (int c0 = 0; c0 < width; c0 += 256) {
    const int c = c0 + tid;
    const int v = c < width ? src[c] : 0;
    const bool is_sep = c < width && v == -1;
    const uint64_t bal = __ballot(is_sep);
    if (lane == 0) s_wave_sep[wave] = __popcll(bal);
    __syncthreads();
    int before = seps_before;
    for (int w = 0; w < wave; ++w) before += s_wave_sep[w];
    before += __popcll(bal & ((1ull << lane) - 1ull));
    if (c < width && !is_sep && before <= 3 && v >= 0 && v < Nk) store_map(map, row * Nk + v, map_elem, 1 << before);
    seps_before += s_wave_sep[0] + s_wave_sep[1] + s_wave_sep[2] + s_wave_sep[3];
    __syncthreads();
  }
}

extern "C" int psa_map_from_list(const int32_t* list, void* map_out, int map_elem_bytes, int64_t rows, int width, int Nk,
                                 psa_stream_t stream) {
  PSA_REQUIRE(list && map_out, PSA_ERR_ARG, "psa_map_from_list: null pointer");
  PSA_REQUIRE(map_elem_bytes == 1 || map_elem_bytes == 4, PSA_ERR_ARG, "psa_map_from_list: map_elem_bytes must be 1 or 4");
  PSA_REQUIRE(rows > 0 && rows < (1ll << 31) && Nk > 0 && width >= Nk, PSA_ERR_ARG, "psa_map_from_list: bad sizes");
  hipLaunchKernelGGL(psa_map_from_list_kernel, dim3((unsigned)rows), dim3(256), 0, (hipStream_t)stream, list, map_out,
                     map_elem_bytes, width, Nk);
  return psa_check_launch("psa_map_from_list");
}

// ---------------------------------------------------------------------------------------
// dense map -> index list (five segments: levels 1, 2, 4, 8, then the skipped blocks; -1 after each)
// ---------------------------------------------------------------------------------------
// One wave per row.  Blocks are listed by level, ascending inside a level; a segment's length is rounded down to a
// multiple of ceil(level / align_div) and the blocks that do not fit lead the next segment.
__global__ __launch_bounds__(256) void psa_list_from_map_kernel(const void* map, int map_elem, int32_t* list, int64_t rows, int Nk,
                                                              int align_div) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int64_t mrow = row * Nk;
  int32_t* out = list + row * (Nk + 5);
  // segment of a level value: 1, 2, 4, 8 -> 0..3, anything else (0 = skipped) -> 4
  auto seg_of = [](int lvl) { return lvl == 1 ? 0 : lvl == 2 ? 1 : lvl == 4 ? 2 : lvl == 8 ? 3 : 4; };
  int cnt[5] = {0, 0, 0, 0, 0};
  for (int j0 = 0; j0 < Nk; j0 += 64) {
    const int j = j0 + lane;
    const int sg = j < Nk ? seg_of(load_map(map, mrow + j, map_elem)) : -1;
#pragma unroll
    for (int t = 0; t < 5; ++t) cnt[t] += __popcll(__ballot(sg == t));
  }
  int start[5], bound[5];  // first sorted position of a level; end of a segment after the rounding
  {
    int a = 0;
#pragma unroll
    for (int t = 0; t < 5; ++t) {
      start[t] = a;
      a += cnt[t];
    }
    int carry = 0, b = 0;
#pragma unroll
    for (int t = 0; t < 5; ++t) {
      int len = cnt[t] + carry;
      carry = 0;
      if (t < 4) {
        const int mult = ((1 << t) + align_div - 1) / align_div;
        carry = mult > 1 ? len % mult : 0;
        len -= carry;
      }
      b += len;
      bound[t] = b;
    }
  }
  if (lane < 5) out[bound[lane] + lane] = -1;  // the separator behind segment `lane`
  int run[5] = {start[0], start[1], start[2], start[3], start[4]};
  const uint64_t lt_mask = (1ull << lane) - 1ull;
  for (int j0 = 0; j0 < Nk; j0 += 64) {
    const int j = j0 + lane;
    const int sg = j < Nk ? seg_of(load_map(map, mrow + j, map_elem)) : -1;
#pragma unroll
    for (int t = 0; t < 5; ++t) {
      const uint64_t bal = __ballot(sg == t);
      if (sg == t) {
        const int pos = run[t] + __popcll(bal & lt_mask);  // position in the list sorted by level
        const int seps = (pos >= bound[0]) + (pos >= bound[1]) + (pos >= bound[2]) + (pos >= bound[3]) + (pos >= bound[4]);
        out[pos + seps] = j;
      }
      run[t] += __popcll(bal);
    }
  }
}

extern "C" int psa_list_from_map(const void* map, int map_elem_bytes, int32_t* list_out, int64_t rows, int Nk, int align_div,
                                 psa_stream_t stream) {
  PSA_REQUIRE(map && list_out, PSA_ERR_ARG, "psa_list_from_map: null pointer");
  PSA_REQUIRE(map_elem_bytes == 1 || map_elem_bytes == 4, PSA_ERR_ARG, "psa_list_from_map: map_elem_bytes must be 1 or 4");
  PSA_REQUIRE(rows > 0 && rows < (1ll << 31) && Nk > 0 && align_div >= 1, PSA_ERR_ARG, "psa_list_from_map: bad sizes");
  hipLaunchKernelGGL(psa_list_from_map_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, (hipStream_t)stream, map,
                     map_elem_bytes, list_out, rows, Nk, align_div);
  return psa_check_launch("psa_list_from_map");
}

// ---------------------------------------------------------------------------------------
// map = min(map, cap[bh, col])
// ---------------------------------------------------------------------------------------
__global__ void psa_map_min_cap_kernel(void* map, int map_elem, const int32_t* cap, int Hq, int n_rep, int Mq, int Nk) {
  const int64_t bh = blockIdx.y;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)Mq * Nk) return;
  const int col = (int)(i % Nk);
  const int64_t idx = bh * Mq * Nk + i;
  const int m = load_map(map, idx, map_elem);
  const int c = cap[((bh / Hq) * (Hq / n_rep) + (bh % Hq) / n_rep) * Nk + col];
  if (c < m) store_map(map, idx, map_elem, c);
}

// (cap per kv head: query head h of a batch takes the cap of kv head h / (Hq / Hkv))
int psa_map_min_cap_heads(void* map, int map_elem_bytes, const int32_t* cap, int B, int Hq, int Hkv, int Mq, int Nk, psa_stream_t stream) {
  const int64_t bh = (int64_t)B * Hq;
  PSA_REQUIRE(map && cap, PSA_ERR_ARG, "psa_map_min_cap: null pointer");
  PSA_REQUIRE(map_elem_bytes == 1 || map_elem_bytes == 4, PSA_ERR_ARG, "psa_map_min_cap: map_elem_bytes must be 1 or 4");
  PSA_REQUIRE(bh > 0 && bh <= 65535 && Mq > 0 && Nk > 0 && Hkv > 0 && Hq % Hkv == 0, PSA_ERR_ARG, "psa_map_min_cap: bad sizes");
  int64_t n = (int64_t)Mq * Nk;
  hipLaunchKernelGGL(psa_map_min_cap_kernel, dim3((unsigned)((n + 255) / 256), (unsigned)bh), dim3(256), 0,
                     (hipStream_t)stream, map, map_elem_bytes, cap, Hq, Hq / Hkv, Mq, Nk);
  return psa_check_launch("psa_map_min_cap");
}

extern "C" int psa_map_min_cap(void* map, int map_elem_bytes, const int32_t* cap, int64_t bh, int Mq, int Nk,
                               psa_stream_t stream) {
  PSA_REQUIRE(bh > 0 && bh <= 65535, PSA_ERR_ARG, "psa_map_min_cap: bad sizes");
  return psa_map_min_cap_heads(map, map_elem_bytes, cap, 1, (int)bh, (int)bh, Mq, Nk, stream);
}

// ---------------------------------------------------------------------------------------
// density = mean(1/level)
// ---------------------------------------------------------------------------------------
// Kernel 1 counts, in eighths (8 / level: exact integers), a share of one (batch, head) map per workgroup; kernel 2 adds the
// shares of every map and forms the means in a fixed order (deterministic).  One workgroup per map used B * H of the 256
// CUs, and a map that does not start on a 16-byte boundary was read byte by byte: 48 maps of 353 x 1410 bytes 259 -> 10 us,
// 12 maps of 256 x 256 bytes 12 -> 5 us (the mean kernel: 5 us, its launch).
constexpr int DENS_UNITS = 4096;   // 16-byte units per workgroup: 16 per thread
constexpr int DENS_MAX_SHARES = 64;

// eighths of the four map bytes in w: a byte counts when it is exactly 1, 2, 4 or 8
__device__ __forceinline__ int density_eighths4(uint32_t w) {
  const uint32_t one = 0x01010101u;
  const uint32_t b1 = w & one, b2 = (w >> 1) & one, b4 = (w >> 2) & one, b8 = (w >> 3) & one;
  uint32_t ok = one;
  // (rare) some byte has several bits set, or one above the fourth
  if (__builtin_expect((((b1 + b2 + b4 + b8) & 0x06060606u) | (w & 0xf0f0f0f0u)) != 0, 0)) {
    ok = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t v = (w >> (8 * e)) & 0xffu;
      ok |= (uint32_t)(v == 1 || v == 2 || v == 4 || v == 8) << (8 * e);
    }
  }
  return 8 * __popc(b1 & ok) + 4 * __popc(b2 & ok) + 2 * __popc(b4 & ok) + __popc(b8 & ok);
}
__device__ __forceinline__ int density_eighths1(int lv) {
  return lv == 1 ? 8 : lv == 2 ? 4 : lv == 4 ? 2 : lv == 8 ? 1 : 0;
}

// part == nullptr (one share per map, whose count may need more than 32 bits): the density itself goes to out.
// NT threads: 256 for shares, 1024 where one workgroup counts a map and only its own loads in flight hide their latency (int8 maps,
// us with 256 / 1024 threads: 12 of 256 x 1024 30 / 18, causal 173 / 71; 48 of 353 x 1410 56 / 30, causal 315 / 125; 1000 of
// 256 x 256 61 / 61, causal 114 / 104; 12 of 64 x 64 9.8 / 8.8).
template <int NT>
__global__ __launch_bounds__(NT) void psa_density_kernel(const void* map, int map_elem, int Mq, int Nk, int causal, int32_t* part, double cells,
                                                          float* out) {
  __shared__ int64_t s_part[NT / 64];
  const int64_t bh = blockIdx.x;
  const int64_t n = (int64_t)Mq * Nk;
  const int tid = threadIdx.x, shares = gridDim.y;
  const unsigned char* base = (const unsigned char*)map + bh * n * map_elem;
  const int epu = 16 / map_elem;  // map entries per 16-byte load
  // entries in front of the first 16-byte boundary (maps of odd sizes start anywhere) and behind the last one: one by one
  const int64_t to_16 = (int64_t)((16 - ((uintptr_t)base & 15)) & 15) / map_elem;
  const int64_t head = to_16 < n ? to_16 : n;
  const int64_t units = (n - head) / epu;
  const unsigned char* body = base + head * map_elem;
  int acc = 0;
  for (int64_t u = (int64_t)blockIdx.y * NT + tid; u < units; u += (int64_t)shares * NT) {
    const u32x4 w = *(const u32x4*)(body + u * 16);
    if (causal) {
      const int64_t i0 = head + u * epu;
      int64_t r = i0 / Nk;
      int c = (int)(i0 - r * Nk);
      for (int e = 0; e < epu; ++e) {
        const int lv = map_elem == 1 ? (int)(signed char)((w[e >> 2] >> ((e & 3) * 8)) & 0xff) : (int)w[e & 3];
        acc += c <= r ? density_eighths1(lv) : 0;
        if (++c == Nk) {
          c = 0;
          ++r;
        }
      }
    } else if (map_elem == 1) {
#pragma unroll
      for (int e = 0; e < 4; ++e) acc += density_eighths4(w[e]);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) acc += density_eighths1((int)w[e]);
    }
  }
  const int64_t singles = n - units * epu;
  for (int64_t i = (int64_t)blockIdx.y * NT + tid; i < singles; i += (int64_t)shares * NT) {
    const int64_t idx = i < head ? i : i + units * epu;
    const int64_t r = idx / Nk;
    if (!causal || idx - r * Nk <= r) acc += density_eighths1(load_map(map, bh * n + idx, map_elem));
  }
  int64_t sum;
  if constexpr (NT == 256) {  // (a share's count has 32 bits)
    sum = wave_scan_add(acc);
  } else {
    sum = acc;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
  }
  if ((tid & 63) == 63) s_part[tid >> 6] = sum;
  __syncthreads();
  if (tid != 0) return;
  sum = 0;
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) sum += s_part[w];
  if (part != nullptr) part[bh * shares + blockIdx.y] = (int32_t)sum;
  else out[bh] = (float)((double)sum * 0.125 / cells);
}

// out: the BH densities (of part's counts; part == nullptr: there already), then their mean (summed in index order); with H > 0
// also 1 - mean and the H per-head means over the BH / H batches.  One workgroup, behind the layer's last kernel: latency.  Neighbouring lanes, one
// per four shares, add up a map's counts, and up to 256 densities are read back from LDS (12 heads of 256 x 1024 and
// 2 x 48 of 139 x 556: one thread per map and densities from memory 6.7 and 6.6 us, now 2.9 and 3.2).
__global__ __launch_bounds__(256) void psa_density_mean_kernel(const int32_t* part, int shares, int BH, int H, double cells, float* out) {
  __shared__ float s_d[256];
  const int tid = threadIdx.x;
  int g_log2 = 0;
  while (g_log2 < 6 && (4 << g_log2) < shares) ++g_log2;
  double acc = 0.0;
  for (int i0 = 0; i0 < BH; i0 += 256) {
    const int maps = BH - i0 < 256 ? BH - i0 : 256;
    if (part != nullptr) {
      for (int m0 = 0; m0 < maps; m0 += 256 >> g_log2) {
        const int m = m0 + (tid >> g_log2);
        int64_t t = 0;
        if (m < maps)
          for (int s = tid & ((1 << g_log2) - 1); s < shares; s += 1 << g_log2) t += part[(int64_t)(i0 + m) * shares + s];
        for (int o = 1 << g_log2 >> 1; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
        if (m < maps && (tid & ((1 << g_log2) - 1)) == 0) out[i0 + m] = s_d[m] = (float)((double)t * 0.125 / cells);
      }
    } else if (tid < maps) {
      s_d[tid] = out[i0 + tid];
    }
    __syncthreads();
    if (tid == 0)
      for (int e = 0; e < maps; ++e) acc += (double)s_d[e];
    if (BH > 256) __syncthreads();
  }
  if (tid == 0) {
    const float mean = (float)(acc / (double)BH);
    out[BH] = mean;
    if (H > 0) out[BH + 1] = 1.0f - mean;
  }
  const float* d = BH <= 256 ? s_d : out;
  for (int h = tid; h < H; h += 256) {
    float sum = 0.f;
    for (int b = 0; b * H + h < BH; ++b) sum += d[b * H + h];
    out[BH + 2 + h] = sum / (float)(BH / H);
  }
}

static int density_run(const void* map, int map_elem_bytes, int64_t bh, int H, int Mq, int Nk, int causal, int shares, int32_t* part,
                       float* out, psa_stream_t stream) {
  PSA_REQUIRE(map && out, PSA_ERR_ARG, "psa_density: null pointer");
  PSA_REQUIRE(map_elem_bytes == 1 || map_elem_bytes == 4, PSA_ERR_ARG, "psa_density: map_elem_bytes must be 1 or 4");
  PSA_REQUIRE(bh > 0 && bh < (1 << 30) && Mq > 0 && Nk > 0, PSA_ERR_ARG, "psa_density: bad sizes");
  const int sq = Mq < Nk ? Mq : Nk;
  const double cells = causal ? (double)sq * (sq + 1) / 2.0 + (Mq > Nk ? (double)(Mq - Nk) * Nk : 0.0) : (double)Mq * Nk;
  const bool wide = part == nullptr;
  auto kern = wide ? psa_density_kernel<1024> : psa_density_kernel<256>;
  hipLaunchKernelGGL(kern, dim3((unsigned)bh, (unsigned)shares), dim3(wide ? 1024 : 256), 0, (hipStream_t)stream, map, map_elem_bytes, Mq, Nk,
                     causal, part, cells, out);
  hipLaunchKernelGGL(psa_density_mean_kernel, dim3(1), dim3(256), 0, (hipStream_t)stream, part, shares, (int)bh, H, cells, out);
  return psa_check_launch("psa_density");
}

// (no workspace: one share per map)
extern "C" int psa_density(const void* map, int map_elem_bytes, int64_t bh, int Mq, int Nk, int causal, float* density_out,
                           psa_stream_t stream) {
  return density_run(map, map_elem_bytes, bh, 0, Mq, Nk, causal, 1, nullptr, density_out, stream);
}

static int density_shares(int map_elem_bytes, int64_t bh, int Mq, int Nk) {
  const int64_t units = ((int64_t)Mq * Nk * map_elem_bytes + 15) / 16;
  int64_t s = (units + DENS_UNITS - 1) / DENS_UNITS;
  // at least about two workgroups per CU, down to one 16-byte unit per thread
  while (s * bh < 512 && s * 256 < units) s *= 2;
  // (a share's count has 32 bits: at most 2^27 map entries per share)
  const int64_t least = ((int64_t)Mq * Nk) >> 27, most = least > DENS_MAX_SHARES ? least : DENS_MAX_SHARES;
  return (int)(s < 1 ? 1 : (s > most ? most : s));
}
extern "C" int64_t psa_density_stats_workspace_bytes(int map_elem_bytes, int B, int H, int Mq, int Nk) {
  if (B <= 0 || H <= 0 || Mq <= 0 || Nk <= 0) return 0;
  return (int64_t)B * H * density_shares(map_elem_bytes, (int64_t)B * H, Mq, Nk) * (int64_t)sizeof(int32_t);
}
extern "C" int psa_density_stats(const void* map, int map_elem_bytes, int B, int H, int Mq, int Nk, int causal, void* workspace,
                                 float* stats_out, psa_stream_t stream) {
  PSA_REQUIRE(B > 0 && H > 0, PSA_ERR_ARG, "psa_density_stats: B and H must be positive");
  PSA_REQUIRE(Mq > 0 && Nk > 0, PSA_ERR_ARG, "psa_density_stats: bad sizes");
  PSA_REQUIRE(workspace, PSA_ERR_ARG, "psa_density_stats: null pointer");
  return density_run(map, map_elem_bytes, (int64_t)B * H, H, Mq, Nk, causal, density_shares(map_elem_bytes, (int64_t)B * H, Mq, Nk),
                     (int32_t*)workspace, stats_out, stream);
}
